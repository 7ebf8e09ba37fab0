// FP32 triangle-to-triangle farfield N-body (far_tri.h).
#include "far_tri.h"

namespace tct {
template <>
int far_tri_launch<float>(int kernel, int nq, const double *params, const double *qw,
                          const TriSegTable<float> &t, unsigned blocks, hipStream_t st) {
    return far_tri_nq<float>(kernel, nq, params, qw, t, blocks, st);
}
template <>
int far_tri_resident<float>(int kernel, int nq, int *blocks) {
    return far_tri_occ_nq<float>(kernel, nq, blocks);
}
}  // namespace tct
