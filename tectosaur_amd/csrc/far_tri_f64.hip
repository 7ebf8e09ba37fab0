// FP64 triangle-to-triangle farfield N-body (far_tri.h).
#include "far_tri.h"

namespace tct {
template <>
int far_tri_launch<double>(int kernel, int nq, const double *params, const double *qw,
                           const TriSegTable<double> &t, unsigned blocks, hipStream_t st) {
    return far_tri_nq<double>(kernel, nq, params, qw, t, blocks, st);
}
template <>
int far_tri_resident<double>(int kernel, int nq, int *blocks) {
    return far_tri_occ_nq<double>(kernel, nq, blocks);
}
}  // namespace tct
