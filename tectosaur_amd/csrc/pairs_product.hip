// Pair integrals with a product rule (an obs triangle rule times a src
// triangle rule), FP64, gfx950: the near rule and the farfield correction of
// the nearfield (gauss4d_tri), by the formulas of pairs.hip.
//
// What bounds it: FP64 VALU.  A general 4-D rule costs every point the whole
// of D = y - x (12 FMAs) and, for all but RH, the products of both bases.
// Here a lane fixes P points of one side and walks the other side's points:
//   * the moving point costs 6 FMAs for P pairs, D three subtractions;
//   * the fixed point's weight and basis leave the loop, and with P1 bases
//     the moving side's are the moments 1, xi, eta of the moving parameters;
//   * n . D with the moving side's normal is one number per fixed point (RT,
//     whose normal is the src one; RA is the same with the sides exchanged).
// FP64 VALU instructions per point, general rule -> here: RH 34 -> 26.5
// (P = 4), RT and RA 92 -> 32, U 134 -> 48, T, A and H 160 -> 90.
// The walked rule is wave-uniform (scalar loads, one step ahead).  GL lanes
// share a pair where the pairs alone are too few: each takes every GL-th
// group of P fixed points, so the walked rule stays uniform; their sums meet
// in an xor butterfly.
#include "pair_common.h"

namespace tct {

// RA fixes src points and walks obs points; the others the other way round.
template <int KID>
constexpr bool fix_src() { return KID == TCT_RA; }
// Inner sums per fixed point (RH has none).
template <int KID>
constexpr int n_inner() {
    return KID == TCT_RH ? 1 : (KID == TCT_RT || KID == TCT_RA) ? 10 : (KID == TCT_U ? 21 : 27);
}
// Sums per pair: U keeps, per (obs basis, src basis), 1/r and six D D / r^3
// sums; the others the accumulators of the general integrator.
template <int KID>
constexpr int n_outer() { return KID == TCT_U ? 63 : n_acc<KID>(); }

// One rule of a side: points q [n][2], weights w [n].
struct SideRule {
    int n;
    const double *q, *w;
};
// The walked rule is read through the constant address space (the kernel
// never writes it): uniform loads from there are scalar loads although the
// pointer comes from a struct.
typedef const __attribute__((address_space(4))) double *rule_ptr;

template <int KID, int P, int CK>
__device__ __forceinline__ void walk_point(const double (&M)[3], double mx, double my, double w,
                                           const double (&F)[P][3], const double (&fq)[P][2],
                                           const double (&wf)[P], bool same, const double *mo,
                                           const double *ns, const ElasticConsts &c, double *acc,
                                           double (&a)[P][n_inner<KID>()]) {
#pragma unroll
    for (int p = 0; p < P; ++p) {
        double D[3];
#pragma unroll
        for (int d = 0; d < 3; ++d) D[d] = M[d] - F[p][d];
        const double r2 = D[0] * D[0] + D[1] * D[1] + D[2] * D[2];
        double invr = rsq_pos(r2);
        if constexpr (CK == CK_FULL) {
            const bool skip = (same && mx == fq[p][0] && my == fq[p][1]) || r2 == 0.0;
            invr = skip ? 0.0 : invr;
        }
        if constexpr (KID == TCT_T || KID == TCT_A || KID == TCT_H) {
            double K[9];
            tensor_invr<KID>(D, invr, mo, ns, c, K);
            const double wx = w * mx, wy = w * my;
#pragma unroll
            for (int k = 0; k < 9; ++k) {
                a[p][3 * k] = fma(w, K[k], a[p][3 * k]);
                a[p][3 * k + 1] = fma(wx, K[k], a[p][3 * k + 1]);
                a[p][3 * k + 2] = fma(wy, K[k], a[p][3 * k + 2]);
            }
        } else if constexpr (KID == TCT_RH) {
            // straight into the pair's seven sums: one product of weights
            // more a point, but P sets of inner sums fewer (P = 4: 162 -> 120
            // registers, a fourth wave per SIMD)
            const double wi = (w * wf[p]) * invr;
            const double wi3 = wi * (invr * invr);
            const double e[3] = {wi3 * D[0], wi3 * D[1], wi3 * D[2]};
            acc[0] += wi;
#pragma unroll
            for (int i = 0; i < 3; ++i)
#pragma unroll
                for (int j = i; j < 3; ++j)
                    acc[1 + sym6(i, j)] = fma(e[i], D[j], acc[1 + sym6(i, j)]);
        } else {
            const double wi = w * invr;
            const double wi3 = wi * (invr * invr);
            const double e[3] = {wi3 * D[0], wi3 * D[1], wi3 * D[2]};
            if constexpr (KID == TCT_U) {
                a[p][0] += wi;
                a[p][1] = fma(wi, mx, a[p][1]);
                a[p][2] = fma(wi, my, a[p][2]);
#pragma unroll
                for (int i = 0; i < 3; ++i)
#pragma unroll
                    for (int j = i; j < 3; ++j) {
                        const double t = e[i] * D[j];
                        double *b = &a[p][3 + 3 * sym6(i, j)];
                        b[0] += t;
                        b[1] = fma(t, mx, b[1]);
                        b[2] = fma(t, my, b[2]);
                    }
            } else {
                a[p][0] += wi;
#pragma unroll
                for (int i = 0; i < 3; ++i)
#pragma unroll
                    for (int j = i; j < 3; ++j)
                        a[p][1 + sym6(i, j)] = fma(e[i], D[j], a[p][1 + sym6(i, j)]);
                a[p][7] += wi3;
                a[p][8] = fma(wi3, mx, a[p][8]);
                a[p][9] = fma(wi3, my, a[p][9]);
            }
        }
    }
}

// acc += w_f phi_b(fixed point) x the inner sums a.  dn: n . D of the fixed
// point with the moving side's normal (D = moving - fixed).
template <int KID>
__device__ __forceinline__ void fold_point(const double *a, double wf, double fx, double fy,
                                           double dn, const ElasticConsts &c, double *acc) {
    const double pf[3] = {1.0 - fx - fy, fx, fy};
    if constexpr (KID == TCT_RT || KID == TCT_RA) {
        // RT's D is src - obs, RA's the same: moving - fixed with the sign of n . D
        const double q3 = (KID == TCT_RT ? c.CsRT2 : -c.CsRT2) * dn;
        const double m3[3] = {q3 * (a[7] - a[8] - a[9]), q3 * a[8], q3 * a[9]};
#pragma unroll
        for (int b = 0; b < 3; ++b) {
            const double wl = wf * pf[b];
            acc[b] = fma(wl, c.CsRT1 * a[0], acc[b]);
            const double wq = wl * c.CsRT0;
#pragma unroll
            for (int k = 0; k < 6; ++k) acc[3 + 6 * b + k] = fma(wq, a[1 + k], acc[3 + 6 * b + k]);
#pragma unroll
            for (int bm = 0; bm < 3; ++bm) {
                const int o = KID == TCT_RT ? 21 + 3 * b + bm : 21 + 3 * bm + b;
                acc[o] = fma(wl, m3[bm], acc[o]);
            }
        }
    } else {
        // U: seven sums, T, A, H: nine entries, each with the moving moments
        constexpr int NK = KID == TCT_U ? 7 : 9;
#pragma unroll
        for (int k = 0; k < NK; ++k) {
            const double mm[3] = {a[3 * k] - a[3 * k + 1] - a[3 * k + 2], a[3 * k + 1],
                                  a[3 * k + 2]};
#pragma unroll
            for (int b = 0; b < 3; ++b)
#pragma unroll
                for (int bs = 0; bs < 3; ++bs) {
                    const int o = KID == TCT_U ? (3 * b + bs) * 7 + k
                                               : b * 27 + (k / 3) * 9 + bs * 3 + k % 3;
                    acc[o] = fma(wf * pf[b], mm[bs], acc[o]);
                }
        }
    }
}

template <int KID, int P, int GL, int CK, bool SUB>
__global__ __launch_bounds__(256) void pairs_product_kernel(
    SideRule ro, SideRule rs, SideRule minus, const double *__restrict__ pts,
    const int32_t *__restrict__ tris, int n_pairs, const int32_t *__restrict__ pairs,
    int pair_width, ElasticConsts c, const int32_t *__restrict__ rows,
    double *__restrict__ out) {
    constexpr int NI = n_inner<KID>(), NA = n_outer<KID>();
    constexpr bool FS = fix_src<KID>();
    __shared__ PairTable table;
    __shared__ PairStage<KID, GL> stage[4];
    fill_pair_table<KID>(table);
    __syncthreads();
    const int gid = blockIdx.x * blockDim.x + threadIdx.x;
    const int pair = gid / GL, sub = gid % GL;
    // lanes past the end walk the last pair (the butterfly and the uniform
    // loop take every lane) and write nothing
    const bool live = pair < n_pairs;
    const int32_t *pp = pairs + (size_t)(live ? pair : n_pairs - 1) * pair_width;
    int oc = 0, sc = 0, flip = 0;
    if (pair_width == 5) {
        oc = pp[2];
        sc = pp[3];
        flip = pp[4] != 0;
    }
    // F: edges of the fixed triangle; m0, me: base and edges of the moving
    // one, both relative to the fixed triangle's vertex 0
    double fe[2][3], m0[3], me[2][3], mo[3], ns[3];
    {
        Tri ot, st;
        load_tri(ot, pts, tris, pp[0], oc, 0);
        load_tri(st, pts, tris, pp[1], sc, flip);
        const Tri &f = FS ? st : ot, &m = FS ? ot : st;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            fe[0][d] = f.v[1][d] - f.v[0][d];
            fe[1][d] = f.v[2][d] - f.v[0][d];
            me[0][d] = m.v[1][d] - m.v[0][d];
            me[1][d] = m.v[2][d] - m.v[0][d];
            m0[d] = m.v[0][d] - f.v[0][d];
            mo[d] = ot.n[d];
            ns[d] = st.n[d];
        }
    }
    const bool same = pp[0] == pp[1] && oc == sc && !flip;
    const double *mn = FS ? mo : ns;   // the moving side's normal

    double acc[NA];
#pragma unroll
    for (int k = 0; k < NA; ++k) acc[k] = 0.0;
    // the rule, then the one to subtract (on both sides, with the fixed
    // points' weights negative): the outputs are linear in the sums
#pragma unroll 1
    for (int pass = 0; pass < (minus.n > 0 ? 2 : 1); ++pass) {
        const SideRule rf = pass ? minus : (FS ? rs : ro), rm = pass ? minus : (FS ? ro : rs);
        const rule_ptr mq = (rule_ptr)rm.q, mw = (rule_ptr)rm.w;
        const int groups = (rf.n + P - 1) / P;
        for (int g0 = 0; g0 < groups; g0 += GL) {
            // a lane without a group, and points past the end of the rule, repeat
            // the last point with weight zero
            double F[P][3], fq[P][2], wf[P], a[P][NI];
#pragma unroll
            for (int p = 0; p < P; ++p) {
                const int i = (g0 + sub) * P + p;
                const int ic = i < rf.n ? i : rf.n - 1;
                fq[p][0] = rf.q[2 * ic];
                fq[p][1] = rf.q[2 * ic + 1];
                wf[p] = i < rf.n ? (pass ? -rf.w[ic] : rf.w[ic]) : 0.0;
#pragma unroll
                for (int d = 0; d < 3; ++d) F[p][d] = fma(fq[p][1], fe[1][d], fq[p][0] * fe[0][d]);
#pragma unroll
                for (int k = 0; k < NI; ++k) a[p][k] = 0.0;
            }
            double qx = mq[0], qy = mq[1], qw = mw[0];
#pragma unroll 1
            for (int j = 0; j < rm.n; ++j) {
                // wait for this point's scalar loads here, then issue the next
                // one's: they come back while this point computes
                double &dep = KID == TCT_RH ? acc[0] : a[P - 1][NI - 1];
                asm volatile("" : "+v"(m0[0]), "+v"(m0[1]), "+v"(m0[2]), "+v"(dep)
                             : "s"(qw) : "memory");
                const double x = qx, y = qy, w = qw;
                const int jn = j + 1 < rm.n ? j + 1 : j;
                qx = mq[2 * jn];
                qy = mq[2 * jn + 1];
                qw = mw[jn];
                double M[3];
#pragma unroll
                for (int d = 0; d < 3; ++d) M[d] = fma(y, me[1][d], fma(x, me[0][d], m0[d]));
                walk_point<KID, P, CK>(M, x, y, w, F, fq, wf, same, mo, ns, c, acc, a);
            }
            if constexpr (KID != TCT_RH) {
#pragma unroll
                for (int p = 0; p < P; ++p) {
                    double dn = 0.0;
                    if constexpr (KID == TCT_RT || KID == TCT_RA)
#pragma unroll
                        for (int d = 0; d < 3; ++d) dn = fma(mn[d], m0[d] - F[p][d], dn);
                    fold_point<KID>(a[p], wf[p], fq[p][0], fq[p][1], dn, c, acc);
                }
            }
        }
    }
    if constexpr (GL > 1) {
#pragma unroll
        for (int k = 0; k < NA; ++k) {
            double v = acc[k];
#pragma unroll
            for (int off = GL / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
            acc[k] = v;
        }
    }
    Tri ot, st;
    tri_from_edges(FS ? st : ot, fe[0], fe[1]);
    tri_from_edges(FS ? ot : st, me[0], me[1]);
    write_pairs<KID, GL, SUB, write_unroll<KID, GL>()>(
        [&](double *p) {
            if constexpr (KID == TCT_U) {
                // the six D D sums and the 1/r sum to the six entries of K
                double k6[81];
#pragma unroll
                for (int b = 0; b < 3; ++b)
#pragma unroll
                    for (int e = 0; e < 3; ++e)
#pragma unroll
                        for (int d = 0; d < 3; ++d)
#pragma unroll
                            for (int f = d; f < 3; ++f) {
                                const double *s = acc + (3 * b + e) * 7;
                                const double k2 = c.CsU1 * s[1 + sym6(d, f)];
                                k6[b * 27 + d * 9 + e * 3 + f] = d == f ? fma(c.CsU0, s[0], k2) : k2;
                            }
                pack_pair<KID>(k6, ot, st, c, oc, sc, flip, p);
            } else {
                pack_pair<KID>(acc, ot, st, c, oc, sc, flip, p);
            }
        },
        table, stage[threadIdx.x / 64], (int)(threadIdx.x % 64) / GL, sub == 0,
        live ? out_row(rows, pair) : -1, out);
}

// Fixed points per lane (P) and lanes per pair (GL) for a rule of nf fixed
// and nm walked points: the fewest issue slots of a SIMD, 6 a walked point
// and group of P and about 26 a pair of points, plus what every lane pays
// once, times the waves that the SIMD runs -- whole ones while they are few,
// and never less than two, which a SIMD needs to issue at its rate.  (19 x 19
// points, RH, 226,590 pairs: P = 4 with four lanes for five groups 191 us,
// P = 2 with two lanes for ten 160 us.)  The outputs of a wave's pairs leave
// sixteen pairs at a time, 350 slots each time.
struct Split {
    int P, GL;
};
inline Split product_split(int kernel, int nf, int nm, int64_t n_pairs) {
    const bool tensor = kernel <= TCT_H;      // U, T, A, H: one point per lane
    const int pmax = kernel == TCT_RH ? 4 : (tensor ? 1 : 2);
    const int na = kernel == TCT_U ? 63 : (tensor ? 81 : (kernel == TCT_RH ? 7 : 30));
    Split best{1, 1};
    double cost = 0.0;
    for (int P = 1; P <= pmax; P *= 2) {
        // with so few points the registers of a wider group cost more
        // (RT, 4 x 4 points: 153 us with P = 2, 130 with 1)
        if (P > 1 && nf <= 4 && kernel != TCT_RH) break;
        const int groups = (nf + P - 1) / P;
        for (int gl = 1, lg = 0; gl <= 16 && gl <= groups; gl *= 2, ++lg) {
            if (tensor && (gl == 2 || gl == 8)) continue;
            const double serial = (double)((groups + gl - 1) / gl) * nm * (6 + 26 * P) + 800.0 +
                                  (gl < 4 ? 1400.0 / gl : 350.0) + 5.0 * na * lg;
            double waves = (double)n_pairs * gl / 64.0 / 1024.0;
            waves = waves < 2.0 ? 2.0 : (waves < 8.0 ? std::ceil(waves) : waves + 0.5);
            if (cost == 0.0 || serial * waves < cost) {
                cost = serial * waves;
                best = Split{P, gl};
            }
        }
    }
    return best;
}

struct ProductArgs {
    SideRule ro, rs, minus;
    const double *pts;
    const int32_t *tris;
    int n_pairs;
    const int32_t *pairs;
    int pair_width, check0;
    ElasticConsts c;
    const int32_t *rows;
    bool subtract;
    double *out;
};

template <int KID, int P, int GL, int CK, bool SUB>
static void product_launch(const ProductArgs &a, hipStream_t st) {
    const unsigned nb = (unsigned)ceil_div((int64_t)a.n_pairs * GL, (int64_t)256);
    hipLaunchKernelGGL((pairs_product_kernel<KID, P, GL, CK, SUB>), dim3(nb), dim3(256), 0, st,
                       a.ro, a.rs, a.minus, a.pts, a.tris, a.n_pairs, a.pairs, a.pair_width, a.c,
                       a.rows, a.out);
}

template <int KID, int P, int GL>
static void product_go(const ProductArgs &a, hipStream_t st) {
    // where no point has equal parameters the full test is the r2 == 0 test
    if (a.check0 == CK_NONE) {
        if (a.subtract)
            product_launch<KID, P, GL, CK_NONE, true>(a, st);
        else
            product_launch<KID, P, GL, CK_NONE, false>(a, st);
    } else {
        if (a.subtract)
            product_launch<KID, P, GL, CK_FULL, true>(a, st);
        else
            product_launch<KID, P, GL, CK_FULL, false>(a, st);
    }
}

}  // namespace tct

using namespace tct;

extern "C" int tct_pairs_product(int kernel, int n_o, const double *qo, const double *wo, int n_s,
                                 const double *qs, const double *ws, int n_minus,
                                 const double *q_minus, const double *w_minus, const double *pts,
                                 const int32_t *tris, int64_t n_pairs, const int32_t *pairs,
                                 int pair_width, int check0, const double *params_host,
                                 const int32_t *rows, int subtract, double *out, void *stream) {
    TCT_CHECK_ARG(kernel >= TCT_U && kernel <= TCT_RH, "pairs_product: kernel id %d", kernel);
    TCT_CHECK_ARG(n_o > 0 && n_s > 0 && n_o < (1 << 20) && n_s < (1 << 20),
                  "pairs_product: rules of %d x %d points", n_o, n_s);
    TCT_CHECK_ARG(n_pairs >= 0 && n_pairs < (1LL << 26),
                  "pairs_product: n_pairs %lld (max 2^26 per call)", (long long)n_pairs);
    TCT_CHECK_ARG(pair_width == 2 || pair_width == 5, "pairs_product: pair_width %d", pair_width);
    TCT_CHECK_ARG(check0 == CK_NONE || check0 == CK_FULL || check0 == CK_R2,
                  "pairs_product: check0 %d", check0);
    TCT_CHECK_ARG(n_minus >= 0 && n_minus < (1 << 20) && (n_minus == 0 || (q_minus && w_minus)),
                  "pairs_product: rule of %d points to subtract", n_minus);
    TCT_CHECK_ARG(qo && wo && qs && ws && pts && tris && params_host && out &&
                      (pairs || n_pairs == 0),
                  "pairs_product: null pointer");
    if (n_pairs == 0) return TCT_OK;
    const int nf = kernel == TCT_RA ? n_s : n_o;
    const Split sp = product_split(kernel, nf, kernel == TCT_RA ? n_o : n_s, n_pairs);
    const int P = sp.P, gl = sp.GL;
    hipStream_t st = as_stream(stream);
    const ProductArgs args{{n_o, qo, wo}, {n_s, qs, ws}, {n_minus, q_minus, w_minus},
                           pts, tris, (int)n_pairs, pairs, pair_width, check0,
                           elastic_consts(params_host), rows, subtract != 0, out};
#define TCT_GO(K, P, GL) product_go<K, P, GL>(args, st)
#define TCT_GL(K, P)                                                                             \
    switch (gl) {                                                                                \
    case 1: TCT_GO(K, P, 1); break;                                                              \
    case 2: TCT_GO(K, P, 2); break;                                                              \
    case 4: TCT_GO(K, P, 4); break;                                                              \
    case 8: TCT_GO(K, P, 8); break;                                                              \
    default: TCT_GO(K, P, 16); break;                                                            \
    }
#define TCT_GL3(K)                                                                               \
    switch (gl) {                                                                                \
    case 1: TCT_GO(K, 1, 1); break;                                                              \
    case 4: TCT_GO(K, 1, 4); break;                                                              \
    default: TCT_GO(K, 1, 16); break;                                                            \
    }
#define TCT_P2(K)                                                                                \
    if (P == 2) {                                                                                \
        TCT_GL(K, 2)                                                                             \
    } else {                                                                                     \
        TCT_GL(K, 1)                                                                             \
    }
    switch (kernel) {
    case TCT_U: TCT_GL3(TCT_U) break;
    case TCT_T: TCT_GL3(TCT_T) break;
    case TCT_A: TCT_GL3(TCT_A) break;
    case TCT_H: TCT_GL3(TCT_H) break;
    case TCT_RT: TCT_P2(TCT_RT) break;
    case TCT_RA: TCT_P2(TCT_RA) break;
    default:
        if (P == 4) {
            TCT_GL(TCT_RH, 4)
        } else {
            TCT_P2(TCT_RH)
        }
    }
#undef TCT_P2
#undef TCT_GL3
#undef TCT_GL
#undef TCT_GO
    TCT_CHECK_LAUNCH("pairs_product");
    return TCT_OK;
}
