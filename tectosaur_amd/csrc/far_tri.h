// Triangle-to-triangle farfield N-body: the pair body of one (observation
// triangle, source triangle) pair, shared by the FP32 and FP64 units
// far_tri_f32.hip and far_tri_f64.hip.
//
// Reference semantics: farfield_tris_to_tris{K} (tectosaur/matrix_free.cl:
// 19-107) with the kernel bodies of tectosaur/kernels/kernels.cl: every
// quadrature point of one triangle against every one of the other, pairs at
// r2 == 0 skipped.
//
// What bounds it: VALU issue.  The point N-body (far_p2p.hip) evaluates every
// pair of points by itself; here a lane holds the NQ points of one
// observation triangle and walks whole source triangles, so what is constant
// over a flat triangle is formed once per triangle pair or once per point:
//   * n . D is the same for the NQ points of a source triangle, m . D for
//     those of an observation triangle, m . n for the pair, m . s for the
//     source point (T, A, H, RT, RA);
//   * terms along n are summed as scalars over the source triangle (T, H);
//   * the surface curls of RH are constant on both triangles, so a triangle
//     pair needs only 7 moments, sum 1/r and sum D_k D_l / r^3, and one
//     contraction with the source curl (RH); RT's 1/r term likewise;
//   * U keeps its two terms in separate sums, scaled once per tile.
// VALU instructions per point pair with a three-point rule in FP32, counted in
// the compiled loops that far tiles run (T, A and RT with the r2 test, two more),
// point form -> this: H 54 -> 39, RH 40 -> 23, T 31 -> 28, A 31 -> 28, RT 27 -> 25,
// RA 26 -> 24, U 20 -> 19; near tiles take two more.
// FP64: 24 to 47 a pair, and few waves to hide their latency: the registers
// leave three a SIMD for U, A and RA with three points, two for the others, one
// for H and RH with four (256 VGPRs and 66 or 44 AGPRs).  It rounds as the point
// form does except that T, A, RT and RA take one n . D or m . D for all points of
// the other triangle, whose error then does not average out: relative L2 error
// against 64-bit formulas 1.05 to 1.15 times the point form's (2,046 triangles, T
// with four points 1.7e-14 -> 2.0e-14), U, H and RH 0.96 to 1.01 times.
#pragma once
#include "far_pair.h"

namespace tct {

constexpr int TT = TCT_TRI_TILE;   // source triangles per tile (one origin)

// Weights relative to the last one: the rules of three points have equal
// ones, those of four points (the centre and a ring of three) one that
// differs, the first.
template <int NQ>
constexpr bool unit_w(int q) { return NQ == 3 || q > 0; }

// Record of one source triangle: a block of SW words per point, so that a
// point is read with whole 16-byte vectors, and the words of the triangle in
// the blocks' spare words or after them:
//   U, A, RA: [y s - -]              T: [y s e0 n_j]        H: [y s e0 e1] .. n
//   RT:       [y s n_j e_j]          RH: [y G_j] .. G_3 to G_8
// (n_j: component j of the normal, in the blocks of the first three points).
template <int KID>
constexpr int tri_sw() { return KID == TCT_RH ? 4 : 8; }
template <int KID, int NQ>
constexpr int tri_words() {
    return tri_sw<KID>() * NQ + (KID == TCT_H ? 4 : (KID == TCT_RH ? 8 : 0));
}
template <int KID, int NQ>
constexpr int tri_n_word(int d) {
    return KID == TCT_T ? 8 * d + 7 : (KID == TCT_RT ? 8 * d + 6 : 8 * NQ + d);
}
constexpr int tri_e_word(int d) { return 8 * d + 7; }                  // RT
template <int NQ>
constexpr int tri_g_word(int a) { return a < 3 ? 4 * a + 3 : 4 * NQ + a - 3; }   // RH
// Outputs per observation triangle: NQ 3-vectors; RH the 9 sums weighted by
// the observation rule; RA one weighted 3-vector and NQ 3-vectors.
template <int KID, int NQ>
constexpr int tri_out() { return KID == TCT_RH ? 9 : (KID == TCT_RA ? 3 + 3 * NQ : 3 * NQ); }
// Accumulators kept through a tile.
template <int KID, int NQ>
constexpr int tri_acc() {
    return KID == TCT_U ? 6 * NQ
           : KID == TCT_A ? 4 * NQ
           : KID == TCT_H ? 5 * NQ
           : KID == TCT_RA ? 6 + 3 * NQ
           : KID == TCT_RH ? 18
                           : 3 * NQ;
}
template <int KID>
constexpr bool tri_obs_normal() { return KID == TCT_A || KID == TCT_H || KID == TCT_RA; }
template <int KID>
constexpr bool tri_src_normal() { return KID == TCT_T || KID == TCT_H || KID == TCT_RT; }

// Kernel constants, and of a four-point rule the first weight relative to the
// others (rw), its square (rw2) and c0 times it (rwc).
template <typename T>
struct TriConst {
    T c0, c1, c2, c3, c4, eps2, rw, rw2, rwc;
};

// Words [w, w + SW) of a record (w a multiple of the vector length).
template <int SW, typename T>
__device__ __forceinline__ void tri_load(const T *r, int w, T (&q)[SW]) {
    constexpr int VW = 16 / sizeof(T);
    typedef T vec __attribute__((ext_vector_type(VW)));
#pragma unroll
    for (int v = 0; v < SW / VW; ++v) {
        const vec f = *(const vec *)(r + w + v * VW);
#pragma unroll
        for (int c = 0; c < VW; ++c) q[v * VW + c] = f[c];
    }
}

// What a triangle pair starts from: the first point's block, the normal and
// RT's curl term of the source triangle.
template <int KID, typename T>
struct TriHead {
    T q[tri_sw<KID>()], n[3], e[3];
};
template <int KID, int NQ, typename T>
__device__ __forceinline__ void tri_head(const T *r, TriHead<KID, T> &h) {
    tri_load<tri_sw<KID>(), T>(r, 0, h.q);
    if constexpr (tri_src_normal<KID>())
#pragma unroll
        for (int d = 0; d < 3; ++d) h.n[d] = r[tri_n_word<KID, NQ>(d)];
    if constexpr (KID == TCT_RT)
#pragma unroll
        for (int d = 0; d < 3; ++d) h.e[d] = r[tri_e_word(d)];
}

// Fences keep the scheduler from moving instructions across: NQ: one after
// each source point; 1: one between the observation points of a source point;
// 0: none.  They hold few points in registers at a time, and with the order of
// the terms in tri_pair they decide which instructions can meet in the FP32
// unit's two-at-once issue (which register numbers may forbid), so only
// measurement tells.  15,842 triangles, FP32, us, terms in any order and one
// fence per source point -> the order below and this:
//   3 points  U 1045 -> 961, T 1337 -> 1188, A 1443 -> 1186, H 1824 -> 1685,
//             RT 1234 -> 1065, RA 1292 -> 1113, RH 1208 -> 1170
//   4 points  U 1970 -> 1650, T 2503 -> 2102, A 2602 -> 2014, H 3364 -> 3058,
//             RT 2383 -> 1936, RA 2345 -> 1924, RH 2201 -> 1990
// (point form, 3 and 4 points: U 1150 2015, T 1453 2540, A 1354 2426,
// H 2335 4108, RT 1385 2459, RA 1219 2166, RH 1790 3073).  FP64 issues no pairs
// and is within 2% either way.
template <int KID, int NQ, typename T>
constexpr int tri_fence() {
    if (sizeof(T) == 8) return NQ;
    return KID == TCT_U || KID == TCT_A || KID == TCT_RA || (KID == TCT_H && NQ == 3) ? 1 : 0;
}

// Whether every tile runs the body with the r2 test: its two instructions more
// a pair change which others pair up, for the better with these (147,456
// triangles, FP32, ms, tiles far from the lane without the test -> all with it):
//   3 points  T 121.0 -> 95.1, A 106.1 -> 96.6, RT 93.0 -> 85.9
//   4 points  T 212.2 -> 174.8, A 203.9 -> 165.3, RH 175.3 -> 166.1
// and for the worse with the others (three and four points, U 70.2 -> 73.1, 131.7
// -> 141.8; H 132.7 -> 142.0, 252.8 -> 257.2; RA 85.7 -> 90.8, 159.6 -> 162.0; RH
// 89.2 -> 93.7; RT 167.3 -> 178.4).  FP64 keeps both bodies: at 15,842 triangles,
// where most tiles have the test anyway, one body is 1% faster, with H and RH with
// four points, which it frees of register moves, 7 and 10%.
template <int KID, int NQ, typename T>
constexpr bool tri_always_masked() {
    return sizeof(T) == 4 && (KID == TCT_T || KID == TCT_A || (KID == TCT_RT && NQ == 3) ||
                              (KID == TCT_RH && NQ == 4));
}

// a += f v
template <typename T>
__device__ __forceinline__ void add3(T *a, T f, const T *v) {
#pragma unroll
    for (int d = 0; d < 3; ++d) a[d] = fma_t(f, v[d], a[d]);
}

// One observation triangle (points x, normal m) against one source triangle
// (record r, in LDS, its head already in h): acc += its terms, and h becomes
// the head of the record `next`.  The source points come one after another;
// each one's words are read while the point before it computes.  Every fused
// multiply-add is written out, as in pair_eval, so every copy of the body
// performs the same operations.
template <int KID, int NQ, typename T, bool MASK>
__device__ __forceinline__ void tri_pair(const T (&x)[NQ][3], const T (&m)[3], const T *r,
                                         const T *next, const TriConst<T> &k,
                                         TriHead<KID, T> &h, T *acc) {
#pragma clang fp contract(off)
    constexpr int SW = tri_sw<KID>();
    constexpr int F = tri_fence<KID, NQ, T>();
    T an[NQ], ca[NQ], nt[NQ], s0 = T(0), s2[6], G[9];
    const T n[3] = {h.n[0], h.n[1], h.n[2]}, e[3] = {h.e[0], h.e[1], h.e[2]};
    T mn0 = T(0), mn1 = T(0);
    if constexpr (KID == TCT_H) {
        const T mn = dot3(m[0], m[1], m[2], n[0], n[1], n[2]);
        mn0 = k.c0 * mn;
        mn1 = k.c1 * mn;
    }
#pragma unroll
    for (int j = 0; j < NQ; ++j) {
        T q[SW];
#pragma unroll
        for (int w = 0; w < SW; ++w) q[w] = h.q[w];
        if (j + 1 < NQ) {
            tri_load<SW, T>(r, SW * (j + 1), h.q);
        } else {
            if constexpr (KID == TCT_RH)
#pragma unroll
                for (int a = 0; a < 9; ++a) G[a] = r[tri_g_word<NQ>(a)];
            tri_head<KID, NQ, T>(next, h);
        }
        const T *s = q + 3;
        // the same for every observation point: m . D, m . s and products
        T bm = T(0), cb = T(0), sm = T(0), sm4 = T(0), e1b = T(0), b4 = T(0), si = T(0);
        T ce = T(0), ej[3] = {T(0), T(0), T(0)};
        const bool uj = unit_w<NQ>(j);
        if constexpr (tri_obs_normal<KID>())
            bm = dot3(m[0], m[1], m[2], q[0] - x[0][0], q[1] - x[0][1], q[2] - x[0][2]);
        if constexpr (KID == TCT_H || KID == TCT_A)
            sm = dot3(m[0], m[1], m[2], s[0], s[1], s[2]);
        if constexpr (KID == TCT_H) {
            sm4 = k.c4 * sm;
            sm = k.c0 * sm;
            e1b = q[7] * bm;
            b4 = k.c4 * bm;
        }
        if constexpr (KID == TCT_A) {
            sm = k.c0 * sm;
            cb = k.c0 * bm;
        }
        if constexpr (KID == TCT_T) ce = k.c0 * q[6];
        if constexpr (KID == TCT_RT)
#pragma unroll
            for (int d = 0; d < 3; ++d) ej[d] = (uj ? k.c0 : k.rwc) * e[d];
#pragma unroll
        for (int p = 0; p < NQ; ++p) {
            const T D[3] = {q[0] - x[p][0], q[1] - x[p][1], q[2] - x[p][2]};
            if constexpr (F == 1)
                if (p > 0) __builtin_amdgcn_sched_barrier(0);
            const T r2 = dot3(D[0], D[1], D[2], D[0], D[1], D[2]);
            const T invr = MASK ? rsq_masked(r2, k.eps2) : rsq_plain(r2);
            const T w = invr * invr;
            // n . D, the same for every source point
            if constexpr (tri_src_normal<KID>())
                if (j == 0) {
                    an[p] = dot3(n[0], n[1], n[2], D[0], D[1], D[2]);
                    // in units of the constant its products carry
                    if constexpr (KID == TCT_T) ca[p] = -k.c0 * an[p];
                }
            if constexpr (KID == TCT_RH) {
                const bool up = unit_w<NQ>(p);
                const T iw = up && uj ? invr : invr * (up || uj ? k.rw : k.rw2);
                const T i3 = iw * w;
                const T e0 = i3 * D[0], e1 = i3 * D[1], e2 = i3 * D[2];
                if (p == 0 && j == 0) {
                    s0 = iw;
                    s2[0] = e0 * D[0];
                    s2[1] = e0 * D[1];
                    s2[2] = e0 * D[2];
                    s2[3] = e1 * D[1];
                    s2[4] = e1 * D[2];
                    s2[5] = e2 * D[2];
                } else {
                    s0 = s0 + iw;
                    s2[0] = fma_t(e0, D[0], s2[0]);
                    s2[1] = fma_t(e0, D[1], s2[1]);
                    s2[2] = fma_t(e0, D[2], s2[2]);
                    s2[3] = fma_t(e1, D[1], s2[3]);
                    s2[4] = fma_t(e1, D[2], s2[4]);
                    s2[5] = fma_t(e2, D[2], s2[5]);
                }
                continue;
            }
            const T i3 = invr * w;
            if constexpr (KID == TCT_U) {
                add3(acc + 6 * p, invr, s);
                add3(acc + 6 * p + 3, i3 * dot3(D[0], D[1], D[2], s[0], s[1], s[2]), D);
            } else if constexpr (KID == TCT_T) {
                const T ds = dot3(D[0], D[1], D[2], s[0], s[1], s[2]);
                nt[p] = j == 0 ? i3 * ds : fma_t(i3, ds, nt[p]);
                const T be = i3 * ca[p];
                if (NQ == 4) add3(acc + 3 * p, be, s);
                add3(acc + 3 * p, i3 * fma_t(-(w * an[p]), ds, ce), D);
                if (NQ == 3) add3(acc + 3 * p, be, s);
            } else if constexpr (KID == TCT_A) {
                add3(acc + 4 * p, i3 * cb, s);
                const T ds = dot3(D[0], D[1], D[2], s[0], s[1], s[2]);
                acc[4 * p + 3] = fma_t(i3, ds, acc[4 * p + 3]);
                add3(acc + 4 * p, i3 * fma_t(w * bm, ds, sm), D);
            } else if constexpr (KID == TCT_H && NQ == 3) {
                const T wa = w * an[p];
                add3(acc + 5 * p, i3 * fma_t(wa, b4, mn0), s);
                acc[5 * p + 3] = fma_t(i3, q[6], acc[5 * p + 3]);
                const T c = dot3(s[0], s[1], s[2], D[0], D[1], D[2]);
                acc[5 * p + 4] = fma_t(i3, wa * c, acc[5 * p + 4]);
                const T wbc = (w * bm) * c;
                const T ni = fma_t(k.c1, wbc, sm);
                nt[p] = j == 0 ? i3 * ni : fma_t(i3, ni, nt[p]);
                const T inner = fma_t(T(-15), wbc, sm4);
                add3(acc + 5 * p, (i3 * w) * fma_t(an[p], inner, fma_t(c, mn1, e1b)), D);
            } else if constexpr (KID == TCT_H) {
                // the same in the order that is the faster one with four
                // points (32,256 triangles: 11.85 ms, 13.2 in the order above;
                // with three points the other way round, 6.84 and 6.58)
                const T c = dot3(s[0], s[1], s[2], D[0], D[1], D[2]);
                const T wbc = (w * bm) * c;
                const T ni = fma_t(k.c1, wbc, sm);
                nt[p] = j == 0 ? i3 * ni : fma_t(i3, ni, nt[p]);
                const T wa = w * an[p];
                acc[5 * p + 3] = fma_t(i3, q[6], acc[5 * p + 3]);
                acc[5 * p + 4] = fma_t(i3, wa * c, acc[5 * p + 4]);
                const T inner = fma_t(T(-15), wbc, sm4);
                add3(acc + 5 * p, (i3 * w) * fma_t(an[p], inner, fma_t(c, mn1, e1b)), D);
                add3(acc + 5 * p, i3 * fma_t(wa, b4, mn0), s);
            } else if constexpr (KID == TCT_RT) {
                const T iw = uj ? invr : invr * k.rw;
                nt[p] = j == 0 ? iw : nt[p] + iw;
                add3(acc + 3 * p, i3 * an[p], s);
                add3(acc + 3 * p, i3 * dot3(D[0], D[1], D[2], ej[0], ej[1], ej[2]), D);
            } else {
                // RA: acc = [sum w_p s/r (3), sum w_p (D.s) D/r^3 (3),
                // per point sum (m.D) s/r^3 (3 NQ)]
                const bool up = unit_w<NQ>(p);
                const T iw = up ? invr : invr * k.rw;
                si = p == 0 ? iw : si + iw;
                add3(acc + 6 + 3 * p, i3 * bm, s);
                add3(acc + 3,
                     (up ? i3 : i3 * k.rw) * dot3(D[0], D[1], D[2], s[0], s[1], s[2]), D);
            }
        }
        if constexpr (KID == TCT_RA)
#pragma unroll
            for (int d = 0; d < 3; ++d) acc[d] = fma_t(si, s[d], acc[d]);
        if constexpr (F == NQ) __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (KID == TCT_RH) {
        // acc[0..9) += s0 G; acc[9..18) += S2 G
#pragma unroll
        for (int a = 0; a < 9; ++a) acc[a] = fma_t(s0, G[a], acc[a]);
        const T S[3][3] = {{s2[0], s2[1], s2[2]}, {s2[1], s2[3], s2[4]}, {s2[2], s2[4], s2[5]}};
#pragma unroll
        for (int a = 0; a < 3; ++a)
#pragma unroll
            for (int b = 0; b < 3; ++b)
#pragma unroll
                for (int c = 0; c < 3; ++c)
                    acc[9 + 3 * a + c] = fma_t(S[a][b], G[3 * b + c], acc[9 + 3 * a + c]);
    } else if constexpr (tri_src_normal<KID>()) {
        // the sums along n (T, H) or of 1/r (RT)
        constexpr int A = KID == TCT_H ? 5 : 3;
#pragma unroll
        for (int p = 0; p < NQ; ++p) {
            const T f = KID == TCT_T ? -k.c0 * nt[p] : nt[p];
#pragma unroll
            for (int d = 0; d < 3; ++d)
                acc[A * p + d] = fma_t(f, KID == TCT_RT ? e[d] : n[d], acc[A * p + d]);
        }
    }
}

// The outputs of a tile's accumulators.
template <int KID, int NQ, typename T>
__device__ __forceinline__ void tri_fold(const T (&m)[3], const TriConst<T> &k, const T *acc,
                                         T (&o)[tri_out<KID, NQ>()]) {
#pragma clang fp contract(off)
    if constexpr (KID == TCT_RH) {
        const T tr = (acc[0] + acc[4]) + acc[8];
#pragma unroll
        for (int a = 0; a < 3; ++a)
#pragma unroll
            for (int b = 0; b < 3; ++b) {
                T v = T(-2) * (acc[9 + 3 * a + b] + acc[3 * a + b]);
                v = fma_t(k.c1, acc[3 * b + a], v);
                if (a == b) v = fma_t(k.c0, tr, v);
                o[3 * a + b] = v;
            }
    } else if constexpr (KID == TCT_RA) {
#pragma unroll
        for (int d = 0; d < 3; ++d) o[d] = fma_t(k.c0, acc[d], k.c1 * acc[3 + d]);
#pragma unroll
        for (int a = 0; a < 3 * NQ; ++a) o[3 + a] = acc[6 + a];
    } else {
#pragma unroll
        for (int p = 0; p < NQ; ++p)
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                if constexpr (KID == TCT_U) {
                    o[3 * p + d] = fma_t(k.c0, acc[6 * p + d], acc[6 * p + 3 + d]);
                } else if constexpr (KID == TCT_A) {
                    o[3 * p + d] = fma_t(m[d], -k.c0 * acc[4 * p + 3], acc[4 * p + d]);
                } else if constexpr (KID == TCT_H) {
                    const T f = fma_t(k.c2, acc[5 * p + 4], acc[5 * p + 3]);
                    o[3 * p + d] = fma_t(m[d], f, acc[5 * p + d]);
                } else {
                    o[3 * p + d] = acc[3 * p + d];
                }
            }
    }
}

// One problem of a launch; several problems' N-bodies share one launch
// through a table passed by value (segment s owns workgroups [blk0, next
// blk0), observation block fastest, then chunk).
template <typename T>
struct TriSeg {
    const double *obs;       // [3 NQ + 3][n_obs_pad]: points, normal
    const double *obs_org;   // [3][n_obs_pad]
    const T *rec;            // [n_tiles * TT][tri_words]
    const double *src_org;   // [n_tiles][3]
    double *partial;         // [chunks][tri_out][n_obs_pad]
    double sep2;
    float eps2;
    int n_obs_pad, n_src, n_tiles, chunks, blk0;
};
constexpr int TRI_SEG_MAX = 16;
template <typename T>
struct TriSegTable {
    int n;
    TriSeg<T> s[TRI_SEG_MAX];
};

constexpr int TRI_WAVES = 4;   // waves of a workgroup, one source tile each at a time

// Chunk ch of a problem's n_tiles source tiles: tiles [t0, t1).  Chunks are made
// of whole groups of four tiles, one for each wave, where there are groups for
// all of them, else of pairs or single tiles.
struct TriChunk {
    int t0, t1;
};
__device__ __forceinline__ TriChunk tri_chunk(int n_tiles, int chunks, int ch) {
    const int unit = chunks <= (n_tiles + 3) / 4 ? 4 : (chunks <= (n_tiles + 1) / 2 ? 2 : 1);
    const int64_t units = (n_tiles + unit - 1) / unit;
    return {unit * (int)(units * ch / chunks),
            min(n_tiles, unit * (int)(units * (ch + 1) / chunks))};
}

// What a wave takes of its workgroup's chunk of source tiles [t0, t1): tiles
// t0 + wave, t0 + wave + 4, ...; of a chunk of one or two tiles, where that
// would leave waves without work, the tile's triangles in four or two parts.
// The real triangles only: a tile's padding is never walked.  (Few sources
// against many observers, FP64, four points, 59,700 x 9 triangles: one wave of
// four walking 16 triangles took 110 us for H and 52 for T, this 38 and 26, the
// point form 55 and 42.)
struct TriShare {
    int first, step, part, parts;
    // triangles [j0, j1) of a tile with n real ones
    __device__ __forceinline__ int j0(int n) const { return n * part / parts; }
    __device__ __forceinline__ int j1(int n) const { return n * (part + 1) / parts; }
};
__device__ __forceinline__ TriShare tri_share(int wave, int t0, int t1) {
    const int n = t1 - t0, parts = n == 1 ? TRI_WAVES : (n == 2 ? TRI_WAVES / 2 : 1);
    return {t0 + wave / parts, TRI_WAVES / parts, wave % parts, parts};
}

// Bytes of LDS: every wave's sums and its current source tile.
template <int KID, int NQ, typename T>
constexpr size_t tri_lds_bytes() {
    return TRI_WAVES * (sizeof(double) * 64 * tri_out<KID, NQ>() +
                        sizeof(T) * TT * tri_words<KID, NQ>());
}

// N-body.  A workgroup of four waves holds 64 observation triangles (one per
// lane, the same in every wave) and one chunk of the source tiles; wave w
// takes the chunk's tiles w, w + 4, ...  A wave stages its tile in LDS (the
// next tile's words are loaded a tile ahead) and reads the records back with
// broadcast reads, so they are VGPR operands.  The four waves' sums are added
// in wave order through LDS, so a chunk has one partial sum whatever its
// number of waves: a quarter of the partial sums that one wave per chunk
// would write and the scatter would read.
// FP32: points are relative to the source tile's FP64 origin; a tile's sums are
// FP32, the sums over tiles FP64.  Tiles whose origin is farther than sqrt(sep2) from every
// lane's origin hold no pair with r2 <= eps2 and run without the test.
template <int KID, int NQ, typename T>
__global__ __launch_bounds__(64 * TRI_WAVES) void far_tri_kernel(TriSegTable<T> segs,
                                                               TriConst<T> kc) {
    constexpr bool F32 = sizeof(T) == 4;
    constexpr int RW = tri_words<KID, NQ>();
    constexpr int NO = tri_out<KID, NQ>();
    constexpr int NA = tri_acc<KID, NQ>();
    constexpr int VW = 16 / sizeof(T);                  // words per 16-byte vector
    constexpr int NVEC = TT * RW / VW;                  // vectors per tile
    constexpr int NV = (NVEC + 63) / 64;                // per lane
    typedef T vec __attribute__((ext_vector_type(VW)));
    extern __shared__ double lds_raw[];
    const int L = (int)blockIdx.x;
    int si = 0;
    while (si + 1 < segs.n && L >= segs.s[si + 1].blk0) ++si;
    const TriSeg<T> &g = segs.s[si];
    const int n_obs_pad = g.n_obs_pad, n_src = g.n_src, n_tiles = g.n_tiles, chunks = g.chunks;
    const int obs_blocks = n_obs_pad / 64;
    const int l = L - g.blk0;
    const int ob = l % obs_blocks, ch = l / obs_blocks;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int lane = (int)threadIdx.x & 63;
    const TriChunk tc = tri_chunk(n_tiles, chunks, ch);
    const int t0 = tc.t0, t1 = tc.t1;
    const int i = ob * 64 + lane;

    // FP32 reads its points again for every tile (coalesced, and in cache by
    // then) and moves them to the tile's frame in FP64: one rounding, the same
    // as that of a source point there, so D of a pair and of the pair the other
    // way round are opposite numbers, as in the point form.  (Points stored in
    // FP32 against an origin of their triangle were rounded twice more: eight
    // meshes of 3,000 to 10,000 triangles, relative L2 error over the point
    // form's, three points T 0.85, A 0.87, H 0.85, RH 1.01, RA 1.16, four points
    // T 1.13, A 1.22; this 0.68, 0.68, 0.67, 0.90, 1.03, 1.04 and 1.06, and the
    // same time.)
    T x[NQ][3], m[3];
    if constexpr (!F32)
#pragma unroll
        for (int p = 0; p < NQ; ++p)
#pragma unroll
            for (int d = 0; d < 3; ++d) x[p][d] = g.obs[(size_t)(3 * p + d) * n_obs_pad + i];
#pragma unroll
    for (int d = 0; d < 3; ++d)
        m[d] = tri_obs_normal<KID>() ? (T)g.obs[(size_t)(3 * NQ + d) * n_obs_pad + i] : T(0);
    TriConst<T> k = kc;
    k.eps2 = F32 ? (T)g.eps2 : T(0);
    if constexpr (F32) {
        // an instruction that reads an SGPR is never dual-issued
        asm volatile("" : "+v"(k.c0), "+v"(k.c1), "+v"(k.c2), "+v"(k.c4), "+v"(k.eps2));
    }
    // the wave's FP64 sums: in LDS, read and written once per tile
    double *out = lds_raw + (size_t)wave * NO * 64 + lane;
#pragma unroll
    for (int a = 0; a < NO; ++a) out[a * 64] = 0.0;
    T acc[NA];
#pragma unroll
    for (int a = 0; a < NA; ++a) acc[a] = T(0);

    vec *tile = (vec *)(lds_raw + TRI_WAVES * NO * 64) + wave * NVEC;
    const T *tw = (const T *)tile;
    vec pre[NV];
    const TriShare sh = tri_share(wave, t0, t1);
    {
        const int tf = sh.first < t1 ? sh.first : t0;      // a chunk holds a tile
        const vec *src = (const vec *)(g.rec + (size_t)tf * TT * RW);
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const int e = v * 64 + lane;
            pre[v] = src[e < NVEC ? e : NVEC - 1];
        }
    }
    for (int t = sh.first; t < t1; t += sh.step) {
        const int real = min(TT, n_src - t * TT), j0 = sh.j0(real), j1 = sh.j1(real);
        if (j0 == j1) break;   // fewer triangles than parts: nothing for this wave
        wave_lds_order();
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const int e = v * 64 + lane;
            if (e < NVEC) tile[e] = pre[v];
        }
        wave_lds_order();
        {
            const int tn = t + sh.step < t1 ? t + sh.step : t;
            const vec *src = (const vec *)(g.rec + (size_t)tn * TT * RW);
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                const int e = v * 64 + lane;
                pre[v] = src[e < NVEC ? e : NVEC - 1];
            }
        }
        // an index the compiler cannot see through: it would otherwise move
        // these loads out of the loop and hold their registers through it
        int ii = i;
        asm volatile("" : "+v"(ii));
        double org[3], dd[3];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            org[d] = g.src_org[3 * t + d];
            dd[d] = org[d] - g.obs_org[(size_t)d * n_obs_pad + ii];
        }
        const bool close = dd[0] * dd[0] + dd[1] * dd[1] + dd[2] * dd[2] <= g.sep2;
        if constexpr (F32)
#pragma unroll
            for (int p = 0; p < NQ; ++p)
#pragma unroll
                for (int d = 0; d < 3; ++d)
                    x[p][d] = (T)(g.obs[(size_t)(3 * p + d) * n_obs_pad + ii] - org[d]);
        const bool mask = __any(close);
        TriHead<KID, T> h;
        tri_head<KID, NQ, T>(tw + j0 * RW, h);
        // one triangle per step: two (no register copies between a record's
        // head and the next one's) measured 2-9% slower
        // RA in FP32: the sums that its observation points share, folded after
        // each triangle pair: through a whole tile they would be 48 and 144
        // terms long with three points, where the point form adds 64 (median
        // error 1.33 times its, 1.00 with this; 32,256 triangles 4.12 -> 4.26 ms)
        T ra[3] = {T(0), T(0), T(0)};
        auto fold_ra = [&]() {
            if constexpr (F32 && KID == TCT_RA)
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    ra[d] = ra[d] + fma_t(k.c0, acc[d], k.c1 * acc[3 + d]);
                    acc[d] = acc[3 + d] = T(0);
                }
        };
        int j = j0;
        if (tri_always_masked<KID, NQ, T>() || mask) {
#pragma unroll 1
            do {
                tri_pair<KID, NQ, T, true>(x, m, tw + j * RW, tw + min(j + 1, TT - 1) * RW, k, h,
                                           acc);
                fold_ra();
            } while (++j < j1);
        } else {
#pragma unroll 1
            do {
                tri_pair<KID, NQ, T, false>(x, m, tw + j * RW, tw + min(j + 1, TT - 1) * RW, k,
                                            h, acc);
                fold_ra();
            } while (++j < j1);
        }
        if constexpr (F32) {
            T o[NO];
            tri_fold<KID, NQ, T>(m, k, acc, o);
            if constexpr (KID == TCT_RA)
#pragma unroll
                for (int d = 0; d < 3; ++d) o[d] = ra[d];
#pragma unroll
            for (int a = 0; a < NO; ++a) out[a * 64] += (double)o[a];
#pragma unroll
            for (int a = 0; a < NA; ++a) acc[a] = T(0);
        }
    }
    if constexpr (!F32) {
        T o[NO];
        tri_fold<KID, NQ, T>(m, k, acc, o);
#pragma unroll
        for (int a = 0; a < NO; ++a) out[a * 64] = o[a];
    }
    __syncthreads();
    const double *red = lds_raw;
    double *po = g.partial + (size_t)ch * NO * n_obs_pad + ob * 64;
    for (int e = (int)threadIdx.x; e < NO * 64; e += 64 * TRI_WAVES) {
        double s = red[e];
#pragma unroll
        for (int w = 1; w < TRI_WAVES; ++w) s += red[w * NO * 64 + e];
        po[(size_t)(e >> 6) * n_obs_pad + (e & 63)] = s;
    }
}

// Launches the N-bodies of the problems of a table (one kernel, rule and
// precision), and the workgroups of such a launch that a CU holds (defined
// in far_tri_f32.hip and far_tri_f64.hip).
template <typename T>
int far_tri_launch(int kernel, int nq, const double *params, const double *qw,
                   const TriSegTable<T> &t, unsigned blocks, hipStream_t st);
template <typename T>
int far_tri_resident(int kernel, int nq, int *blocks);

template <int KID, int NQ, typename T>
inline hipError_t far_tri_occ(int *blocks) {
    const size_t lds = tri_lds_bytes<KID, NQ, T>();
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(
        blocks, (const void *)far_tri_kernel<KID, NQ, T>, 64 * TRI_WAVES, lds);
}

template <int KID, int NQ, typename T>
inline void far_tri_go(const double *params, const double *qw, const TriSegTable<T> &t,
                       unsigned blocks, hipStream_t st) {
    const KConst<T> kc = kernel_consts<T>(KID, params, 0.0);
    TriConst<T> k{kc.c0, kc.c1, kc.c2, kc.c3, kc.c4, T(0), T(1), T(1), kc.c0};
    if (KID == TCT_RA) {
        const ElasticConsts c = elastic_consts(params);
        k.c0 = (T)c.CsRT1;
        k.c1 = (T)c.CsRT0;
    }
    if (NQ == 4) {
        const double rw = qw[0] / qw[NQ - 1];
        k.rw = (T)rw;
        k.rw2 = (T)(rw * rw);
        k.rwc = (T)(kc.c0 * rw);
    }
    const unsigned lds = (unsigned)tri_lds_bytes<KID, NQ, T>();
    hipLaunchKernelGGL((far_tri_kernel<KID, NQ, T>), dim3(blocks), dim3(64 * TRI_WAVES), lds, st,
                       t, k);
}

template <int NQ, typename T>
inline void far_tri_kid(int kernel, const double *params, const double *qw,
                        const TriSegTable<T> &t, unsigned blocks, hipStream_t st) {
    switch (kernel) {
    case TCT_U: far_tri_go<TCT_U, NQ, T>(params, qw, t, blocks, st); break;
    case TCT_T: far_tri_go<TCT_T, NQ, T>(params, qw, t, blocks, st); break;
    case TCT_A: far_tri_go<TCT_A, NQ, T>(params, qw, t, blocks, st); break;
    case TCT_H: far_tri_go<TCT_H, NQ, T>(params, qw, t, blocks, st); break;
    case TCT_RT: far_tri_go<TCT_RT, NQ, T>(params, qw, t, blocks, st); break;
    case TCT_RA: far_tri_go<TCT_RA, NQ, T>(params, qw, t, blocks, st); break;
    default: far_tri_go<TCT_RH, NQ, T>(params, qw, t, blocks, st); break;
    }
}

template <int NQ, typename T>
inline hipError_t far_tri_occ_kid(int kernel, int *blocks) {
    switch (kernel) {
    case TCT_U: return far_tri_occ<TCT_U, NQ, T>(blocks);
    case TCT_T: return far_tri_occ<TCT_T, NQ, T>(blocks);
    case TCT_A: return far_tri_occ<TCT_A, NQ, T>(blocks);
    case TCT_H: return far_tri_occ<TCT_H, NQ, T>(blocks);
    case TCT_RT: return far_tri_occ<TCT_RT, NQ, T>(blocks);
    case TCT_RA: return far_tri_occ<TCT_RA, NQ, T>(blocks);
    default: return far_tri_occ<TCT_RH, NQ, T>(blocks);
    }
}

template <typename T>
inline int far_tri_occ_nq(int kernel, int nq, int *blocks) {
    const hipError_t e = nq == 3 ? far_tri_occ_kid<3, T>(kernel, blocks)
                                 : far_tri_occ_kid<4, T>(kernel, blocks);
    if (e != hipSuccess)
        return set_error(TCT_EHIP, "far_tri: occupancy: %s", hipGetErrorString(e));
    return TCT_OK;
}

template <typename T>
inline int far_tri_nq(int kernel, int nq, const double *params, const double *qw,
                      const TriSegTable<T> &t, unsigned blocks, hipStream_t st) {
    if (nq == 3)
        far_tri_kid<3, T>(kernel, params, qw, t, blocks, st);
    else if (nq == 4)
        far_tri_kid<4, T>(kernel, params, qw, t, blocks, st);
    else
        return set_error(TCT_EUNSUPPORTED, "far_tri: rule of %d points (3 or 4)", nq);
    TCT_CHECK_LAUNCH("far_tri");
    return TCT_OK;
}

}  // namespace tct
