// Device code shared by the pair integrators (pairs.hip, interior.hip):
// the source/observation triangle record, its set-up with rotation and
// flip, and the 3x3 kernel tensors.
#pragma once

#include "tct_common.h"

namespace tct {

struct Tri {
    double v[3][3];              // vertices in the rotated frame
    double n[3];                 // unit normal
    double jac;                  // |unscaled normal| = 2 * area
    double curl[3][3];           // surface curl of the basis functions
};

// Vectors at their elements' alignment.
typedef double d2u __attribute__((ext_vector_type(2), aligned(8)));
typedef int i3u __attribute__((ext_vector_type(3), aligned(4)));

__device__ __forceinline__ int pmod3(int i) { return ((i % 3) + 3) % 3; }

// tri_info of tectosaur/integral_primitives.cl:56-93 (+ surf_curl_basis
// :95-112): vertex c of the rotated triangle is original vertex
// (flip(c) + clicks) mod 3; the flip also negates the unscaled normal.
__device__ __forceinline__ void load_tri(Tri &t, const double *__restrict__ pts,
                                         const int32_t *__restrict__ tris, int idx, int clicks,
                                         int flip) {
    // every lane gathers from lines of its own, one line a cycle: the three
    // indices come in one load and a point in two
    const i3u id = *(const i3u *)(tris + 3 * (size_t)idx);
    double v[3][3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        int fc = c;
        if (flip) fc = (c == 0) ? 1 : (c == 1 ? 0 : 2);
        const int r = pmod3(fc + clicks);
        const int p = r == 0 ? id.x : (r == 1 ? id.y : id.z);
        const d2u xy = *(const d2u *)(pts + 3 * (size_t)p);
        v[c][0] = xy.x;
        v[c][1] = xy.y;
        v[c][2] = pts[3 * (size_t)p + 2];
    }
    double s20[3], s21[3], un[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        s20[d] = v[2][d] - v[0][d];
        s21[d] = v[2][d] - v[1][d];
    }
    un[0] = s20[1] * s21[2] - s20[2] * s21[1];
    un[1] = s20[2] * s21[0] - s20[0] * s21[2];
    un[2] = s20[0] * s21[1] - s20[1] * s21[0];
    if (flip)
#pragma unroll
        for (int d = 0; d < 3; ++d) un[d] = -un[d];
    t.jac = sqrt(un[0] * un[0] + un[1] * un[1] + un[2] * un[2]);
    const double inv = 1.0 / t.jac;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        t.n[d] = un[d] * inv;
#pragma unroll
        for (int c = 0; c < 3; ++c) t.v[c][d] = v[c][d];
    }
    // grad of (1-x-y, x, y) = (-1,-1), (1,0), (0,1); curl_b = (g_b0 e2 - g_b1 e1) / J
    // with e1 = v1 - v0, e2 = v2 - v0.
#pragma unroll
    for (int s = 0; s < 3; ++s) {
        const double e1 = v[1][s] - v[0][s], e2 = v[2][s] - v[0][s];
        t.curl[0][s] = (-e2 + e1) * inv;
        t.curl[1][s] = e2 * inv;
        t.curl[2][s] = -e1 * inv;
    }
}

// The Jacobian and surface curls of a triangle (rotated, flipped vertex
// order) from its edges e1 = v1 - v0, e2 = v2 - v0; the vertices and the
// normal stay unset.
__device__ __forceinline__ void tri_from_edges(Tri &t, const double (&e1)[3],
                                               const double (&e2)[3]) {
    const double n0 = e1[1] * e2[2] - e1[2] * e2[1], n1 = e1[2] * e2[0] - e1[0] * e2[2],
                 n2 = e1[0] * e2[1] - e1[1] * e2[0];
    t.jac = sqrt(n0 * n0 + n1 * n1 + n2 * n2);
    const double inv = 1.0 / t.jac;
#pragma unroll
    for (int s = 0; s < 3; ++s) {
        t.curl[0][s] = (e1[s] - e2[s]) * inv;
        t.curl[1][s] = e2[s] * inv;
        t.curl[2][s] = -e1[s] * inv;
    }
}

// Number of accumulators per kernel class.
template <int KID>
constexpr int n_acc() {
    return KID <= TCT_H ? 81 : (KID == TCT_RH ? 7 : 30);
}

// 3x3 kernel tensor (tectosaur/kernels/__init__.py tensor_code), m = obs
// normal, n = src normal, D = y - x.
// invr = 1/r, or 0 to drop the point (every entry is then 0).
template <int KID>
__device__ __forceinline__ void tensor_invr(const double D[3], double invr, const double m[3],
                                            const double n[3], const ElasticConsts &c,
                                            double K[9]) {
    const double invr2 = invr * invr;
    const double invr3 = invr2 * invr;
    if constexpr (KID == TCT_U) {
        const double Q1 = c.CsU0 * invr, Q2 = c.CsU1 * invr3;
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j) K[i * 3 + j] = Q2 * D[i] * D[j] + (i == j ? Q1 : 0.0);
    } else if constexpr (KID == TCT_T || KID == TCT_A) {
        // K = A(-(N.D) I + s W) + C (N.D) D D^T with W the cross-product
        // matrix of N x D (sign s = +1 for T, -1 for A).
        const double *N = KID == TCT_T ? n : m;
        const double s = KID == TCT_T ? 1.0 : -1.0;
        const double rn = N[0] * D[0] + N[1] * D[1] + N[2] * D[2];
        const double A = s * c.CsT0 * invr3;
        const double C = -s * c.CsT1 * invr3 * invr2;
        const double cx = N[1] * D[2] - N[2] * D[1];
        const double cy = N[2] * D[0] - N[0] * D[2];
        const double cz = N[0] * D[1] - N[1] * D[0];
        const double As = A * s;
        K[0] = -A * rn + C * rn * D[0] * D[0];
        K[1] = -As * cz + C * rn * D[0] * D[1];
        K[2] = As * cy + C * rn * D[0] * D[2];
        K[3] = As * cz + C * rn * D[1] * D[0];
        K[4] = -A * rn + C * rn * D[1] * D[1];
        K[5] = -As * cx + C * rn * D[1] * D[2];
        K[6] = -As * cy + C * rn * D[2] * D[0];
        K[7] = As * cx + C * rn * D[2] * D[1];
        K[8] = -A * rn + C * rn * D[2] * D[2];
    } else {
        const double Dr[3] = {D[0] * invr, D[1] * invr, D[2] * invr};
        const double rn = n[0] * Dr[0] + n[1] * Dr[1] + n[2] * Dr[2];
        const double rm = m[0] * Dr[0] + m[1] * Dr[1] + m[2] * Dr[2];
        const double mn = m[0] * n[0] + m[1] * n[1] + m[2] * n[2];
        const double Q = c.CsH0 * invr3;
        const double A = Q * 3.0 * rn;
        const double B = Q * c.CsH1;
        const double C = Q * c.CsH3;
        double MT[3], NT[3], DT[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            MT[k] = Q * c.CsH2 * n[k] + A * c.CsH1 * Dr[k];
            NT[k] = B * m[k] + C * Dr[k] * rm;
            DT[k] = B * 3.0 * n[k] * rm + C * Dr[k] * mn + A * (c.nu * m[k] - 5.0 * Dr[k] * rm);
        }
        const double ST = A * c.nu * rm + B * mn;
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j)
                K[i * 3 + j] = n[i] * NT[j] + m[i] * MT[j] + Dr[i] * DT[j] + (i == j ? ST : 0.0);
    }
}

template <int KID>
__device__ __forceinline__ void tensor(const double D[3], double r2, const double m[3],
                                       const double n[3], const ElasticConsts &c,
                                       double K[9]) {
    tensor_invr<KID>(D, rsqrt(r2), m, n, c, K);
}

// Symmetric index of (p, t) in 6-vector order xx, xy, xz, yy, yz, zz.
__device__ __forceinline__ constexpr int sym6(int p, int t) {
    return p <= t ? (p == 0 ? t : (p == 1 ? 2 + t : 5)) : (t == 0 ? p : (t == 1 ? 2 + p : 5));
}

// Levi-Civita symbol of (i, j, k) in {0,1,2}^3.
__device__ __forceinline__ int levi(int i, int j, int k) { return (i - j) * (j - k) * (k - i) / 2; }

// The r = 0 test of a pair class (CK): CK_NONE for pairs that never touch;
// CK_FULL skips r2 == 0 and the points whose obs and src parameters are
// equal on pairs that are one triangle in one frame; CK_R2 skips r2 == 0
// only, for rules with no point of equal obs and src parameters.
constexpr int CK_NONE = 0, CK_FULL = 1, CK_R2 = 2;

// Normals a kernel body reads: obs (m) and src (n).
struct PairNormals {
    double m[3], n[3];
};

// ---------------------------------------------------------------------------
// From a pair's sums to its 81 outputs.  Memory wants whole lines: rows of
// 648 bytes written lane by lane, or in runs of 72 or 216 bytes, reached
// 2.2 to 2.5 TB/s, whole rows one after another 5.3 (710,704 rows).  So a wave
// puts what its pairs' outputs are made of in LDS, a few pairs at a time, and
// its lanes then form the outputs in the order of memory, each from a few
// LDS words at offsets that a table gives for the 81 entries.
//
// The formulas (integral_primitives.cl:174-213, kernels.cl:29-98), with the
// factor J = J_obs J_src in the packed sums, obs basis b, src basis e,
// components d (obs) and f (src), curls o (obs) and s (src):
//   U       sum[b][e][d f]
//   T, A, H sum[b][d][e][f]
//   RH      P[d f] (o_b . s_e) + A_bd s_ef + B_bf s_ed with P = -2 c0 (S2 +
//           S0 I), A = c0 CsRH1 S0 o, B = c0 CsRH2 S0 o
//   RT      C[b][d, f+2] s_e,f+1 - C[b][d, f+1] s_e,f+2 + (d = f) A3[b][e],
//           C[b] = A2[b] + A1[b] I (the Levi-Civita sums written out)
//   RA      the same with the sides exchanged and -A3.
struct PairTable {
    uint2 off[81];   // six byte-sized offsets per entry
};

// T, A and H: what is in LDS are the 81 entries themselves; no table.
template <int KID>
constexpr bool pair_tensor() { return KID == TCT_T || KID == TCT_A || KID == TCT_H; }

// Doubles of one pair in LDS.
template <int KID>
constexpr int pack_size() {
    return KID == TCT_U ? 54 : (KID <= TCT_H ? 81 : (KID == TCT_RH ? 42 : 37));
}
// Pairs in LDS at a time (GL lanes a pair).
template <int KID, int GL>
constexpr int pack_pairs() {
    return 64 / GL < 16 ? 64 / GL : 16;
}

// Filled by the first 81 threads of a workgroup (a barrier before its use).
template <int KID>
__device__ __forceinline__ void fill_pair_table(PairTable &t) {
    if constexpr (pair_tensor<KID>()) return;
    for (int i = (int)threadIdx.x; i < 81; i += (int)blockDim.x) {
        const int b = i / 27, d = i / 9 % 3, e = i / 3 % 3, f = i % 3;
        int o[6] = {0, 0, 0, 0, 0, 0};
        if constexpr (KID == TCT_U) {
            o[0] = (3 * b + e) * 6 + sym6(d, f);
        } else if constexpr (KID <= TCT_H) {
            o[0] = i;
        } else if constexpr (KID == TCT_RH) {
            // P 0-5, o.s 6-14, A 15-23, B 24-32, s 33-41
            o[0] = sym6(d, f);
            o[1] = 6 + 3 * b + e;
            o[2] = 15 + 3 * b + d;
            o[3] = 33 + 3 * e + f;
            o[4] = 24 + 3 * b + f;
            o[5] = 33 + 3 * e + d;
        } else {
            // C 0-17, A3 18-26, curls 27-35, zero 36
            const int cb = KID == TCT_RT ? b : e, cd = KID == TCT_RT ? d : f;   // side of C
            const int xb = KID == TCT_RT ? e : b, xd = KID == TCT_RT ? f : d;   // side of the curl
            o[0] = 6 * cb + sym6(cd, (xd + 2) % 3);
            o[1] = 27 + 3 * xb + (xd + 1) % 3;
            o[2] = 6 * cb + sym6(cd, (xd + 1) % 3);
            o[3] = 27 + 3 * xb + (xd + 2) % 3;
            o[4] = d == f ? 18 + 3 * b + e : 36;
        }
        t.off[i] = make_uint2(o[0] | o[1] << 8 | o[2] << 16 | o[3] << 24, o[4] | o[5] << 8);
    }
}

template <int KID>
__device__ __forceinline__ double pair_entry(const double *p, uint2 o) {
    if constexpr (KID <= TCT_H) {
        return p[o.x];
    } else {
        const double a = p[o.x & 255], b = p[o.x >> 8 & 255], c = p[o.x >> 16 & 255],
                     d = p[o.x >> 24], e = p[o.y & 255];
        if constexpr (KID == TCT_RH)
            return fma(e, p[o.y >> 8 & 255], fma(c, d, a * b));
        else
            return fma(a, b, e) - c * d;
    }
}

// What the outputs of one pair are made of, from its sums `acc` (rotated
// frame: bases in the integrator's order) into p (bases in the caller's order:
// the de-rotation of assemble.cl:77-101, out[b1] = res[od[b1]] with od[i] =
// (i - clicks) mod 3, entries 0 and 1 of the source map swapped when the
// source was flipped).
template <int KID>
__device__ __forceinline__ void pack_pair(const double *acc, const Tri &ot, const Tri &st,
                                          const ElasticConsts &c, int oc, int sc, int flip,
                                          double *p) {
    int oi[3], si[3];   // caller's position of each basis
    {
        int sd[3];
#pragma unroll
        for (int i = 0; i < 3; ++i) sd[i] = pmod3(i - sc);
        if (flip) {
            const int tmp = sd[0];
            sd[0] = sd[1];
            sd[1] = tmp;
        }
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            oi[i] = pmod3(i + oc);
            si[i] = (sd[0] == i) ? 0 : ((sd[1] == i) ? 1 : 2);
        }
    }
    const double J = ot.jac * st.jac;
    if constexpr (KID == TCT_U) {
#pragma unroll
        for (int b = 0; b < 3; ++b)
#pragma unroll
            for (int e = 0; e < 3; ++e)
#pragma unroll
                for (int d = 0; d < 3; ++d)
#pragma unroll
                    for (int f = d; f < 3; ++f)
                        p[(3 * oi[b] + si[e]) * 6 + sym6(d, f)] =
                            J * acc[b * 27 + d * 9 + e * 3 + f];
    } else if constexpr (KID <= TCT_H) {
#pragma unroll
        for (int b = 0; b < 3; ++b)
#pragma unroll
            for (int d = 0; d < 3; ++d)
#pragma unroll
                for (int e = 0; e < 3; ++e)
#pragma unroll
                    for (int f = 0; f < 3; ++f)
                        p[oi[b] * 27 + d * 9 + si[e] * 3 + f] =
                            J * acc[b * 27 + d * 9 + e * 3 + f];
    } else if constexpr (KID == TCT_RH) {
        const double c0 = J * c.CsRH0, s0 = c0 * acc[0];
#pragma unroll
        for (int d = 0; d < 3; ++d)
#pragma unroll
            for (int f = d; f < 3; ++f) {
                const double s2 = c0 * acc[1 + sym6(d, f)];
                p[sym6(d, f)] = -2.0 * (d == f ? s2 + s0 : s2);
            }
#pragma unroll
        for (int b = 0; b < 3; ++b) {
#pragma unroll
            for (int e = 0; e < 3; ++e)
                p[6 + 3 * oi[b] + si[e]] = ot.curl[b][0] * st.curl[e][0] +
                                           ot.curl[b][1] * st.curl[e][1] +
                                           ot.curl[b][2] * st.curl[e][2];
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                p[15 + 3 * oi[b] + d] = s0 * c.CsRH1 * ot.curl[b][d];
                p[24 + 3 * oi[b] + d] = s0 * c.CsRH2 * ot.curl[b][d];
                p[33 + 3 * si[b] + d] = st.curl[b][d];
            }
        }
    } else {
        const int *ci = KID == TCT_RT ? oi : si;   // side of the weights
        const int *xi = KID == TCT_RT ? si : oi;   // side of the curls
        const Tri &x = KID == TCT_RT ? st : ot;
#pragma unroll
        for (int b = 0; b < 3; ++b) {
#pragma unroll
            for (int d = 0; d < 3; ++d)
#pragma unroll
                for (int f = d; f < 3; ++f) {
                    const double a2 = acc[3 + 6 * b + sym6(d, f)];
                    p[6 * ci[b] + sym6(d, f)] = J * (d == f ? a2 + acc[b] : a2);
                }
#pragma unroll
            for (int e = 0; e < 3; ++e)
                p[18 + 3 * oi[b] + si[e]] = (KID == TCT_RT ? J : -J) * acc[21 + 3 * b + e];
#pragma unroll
            for (int d = 0; d < 3; ++d) p[27 + 3 * xi[b] + d] = x.curl[b][d];
        }
        p[36] = 0.0;
    }
}

// The output row of a pair: rows[pair], or the pair itself.
__device__ __forceinline__ int out_row(const int32_t *__restrict__ rows, int pair) {
    return rows ? rows[pair] : pair;
}

// Entries in flight at a time: as many as leave a kernel's waves per SIMD as
// they are (T, A and H read one LDS word an entry, the others three to seven).
template <int KID, int GL>
constexpr int write_unroll() {
    return KID == TCT_RH && GL >= 4 ? 7 : (KID == TCT_U || KID > TCT_H ? 2 : 11);
}

// LDS of one wave.
template <int KID, int GL>
struct PairStage {
    double v[pack_pairs<KID, GL>() * pack_size<KID>()];
    int row[pack_pairs<KID, GL>()];   // output row (-1: none)
};

// The outputs of the 64 / GL pairs of one wave.  Every lane of the wave
// calls it; the GL lanes of pair pl, of which `writer` has the sums.
// pack(p) puts the pair's sums in LDS (pack_pair).  SUB: subtracted from what
// is there instead of written.  UN entries a lane are formed at a time
// (write_unroll).  Where few waves run this latency is what a launch adds: 8 pairs
// at a time, an entry after another, made 16 points of T on 1,000 pairs take 29 us;
// 16 pairs and all their entries in flight 24, with four lanes a pair 15.
template <int KID, int GL, bool SUB, int UN, typename F>
__device__ __forceinline__ void write_pairs(F &&pack, const PairTable &tab,
                                            PairStage<KID, GL> &sg, int pl, bool writer, int row,
                                            double *__restrict__ out) {
    constexpr int PW = 64 / GL, SP = pack_pairs<KID, GL>(), ND = pack_size<KID>();
    constexpr unsigned NE = SP * 81;
    constexpr int NI = (NE + 63) / 64;
    const int lane = (int)threadIdx.x & 63;
#pragma unroll 1
    for (int h = 0; h < PW / SP; ++h) {
        wave_lds_order();
        if (writer && pl / SP == h) {
            pack(&sg.v[(pl % SP) * ND]);
            sg.row[pl % SP] = row;
        }
        wave_lds_order();
        auto put = [&](int p, int i, double x) {
            const int r = sg.row[p];
            if (r >= 0) {
                double *o = out + (size_t)r * 81 + i;
                *o = SUB ? *o - x : x;
            }
        };
        if constexpr (UN > 2) {
            // entry i of pair p: p * 81 + i = lane + 64 k
#pragma unroll UN
            for (int k = 0; k < NI; ++k) {
                const unsigned e = lane + 64u * k;
                if (k == NI - 1 && e >= NE) break;
                const unsigned p = e / 81u, i = e - 81u * p;
                if constexpr (pair_tensor<KID>())
                    put(p, i, sg.v[e]);      // the entries themselves
                else
                    put(p, i, pair_entry<KID>(&sg.v[p * ND], tab.off[i]));
            }
        } else {
            int p = 0, i = lane;
#pragma unroll UN
            for (unsigned e = lane; e < NE; e += 64) {
                put(p, i, pair_entry<KID>(&sg.v[p * ND], tab.off[i]));
                i += 64;
                if (i >= 81) {
                    i -= 81;
                    ++p;
                }
            }
        }
    }
}

}  // namespace tct
