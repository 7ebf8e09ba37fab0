// Triangle-to-point farfield in FP32: source triangles against observation
// points (U, T, A, H).
//
// Reference semantics: farfield_tris_to_pts{K} (tectosaur/interior.py:139-185
// on tectosaur/matrix_free.cl) with the kernel bodies of tectosaur/kernels/
// kernels.cl: every source quadrature point against every observation point,
// pairs at r2 == 0 skipped.
//
// What bounds it: VALU issue, as the triangle-to-triangle N-body of far_tri.h,
// whose records and tile walk it shares.  A lane holds one observation point
// and walks whole source triangles: n . D and m . n are formed once per
// triangle and terms along n are summed as scalars over it.  Every tile runs
// with the r2 test: a body without it for far tiles was no faster (U 396 us
// with, 406 without; T 484 and 487; seven points, below).
// 62,500 points x 2,048 triangles, us, point form (far_p2p.hip, its sums and
// the permutation of its outputs) -> this:
//   3 points  U 240 -> 177, T 291 -> 224, A 272 -> 238, H 445 -> 336
//   4 points  U 300 -> 221, T 371 -> 284, A 345 -> 305, H 574 -> 428
//   7 points  U 482 -> 377, T 615 -> 464, A 570 -> 518
// Two, three and four points a lane (fewer LDS reads a pair) were slower: U
// 421, 428 and 438, T 518, 557 and 557 with seven rule points.
#include "far_tri.h"

namespace tct {

struct PtsRule {
    double qw[7], phi[21];
};

// Source triangles per tile: as many whole ones as have at most 64 points, up
// to TCT_TRI_TILE.  A tile has one origin and one FP32 sum, so its size sets the
// rounding of the points and of the sums; 64 points is the point form's.  (Tiles
// of 16 triangles with seven points, 112: at points next to a fault of 2,048
// triangles T's and A's median error grew 1.2 to 1.3 times.)
constexpr int pts_tile(int nq) { return nq == 7 ? 9 : TT; }

template <int KID>
constexpr int pts_acc() { return KID == TCT_U ? 6 : (KID == TCT_A ? 4 : (KID == TCT_H ? 5 : 3)); }

// One observation point x (normal m) against one source triangle (record r,
// in LDS, its head already in h): acc += its terms, h becomes the head of the
// record `next`.  One fence per source point: without, T with seven rule
// points takes 520 us in place of 502, U 426 in place of 399.
template <int KID, int NS>
__device__ __forceinline__ void pts_pair(const float (&x)[3], const float (&m)[3], const float *r,
                                         const float *next, const TriConst<float> &k,
                                         TriHead<KID, float> &h, float (&acc)[pts_acc<KID>()]) {
#pragma clang fp contract(off)
    typedef float T;
    constexpr int SW = tri_sw<KID>();
    T an = T(0), ca = T(0), nt = T(0), mn0 = T(0), mn1 = T(0);
    const T n[3] = {h.n[0], h.n[1], h.n[2]};
#pragma unroll
    for (int j = 0; j < NS; ++j) {
        T q[SW];
#pragma unroll
        for (int w = 0; w < SW; ++w) q[w] = h.q[w];
        if (j + 1 < NS)
            tri_load<SW, T>(r, SW * (j + 1), h.q);
        else
            tri_head<KID, NS, T>(next, h);
        const T *s = q + 3;
        const T D[3] = {q[0] - x[0], q[1] - x[1], q[2] - x[2]};
        const T r2 = dot3(D[0], D[1], D[2], D[0], D[1], D[2]);
        const T invr = rsq_masked(r2, k.eps2);
        const T w = invr * invr;
        const T i3 = invr * w;
        if constexpr (tri_src_normal<KID>())
            if (j == 0) {
                an = dot3(n[0], n[1], n[2], D[0], D[1], D[2]);
                if constexpr (KID == TCT_T) ca = -k.c0 * an;
                if constexpr (KID == TCT_H) {
                    const T mn = dot3(m[0], m[1], m[2], n[0], n[1], n[2]);
                    mn0 = k.c0 * mn;
                    mn1 = k.c1 * mn;
                }
            }
        if constexpr (KID == TCT_U) {
            add3(acc, invr, s);
            add3(acc + 3, i3 * dot3(D[0], D[1], D[2], s[0], s[1], s[2]), D);
        } else if constexpr (KID == TCT_T) {
            const T ds = dot3(D[0], D[1], D[2], s[0], s[1], s[2]);
            nt = j == 0 ? i3 * ds : fma_t(i3, ds, nt);
            add3(acc, i3 * ca, s);
            add3(acc, i3 * fma_t(-(w * an), ds, k.c0 * q[6]), D);
        } else if constexpr (KID == TCT_A) {
            const T ds = dot3(D[0], D[1], D[2], s[0], s[1], s[2]);
            acc[3] = fma_t(i3, ds, acc[3]);
            const T bm = dot3(m[0], m[1], m[2], D[0], D[1], D[2]);
            const T sm = dot3(m[0], m[1], m[2], s[0], s[1], s[2]);
            add3(acc, i3 * fma_t(w * bm, ds, k.c0 * sm), D);
            add3(acc, i3 * (k.c0 * bm), s);
        } else {
            const T bm = dot3(m[0], m[1], m[2], D[0], D[1], D[2]);
            const T wa = w * an;
            add3(acc, i3 * fma_t(wa, k.c4 * bm, mn0), s);
            acc[3] = fma_t(i3, q[6], acc[3]);
            const T ds = dot3(D[0], D[1], D[2], s[0], s[1], s[2]);
            acc[4] = fma_t(i3, wa * ds, acc[4]);
            const T wbc = (w * bm) * ds;
            const T sm = dot3(m[0], m[1], m[2], s[0], s[1], s[2]);
            const T ni = fma_t(k.c0, sm, k.c1 * wbc);
            nt = j == 0 ? i3 * ni : fma_t(i3, ni, nt);
            const T inner = fma_t(k.c4, sm, T(-15) * wbc);
            add3(acc, (i3 * w) * fma_t(an, inner, fma_t(ds, mn1, q[7] * bm)), D);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (tri_src_normal<KID>()) add3(acc, KID == TCT_T ? -k.c0 * nt : nt, n);
}

template <int KID>
__device__ __forceinline__ void pts_fold(const float (&m)[3], const TriConst<float> &k,
                                         const float *a, float (&o)[3]) {
#pragma clang fp contract(off)
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        if constexpr (KID == TCT_U)
            o[d] = fma_t(k.c0, a[d], a[3 + d]);
        else if constexpr (KID == TCT_A)
            o[d] = fma_t(m[d], -k.c0 * a[3], a[d]);
        else if constexpr (KID == TCT_H)
            o[d] = fma_t(m[d], fma_t(k.c2, a[4], a[3]), a[d]);
        else
            o[d] = a[d];
    }
}

template <int KID, int NS>
constexpr size_t pts_lds_bytes() {
    return TRI_WAVES *
           (sizeof(double) * 64 * 3 + sizeof(float) * pts_tile(NS) * tri_words<KID, NS>());
}

// A workgroup of four waves holds 64 observation points (one a lane, the same
// in every wave) and one chunk of the source tiles, as in far_tri_kernel: wave
// w takes tiles w, w + 4, ... through its own LDS tile, FP32 sums within a
// tile, FP64 across them, the four waves' sums added in wave order.  The 64
// points have one FP64 origin and are moved to a tile's frame as in
// far_p2p_f32_kernel; with four rule points a tile holds 64 source points, the
// same as there, and every D is the same bit for bit, with three and seven its
// frame is a little smaller (48 and 63 points).  (A point next to the
// surface has large far-rule terms that the near blocks take off again: what
// is left of them is D's rounding.)
// obs [6][n_pad]: local points, normals; obs_org [n_pad / 64][3];
// partial [chunks][3][n_pad].
template <int KID, int NS>
__global__ __launch_bounds__(64 * TRI_WAVES) void tri_pts_kernel(
    int n_pad, int n_src, int n_tiles, int chunks, const float *__restrict__ obs,
    const double *__restrict__ obs_org, const float *__restrict__ rec,
    const double *__restrict__ src_org, TriConst<float> kc,
    double *__restrict__ partial) {
    typedef float vec __attribute__((ext_vector_type(4)));
    constexpr int TP = pts_tile(NS);
    constexpr int RW = tri_words<KID, NS>(), NO = 3;
    constexpr int NVEC = TP * RW / 4, NV = (NVEC + 63) / 64;
    static_assert(TP * RW % 4 == 0 && TP * NS <= 64, "whole vectors, at most 64 points");
    extern __shared__ double lds_raw[];
    const int obs_blocks = n_pad / 64;
    const int ob = (int)blockIdx.x % obs_blocks, ch = (int)blockIdx.x / obs_blocks;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int lane = (int)threadIdx.x & 63;
    const TriChunk tc = tri_chunk(n_tiles, chunks, ch);
    const int t0 = tc.t0, t1 = tc.t1;
    const int i = ob * 64 + lane;
    TriConst<float> k = kc;
    asm volatile("" : "+v"(k.c0), "+v"(k.c1), "+v"(k.c2), "+v"(k.c4), "+v"(k.eps2));
    float m[3], xl[3];
    double oo[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        m[d] = tri_obs_normal<KID>() ? obs[(size_t)(3 + d) * n_pad + i] : 0.0f;
        xl[d] = obs[(size_t)d * n_pad + i];
        oo[d] = obs_org[3 * ob + d];
    }
    double *out = lds_raw + (size_t)wave * NO * 64 + lane;
#pragma unroll
    for (int a = 0; a < NO; ++a) out[a * 64] = 0.0;
    vec *tile = (vec *)(lds_raw + TRI_WAVES * NO * 64) + wave * NVEC;
    const float *tw = (const float *)tile;
    vec pre[NV];
    const TriShare sh = tri_share(wave, t0, t1);
    {
        const int tf = sh.first < t1 ? sh.first : t0;      // a chunk holds a tile
        const vec *src = (const vec *)(rec + (size_t)tf * TP * RW);
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const int e = v * 64 + lane;
            pre[v] = src[e < NVEC ? e : NVEC - 1];
        }
    }
    for (int t = sh.first; t < t1; t += sh.step) {
        const int real = min(TP, n_src - t * TP), j0 = sh.j0(real), j1 = sh.j1(real);
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
            const vec *src = (const vec *)(rec + (size_t)tn * TP * RW);
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                const int e = v * 64 + lane;
                pre[v] = src[e < NVEC ? e : NVEC - 1];
            }
        }
        float x[3], acc[pts_acc<KID>()];
#pragma unroll
        for (int d = 0; d < 3; ++d) x[d] = xl[d] - (float)(src_org[3 * t + d] - oo[d]);
#pragma unroll
        for (int a = 0; a < pts_acc<KID>(); ++a) acc[a] = 0.0f;
        TriHead<KID, float> h;
        tri_head<KID, NS, float>(tw + j0 * RW, h);
        int j = j0;
#pragma unroll 1
        do
            pts_pair<KID, NS>(x, m, tw + j * RW, tw + min(j + 1, TP - 1) * RW, k, h, acc);
        while (++j < j1);
        float o[3];
        pts_fold<KID>(m, k, acc, o);
#pragma unroll
        for (int d = 0; d < 3; ++d) out[d * 64] += (double)o[d];
    }
    __syncthreads();
    double *po = partial + (size_t)ch * NO * n_pad + ob * 64;
    for (int e = (int)threadIdx.x; e < NO * 64; e += 64 * TRI_WAVES) {
        double s = lds_raw[e];
#pragma unroll
        for (int w = 1; w < TRI_WAVES; ++w) s += lds_raw[w * NO * 64 + e];
        po[(size_t)(e >> 6) * n_pad + (e & 63)] = s;
    }
}

// One wave per 64 points: their origin (the mean) and local points.
__global__ __launch_bounds__(64) void pts_pack_obs_kernel(
    int64_t n, int64_t n_pad, const double *__restrict__ pts, const double *__restrict__ ns,
    float *__restrict__ obs, double *__restrict__ org) {
    const int64_t i = (int64_t)blockIdx.x * 64 + threadIdx.x;
    const bool valid = i < n;
    double cnt = valid ? 1.0 : 0.0;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) cnt += __shfl_xor(cnt, off, 64);
    for (int d = 0; d < 3; ++d) {
        const double p = valid ? pts[3 * i + d] : 0.0;
        double o = p;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) o += __shfl_xor(o, off, 64);
        o /= cnt;
        if (threadIdx.x == 0) org[3 * blockIdx.x + d] = o;
        obs[d * n_pad + i] = valid ? (float)(p - o) : 0.0f;
        obs[(3 + d) * n_pad + i] = valid ? (float)ns[3 * i + d] : 0.0f;
    }
}

// One thread per tile and coordinate: the tile's origin (mean of its points)
// and words.  Padding triangles lie far away with zero strengths.
template <int KID, int NS>
__global__ void pts_pack_src_kernel(int64_t n, int64_t n_tiles, const double *__restrict__ pts,
                                    const double *__restrict__ ns, float *__restrict__ rec,
                                    double *__restrict__ org) {
    constexpr int TP = pts_tile(NS);
    constexpr int RW = tri_words<KID, NS>(), SW = tri_sw<KID>();
    const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= n_tiles * 3) return;
    const int64_t t = g / 3;
    const int d = (int)(g % 3);
    const int64_t k0 = t * TP;
    const int cnt = (int)(n - k0 < TP ? n - k0 : TP);
    double o = 0.0;
    for (int e = 0; e < cnt * NS; ++e) o += pts[(k0 * NS + e) * 3 + d];
    o /= cnt * NS;
    org[3 * t + d] = o;
    for (int u = 0; u < TP; ++u) {
        float *r = rec + (k0 + u) * RW;
        for (int w = d; w < RW; w += 3) {
            // strengths are zero until a gather writes them
            const int q = w / SW, c = w % SW;
            if (q >= NS || c >= 3) {
                bool nw = false;
                if constexpr (tri_src_normal<KID>())
                    for (int dd = 0; dd < 3; ++dd) nw = nw || w == tri_n_word<KID, NS>(dd);
                if (!nw) r[w] = 0.0f;
            }
        }
        for (int q = 0; q < NS; ++q)
            r[SW * q + d] = u < cnt ? (float)(pts[((k0 + u) * NS + q) * 3 + d] - o)
                                    : (float)1.0e12;
        if constexpr (tri_src_normal<KID>())
            r[tri_n_word<KID, NS>(d)] = u < cnt ? (float)ns[(k0 + u) * 3 + d] : 0.0f;
    }
}

// Strengths: one thread per (packed source triangle, rule point).
template <int KID, int NS>
__global__ __launch_bounds__(256) void pts_gather_kernel(
    int64_t n, PtsRule rule, const int32_t *__restrict__ tri, const double *__restrict__ jac,
    StrengthConsts sc, const double *__restrict__ v, float *__restrict__ rec) {
    constexpr int RW = tri_words<KID, NS>();
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t k = i / NS;
    const int q = (int)(i % NS);
    if (k >= n) return;
    float *r = rec + k * RW, *rq = r + tri_sw<KID>() * q;
    const double *vt = v + 9 * (int64_t)tri[k];
    double w = 0.0, p0 = 0.0, p1 = 0.0, p2 = 0.0;
    for (int a = 0; a < NS; ++a)
        if (a == q) {
            w = rule.qw[a];
            p0 = rule.phi[3 * a];
            p1 = rule.phi[3 * a + 1];
            p2 = rule.phi[3 * a + 2];
        }
    const double f = sc.scale * (jac[k] * w);
    double sn = 0.0;
    for (int d = 0; d < 3; ++d) {
        const double s = f * (p0 * vt[d] + p1 * vt[3 + d] + p2 * vt[6 + d]);
        rq[3 + d] = (float)s;
        if constexpr (tri_src_normal<KID>()) sn += (double)r[tri_n_word<KID, NS>(d)] * s;
    }
    if constexpr (KID == TCT_T || KID == TCT_H) rq[6] = (float)(sc.x0 * sn);
    if constexpr (KID == TCT_H) rq[7] = (float)(sc.x1 * sn);
}

// Chunk sums, into the caller's point order: thread (output, point) adds the
// partial sums in chunk order, eight loads in flight.
__global__ __launch_bounds__(192) void pts_reduce_kernel(
    int64_t n, int64_t n_pad, int chunks, const int32_t *__restrict__ pt,
    const double *__restrict__ partial, double *__restrict__ out) {
    constexpr int CI = 8;
    const int a = (int)threadIdx.x / 64;
    const int64_t i = (int64_t)blockIdx.x * 64 + threadIdx.x % 64;
    if (i >= n) return;
    const double *p = partial + (size_t)a * n_pad + i;
    const size_t stride = (size_t)3 * n_pad;
    double s = 0.0;
    int ch = 0;
    for (; ch + CI <= chunks; ch += CI) {
        double x[CI];
#pragma unroll
        for (int u = 0; u < CI; ++u) x[u] = p[(size_t)(ch + u) * stride];
#pragma unroll
        for (int u = 0; u < CI; ++u) s += x[u];
    }
    for (; ch < chunks; ++ch) s += p[(size_t)ch * stride];
    out[3 * (int64_t)pt[i] + a] = s;
}

template <int KID, int NS>
static void pts_go(const tct_tri_pts_plan &p, hipStream_t st) {
    const KConst<float> kc = kernel_consts<float>(KID, p.params, 0.0);
    const TriConst<float> k{kc.c0, kc.c1, kc.c2, kc.c3, kc.c4, (float)p.eps2, 1.0f, 1.0f, kc.c0};
    const unsigned lds = (unsigned)pts_lds_bytes<KID, NS>();
    hipLaunchKernelGGL((tri_pts_kernel<KID, NS>), dim3((unsigned)(p.n_obs_pad / 64 * p.chunks)),
                       dim3(64 * TRI_WAVES), lds, st, (int)p.n_obs_pad, (int)p.n_src, (int)p.n_tiles,
                       p.chunks, (const float *)p.obs, (const double *)p.obs_org, (const float *)p.rec,
                       (const double *)p.src_org, k, p.partial);
}

template <int KID, int NS>
static void pts_gather_go(const tct_tri_pts_plan &p, const double *v, hipStream_t st) {
    PtsRule r{};
    for (int q = 0; q < NS; ++q) {
        r.qw[q] = p.qw[q];
        for (int b = 0; b < 3; ++b) r.phi[3 * q + b] = p.phi[3 * q + b];
    }
    hipLaunchKernelGGL((pts_gather_kernel<KID, NS>),
                       dim3((unsigned)ceil_div(p.n_src * NS, (int64_t)256)), dim3(256), 0, st,
                       p.n_src, r, p.src_tri, p.src_jac, strength_consts(KID, p.params), v, p.rec);
}

template <int KID, int NS>
static void pts_pack_go(const tct_tri_pts_plan &p, const double *op, const double *on,
                        const double *sp, const double *sn, hipStream_t st) {
    hipLaunchKernelGGL(pts_pack_obs_kernel, dim3((unsigned)(p.n_obs_pad / 64)), dim3(64), 0, st,
                       p.n_pts, p.n_obs_pad, op, on, p.obs, p.obs_org);
    hipLaunchKernelGGL((pts_pack_src_kernel<KID, NS>),
                       dim3((unsigned)ceil_div(3 * p.n_tiles, (int64_t)64)), dim3(64), 0, st,
                       p.n_src, p.n_tiles, sp, sn, p.rec, p.src_org);
}

template <int KID, int NS>
static hipError_t pts_occ(int *blocks) {
    const size_t lds = pts_lds_bytes<KID, NS>();
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(
        blocks, (const void *)tri_pts_kernel<KID, NS>, 64 * TRI_WAVES, lds);
}

// H with seven points runs over points (far_p2p.hip): with tiles of 112 points,
// as they once were, 1/r^3 next to the surface left the roundings of D in the two
// forms up to 2e-5 of the result apart (770 us in place of 960); with tiles of 63 it
// has not been measured.
static bool pts_has(int kernel, int nq) {
    return kernel >= TCT_U && kernel <= TCT_H &&
           (nq == 3 || nq == 4 || (nq == 7 && kernel != TCT_H));
}

static int check_pts(const tct_tri_pts_plan *p, const char *what) {
    TCT_CHECK_ARG(p, "%s: null plan", what);
    TCT_CHECK_ARG(p->kernel >= TCT_U && p->kernel <= TCT_H, "%s: kernel id %d", what, p->kernel);
    if (!pts_has(p->kernel, p->nq))
        return set_error(TCT_EUNSUPPORTED, "%s: rule of %d points (3, 4 or 7; H: 3 or 4)", what,
                         p->nq);
    TCT_CHECK_ARG(p->n_pts > 0 && p->n_obs_pad % 64 == 0 && p->n_pts <= p->n_obs_pad &&
                      p->n_pts > p->n_obs_pad - 64 &&
                      p->n_obs_pad < (1LL << 28),
                  "%s: bad sizes n_pts=%lld n_obs_pad=%lld", what, (long long)p->n_pts,
                  (long long)p->n_obs_pad);
    const int64_t tile = pts_tile(p->nq);
    TCT_CHECK_ARG(p->n_src > 0 && p->n_tiles < (1LL << 24) && p->n_src <= p->n_tiles * tile &&
                      p->n_src > (p->n_tiles - 1) * tile,
                  "%s: bad sizes n_src=%lld n_tiles=%lld", what, (long long)p->n_src,
                  (long long)p->n_tiles);
    TCT_CHECK_ARG(p->eps2 >= 0.0 && std::isfinite(p->eps2), "%s: eps2", what);
    TCT_CHECK_ARG(p->obs && p->obs_org && p->rec && p->src_org && p->obs_pt && p->src_tri &&
                      p->src_jac,
                  "%s: null pointer", what);
    return TCT_OK;
}

#define TCT_PTS_NQ(K, nq, F)         \
    if (nq == 3) {                   \
        F(K, 3);                     \
    } else if (nq == 4) {            \
        F(K, 4);                     \
    } else {                         \
        F(K, 7);                     \
    }
#define TCT_PTS_SWITCH(kernel, nq, F)             \
    switch (kernel) {                             \
    case TCT_U: TCT_PTS_NQ(TCT_U, nq, F) break;   \
    case TCT_T: TCT_PTS_NQ(TCT_T, nq, F) break;   \
    case TCT_A: TCT_PTS_NQ(TCT_A, nq, F) break;   \
    default:                                      \
        if (nq == 3) {                            \
            F(TCT_H, 3);                          \
        } else {                                  \
            F(TCT_H, 4);                          \
        }                                         \
        break;                                    \
    }

}  // namespace tct

using namespace tct;

extern "C" int tct_tri_pts_words(int kernel, int nq) {
    if (!pts_has(kernel, nq)) return 0;
    int w = 0;
#define TCT_W(K, NS) w = tri_words<K, NS>()
    TCT_PTS_SWITCH(kernel, nq, TCT_W)
#undef TCT_W
    return w;
}

extern "C" int tct_tri_pts_tile(int kernel, int nq) {
    return pts_has(kernel, nq) ? pts_tile(nq) : 0;
}

extern "C" int tct_tri_pts_resident(int kernel, int nq, int *blocks) {
    TCT_CHECK_ARG(tct_tri_pts_words(kernel, nq) > 0, "tri_pts_resident: kernel %d, rule of %d points",
                  kernel, nq);
    TCT_CHECK_ARG(blocks, "tri_pts_resident: null pointer");
    hipError_t e = hipSuccess;
#define TCT_O(K, NS) e = pts_occ<K, NS>(blocks)
    TCT_PTS_SWITCH(kernel, nq, TCT_O)
#undef TCT_O
    if (e != hipSuccess)
        return set_error(TCT_EHIP, "tri_pts_resident: %s", hipGetErrorString(e));
    return TCT_OK;
}

extern "C" int tct_tri_pts_pack(const tct_tri_pts_plan *p, const double *obs_pts,
                                const double *obs_ns, const double *src_pts, const double *src_ns,
                                void *stream) {
    if (int e = check_pts(p, "tri_pts_pack")) return e;
    TCT_CHECK_ARG(obs_pts && obs_ns && src_pts && src_ns, "tri_pts_pack: null pointer");
#define TCT_P(K, NS) pts_pack_go<K, NS>(*p, obs_pts, obs_ns, src_pts, src_ns, as_stream(stream))
    TCT_PTS_SWITCH(p->kernel, p->nq, TCT_P)
#undef TCT_P
    TCT_CHECK_LAUNCH("tri_pts_pack");
    return TCT_OK;
}

extern "C" int tct_tri_pts_matvec(const tct_tri_pts_plan *p, const double *v, double *out,
                                  void *stream) {
    if (int e = check_pts(p, "tri_pts_matvec")) return e;
    TCT_CHECK_ARG(p->chunks >= 1 && p->chunks <= p->n_tiles, "tri_pts_matvec: chunks %d not in [1, %lld]",
                  p->chunks, (long long)p->n_tiles);
    TCT_CHECK_ARG(p->n_obs_pad / 64 * p->chunks < (1LL << 31), "tri_pts_matvec: grid too large");
    TCT_CHECK_ARG(p->partial && v && out, "tri_pts_matvec: null pointer");
    hipStream_t st = as_stream(stream);
#define TCT_M(K, NS)                    \
    pts_gather_go<K, NS>(*p, v, st);    \
    pts_go<K, NS>(*p, st)
    TCT_PTS_SWITCH(p->kernel, p->nq, TCT_M)
#undef TCT_M
    hipLaunchKernelGGL(pts_reduce_kernel, dim3((unsigned)(p->n_obs_pad / 64)), dim3(192), 0, st,
                       p->n_pts, p->n_obs_pad, p->chunks, p->obs_pt,
                       (const double *)p->partial, out);
    TCT_CHECK_LAUNCH("tri_pts_matvec");
    return TCT_OK;
}
