// Triangle-to-triangle farfield: packing, strengths, Galerkin scatter and
// the C ABI.  The N-body and its layout are described in far_tri.h.
#include "far_tri.h"

namespace tct {

constexpr double TRI_FAR_AWAY = 1.0e12;

// The plan's values that the kernels below read.
struct TriRule {
    double qw[4], phi[12];
};

// One thread per observation triangle: points, normal and origin.
template <int NQ>
__global__ void tri_pack_obs_kernel(int64_t n, int64_t n_pad, const double *__restrict__ pts,
                                    const double *__restrict__ ns, double *__restrict__ obs,
                                    double *__restrict__ org) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n_pad) return;
    const bool valid = i < n;
    for (int d = 0; d < 3; ++d) {
        double p[NQ], o = 0.0;
        for (int q = 0; q < NQ; ++q) {
            p[q] = valid ? pts[(i * NQ + q) * 3 + d] : 0.0;
            o += p[q] / NQ;
        }
        org[d * n_pad + i] = o;
        for (int q = 0; q < NQ; ++q) obs[(size_t)(3 * q + d) * n_pad + i] = p[q];
        obs[(size_t)(3 * NQ + d) * n_pad + i] = valid ? ns[3 * i + d] : 0.0;
    }
}

// One wave per source tile: lane (triangle, point); tile origin = mean of
// its points.  Padding triangles lie far away with zero strengths.
template <int KID, int NQ>
__global__ __launch_bounds__(64) void tri_pack_src_kernel(int64_t n,
                                                          const double *__restrict__ pts,
                                                          const double *__restrict__ ns,
                                                          float *__restrict__ r32,
                                                          double *__restrict__ r64,
                                                          double *__restrict__ org) {
    static_assert(TT * NQ <= 64, "one lane per point of a tile");
    constexpr int RW = tri_words<KID, NQ>(), SW = tri_sw<KID>();
    const int64_t t = blockIdx.x;
    const int lane = threadIdx.x;
    const int64_t k = t * TT + lane / NQ;
    const int q = lane % NQ;
    const bool slot = lane < TT * NQ;
    const bool valid = slot && k < n;
    double cnt = valid ? 1.0 : 0.0;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) cnt += __shfl_xor(cnt, off, 64);
    if (slot)   // the words that are not geometry are strengths: zero until a gather
        for (int w = q; w < RW; w += NQ) {
            r32[k * RW + w] = 0.0f;
            r64[k * RW + w] = 0.0;
        }
    __syncthreads();
    for (int d = 0; d < 3; ++d) {
        const double p = valid ? pts[(k * NQ + q) * 3 + d] : 0.0;
        double o = p;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) o += __shfl_xor(o, off, 64);
        o /= cnt;
        if (lane == 0) org[3 * t + d] = o;
        if (!slot) continue;
        r32[k * RW + SW * q + d] = valid ? (float)(p - o) : (float)TRI_FAR_AWAY;
        r64[k * RW + SW * q + d] = valid ? p : TRI_FAR_AWAY;
        if (q == 0 && tri_src_normal<KID>()) {
            const double nn = valid ? ns[3 * k + d] : 0.0;
            r32[k * RW + tri_n_word<KID, NQ>(d)] = (float)nn;
            r64[k * RW + tri_n_word<KID, NQ>(d)] = nn;
        }
    }
}

// Strengths: one thread per (packed source triangle, rule point).  RH: thread
// q < 3 forms row q of the source curl; RT: component q of its curl term.
template <int KID, int NQ, typename T>
__global__ __launch_bounds__(192) void tri_gather_kernel(
    int64_t n, int64_t n_pad, TriRule rule, const int32_t *__restrict__ tri,
    const double *__restrict__ jac, const double *__restrict__ curl, StrengthConsts sc,
    ElasticConsts c, const double *__restrict__ v, T *__restrict__ rec) {
    constexpr int RW = tri_words<KID, NQ>();
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t k = i / NQ;
    const int q = (int)(i % NQ);
    if (k >= n_pad) return;
    T *r = rec + k * RW, *rq = r + tri_sw<KID>() * q;
    const bool valid = k < n;
    const int64_t t = valid ? tri[k] : 0;
    const double J = valid ? jac[k] : 0.0;
    double vt[9];
    for (int a = 0; a < 9; ++a) vt[a] = valid ? v[9 * t + a] : 0.0;
    double S[9];   // S[d][I] = sum_b curl[b][I] v[b][d]
    if constexpr (KID == TCT_RT || KID == TCT_RH) {
        double cu[9];
        for (int a = 0; a < 9; ++a) cu[a] = valid ? curl[9 * t + a] : 0.0;
        for (int d = 0; d < 3; ++d)
            for (int I = 0; I < 3; ++I)
                S[3 * d + I] = cu[I] * vt[d] + cu[3 + I] * vt[3 + d] + cu[6 + I] * vt[6 + d];
    }
    if constexpr (KID == TCT_RH) {
        const double g = J * rule.qw[NQ - 1] * c.CsRH0;
        if (q < 3)
            for (int m = 0; m < 3; ++m) {
                double s = 0.0;   // row q of S without a dynamic register index
                for (int d = 0; d < 3; ++d) s = d == q ? S[3 * d + m] : s;
                r[tri_g_word<NQ>(3 * q + m)] = (T)(g * s);
            }
    } else {
        double w = 0.0, p0 = 0.0, p1 = 0.0, p2 = 0.0;
        for (int a = 0; a < NQ; ++a)
            if (a == q) {
                w = rule.qw[a];
                p0 = rule.phi[3 * a];
                p1 = rule.phi[3 * a + 1];
                p2 = rule.phi[3 * a + 2];
            }
        const double f = (KID == TCT_RT ? c.CsRT2 : sc.scale) * (J * w);
        double s[3];
        for (int d = 0; d < 3; ++d) {
            s[d] = f * (p0 * vt[d] + p1 * vt[3 + d] + p2 * vt[6 + d]);
            rq[3 + d] = (T)s[d];
        }
        if constexpr (KID == TCT_T || KID == TCT_H) {
            double sn = 0.0;
            for (int d = 0; d < 3; ++d) sn += (double)r[tri_n_word<KID, NQ>(d)] * s[d];
            rq[6] = (T)(sc.x0 * sn);
            if constexpr (KID == TCT_H) rq[7] = (T)(sc.x1 * sn);
        }
        if constexpr (KID == TCT_RT) {
            double a = 0.0;
            for (int tt = 0; tt < 3; ++tt) {
                double e = 0.0;
                for (int d = 0; d < 3; ++d)
                    for (int I = 0; I < 3; ++I) e += levi3(I, tt, d) * S[3 * d + I];
                a = tt == q ? e : a;
            }
            if (q < 3) r[tri_e_word(q)] = (T)(c.CsRT1 * (J * rule.qw[NQ - 1]) * a);
        }
    }
}

// Chunk sums and Galerkin scatter in one launch: a workgroup takes 64
// observation triangles; thread (output, triangle) adds the chunks' partial
// sums in chunk order (coalesced, eight loads in flight), then thread (triangle,
// DOF) contracts the triangle's sums with the basis and writes one of its 9
// DOFs.  The separate chunk-sum and scatter launches of the point layout read
// and wrote the sums once more (24 us of a 66 us matvec at 2,048 triangles).
template <int KID, int NQ>
__global__ __launch_bounds__((64 * tri_out<KID, NQ>())) void tri_scatter_kernel(
    int64_t n, int64_t n_pad, int chunks, TriRule rule, const int32_t *__restrict__ tri,
    const double *__restrict__ jac, const double *__restrict__ curl, ElasticConsts c,
    const double *__restrict__ partial, double *__restrict__ out) {
    constexpr int NO = tri_out<KID, NQ>();
    constexpr int CI = 8;
    __shared__ double sum[NO][65];
    const int64_t b0 = (int64_t)blockIdx.x * 64;
    {
        const int a = (int)threadIdx.x / 64, lane = (int)threadIdx.x % 64;
        const double *p = partial + (size_t)a * n_pad + b0 + lane;
        const size_t stride = (size_t)NO * n_pad;
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
        sum[a][lane] = s;
    }
    __syncthreads();
    const int e = (int)threadIdx.x;
    if (e >= 64 * 9) return;
    const int l = e / 9, bd = e % 9, b = bd / 3, d = bd % 3;
    const int64_t k = b0 + l;
    if (k >= n) return;
    const int64_t t = tri[k];
    const double J = jac[k];
    double r = 0.0;
    if constexpr (KID == TCT_RH) {
        const double *cu = curl + 9 * t + 3 * b;
        const double s0 = d == 0 ? sum[0][l] : (d == 1 ? sum[3][l] : sum[6][l]);
        const double s1 = d == 0 ? sum[1][l] : (d == 1 ? sum[4][l] : sum[7][l]);
        const double s2 = d == 0 ? sum[2][l] : (d == 1 ? sum[5][l] : sum[8][l]);
        r = J * rule.qw[NQ - 1] * (s0 * cu[0] + s1 * cu[1] + s2 * cu[2]);
    } else {
        constexpr int O = KID == TCT_RA ? 3 : 0;
        for (int q = 0; q < NQ; ++q) {
            double ph = 0.0;
            for (int bb = 0; bb < 3; ++bb) ph = bb == b ? rule.phi[3 * q + bb] : ph;
            r += J * rule.qw[q] * ph * sum[O + 3 * q + d][l];
        }
        if constexpr (KID == TCT_RA) {
            const double *cu = curl + 9 * t + 3 * b;
            double f = 0.0;
            for (int I = 0; I < 3; ++I)
                for (int ss = 0; ss < 3; ++ss) f += cu[I] * levi3(I, ss, d) * sum[ss][l];
            r = J * rule.qw[NQ - 1] * f - c.CsRT2 * r;
        }
    }
    out[9 * t + bd] = r;
}

static TriRule plan_rule(const tct_tri_plan &p) {
    TriRule r{};
    for (int q = 0; q < p.nq; ++q) {
        r.qw[q] = p.qw[q];
        for (int b = 0; b < 3; ++b) r.phi[3 * q + b] = p.phi[3 * q + b];
    }
    return r;
}

static int check_plan(const tct_tri_plan *p, const char *what) {
    TCT_CHECK_ARG(p, "%s: null plan", what);
    TCT_CHECK_ARG(p->kernel >= TCT_U && p->kernel <= TCT_RH, "%s: kernel id %d", what, p->kernel);
    if (p->nq != 3 && p->nq != 4)
        return set_error(TCT_EUNSUPPORTED, "%s: rule of %d points (3 or 4)", what, p->nq);
    TCT_CHECK_ARG(p->nq != 3 || (p->qw[0] == p->qw[1] && p->qw[1] == p->qw[2]),
                  "%s: a 3-point rule must have equal weights", what);
    TCT_CHECK_ARG(p->nq != 4 || (p->qw[1] == p->qw[2] && p->qw[2] == p->qw[3]),
                  "%s: a 4-point rule must have three equal last weights", what);
    TCT_CHECK_ARG(p->qw[p->nq - 1] != 0.0, "%s: the last weight is zero", what);
    TCT_CHECK_ARG(p->n_obs > 0 && p->n_obs_pad >= p->n_obs && p->n_obs_pad % 64 == 0 &&
                      p->n_obs_pad < (1LL << 28),
                  "%s: bad sizes n_obs=%lld n_obs_pad=%lld", what, (long long)p->n_obs,
                  (long long)p->n_obs_pad);
    TCT_CHECK_ARG(p->n_src > 0 && p->n_tiles < (1LL << 24) && p->n_src <= p->n_tiles * TT &&
                      p->n_src > (p->n_tiles - 1) * TT,
                  "%s: bad sizes n_src=%lld n_tiles=%lld", what, (long long)p->n_src,
                  (long long)p->n_tiles);
    TCT_CHECK_ARG(p->eps2 >= 0.0 && std::isfinite(p->eps2) && !std::isnan(p->group_extent),
                  "%s: eps2 / group_extent", what);
    TCT_CHECK_ARG((p->flags & ~1) == 0, "%s: unknown flags 0x%x", what, (unsigned)p->flags);
    TCT_CHECK_ARG(p->obs && p->obs_org && p->rec32 && p->rec64 && p->src_org &&
                      p->obs_tri && p->src_tri && p->obs_jac && p->src_jac,
                  "%s: null pointer", what);
    const bool so = p->kernel == TCT_RA || p->kernel == TCT_RH;
    const bool ss = p->kernel == TCT_RT || p->kernel == TCT_RH;
    TCT_CHECK_ARG((!so || p->obs_curl) && (!ss || p->src_curl), "%s: null curls", what);
    return TCT_OK;
}

static int check_prec(const tct_tri_plan *p, int prec, const char *what) {
    TCT_CHECK_ARG(prec == TCT_F32 || prec == TCT_F64, "%s: precision %d", what, prec);
    const int ch = p->chunks[prec];
    TCT_CHECK_ARG(ch >= 1 && ch <= p->n_tiles, "%s: chunks %d not in [1, %lld]", what, ch,
                  (long long)p->n_tiles);
    TCT_CHECK_ARG(p->n_obs_pad / 64 * ch < (1LL << 31), "%s: grid too large", what);
    TCT_CHECK_ARG(p->partial[prec], "%s: null partial sums", what);
    return TCT_OK;
}

// sep^2 as the point N-body's: beyond it no pair of a tile can reach r2 <=
// eps2.  FP64 tests r2 == 0 only, on the tiles that can hold such a pair.
static double plan_sep2(const tct_tri_plan &p) {
    if (p.eps2 > 0.0 && p.group_extent >= 0.0 && std::isfinite(p.group_extent) &&
        !(p.flags & 1)) {
        const double sep = p.group_extent * (1.0 + 1e-3) + 5.0 * std::sqrt(p.eps2);
        return sep * sep;
    }
    return INFINITY;
}

template <typename T>
static void set_seg(TriSeg<T> &g, const tct_tri_plan &p, int blk0) {
    constexpr bool F32 = sizeof(T) == 4;
    if constexpr (F32) {
        g.rec = p.rec32;
    } else {
        g.rec = p.rec64;
    }
    g.obs = p.obs;
    g.obs_org = p.obs_org;
    g.src_org = p.src_org;
    g.partial = p.partial[F32 ? TCT_F32 : TCT_F64];
    g.sep2 = plan_sep2(p);
    g.eps2 = (float)p.eps2;
    g.n_obs_pad = (int)p.n_obs_pad;
    g.n_src = (int)p.n_src;
    g.n_tiles = (int)p.n_tiles;
    g.chunks = p.chunks[F32 ? TCT_F32 : TCT_F64];
    g.blk0 = blk0;
}

template <typename T>
static int nbody(int n, const tct_tri_plan *const *plans, hipStream_t st) {
    for (int s0 = 0; s0 < n; s0 += TRI_SEG_MAX) {
        TriSegTable<T> t;
        t.n = n - s0 < TRI_SEG_MAX ? n - s0 : TRI_SEG_MAX;
        int64_t blocks = 0;
        for (int i = 0; i < t.n; ++i) {
            set_seg<T>(t.s[i], *plans[s0 + i], (int)blocks);
            blocks += (int64_t)(t.s[i].n_obs_pad / 64) * t.s[i].chunks;
            TCT_CHECK_ARG(blocks < (1LL << 31), "tri_nbody: grid too large");
        }
        const tct_tri_plan &p = *plans[s0];
        if (int e = far_tri_launch<T>(p.kernel, p.nq, p.params, p.qw, t, (unsigned)blocks, st))
            return e;
    }
    return TCT_OK;
}

template <int KID, int NQ, typename T>
static void gather_go(const tct_tri_plan &p, T *rec, const double *v, hipStream_t st) {
    const int64_t n_pad = p.n_tiles * TT;
    hipLaunchKernelGGL((tri_gather_kernel<KID, NQ, T>),
                       dim3((unsigned)ceil_div(n_pad * NQ, (int64_t)192)), dim3(192), 0, st,
                       p.n_src, n_pad, plan_rule(p), p.src_tri, p.src_jac, p.src_curl,
                       strength_consts(KID, p.params), elastic_consts(p.params), v, rec);
}

template <int KID, int NQ>
static void scatter_go(const tct_tri_plan &p, int prec, double *out, hipStream_t st) {
    const unsigned nt = 64 * (unsigned)tri_out<KID, NQ>();
    hipLaunchKernelGGL((tri_scatter_kernel<KID, NQ>), dim3((unsigned)(p.n_obs_pad / 64)),
                       dim3(nt), 0, st, p.n_obs, p.n_obs_pad, p.chunks[prec], plan_rule(p),
                       p.obs_tri, p.obs_jac, p.obs_curl, elastic_consts(p.params),
                       (const double *)p.partial[prec], out);
}

#define TCT_TRI_SWITCH(kernel, nq, F)                         \
    switch (kernel) {                                         \
    case TCT_U: F(TCT_U, nq); break;                          \
    case TCT_T: F(TCT_T, nq); break;                          \
    case TCT_A: F(TCT_A, nq); break;                          \
    case TCT_H: F(TCT_H, nq); break;                          \
    case TCT_RT: F(TCT_RT, nq); break;                        \
    case TCT_RA: F(TCT_RA, nq); break;                        \
    default: F(TCT_RH, nq); break;                            \
    }

}  // namespace tct

using namespace tct;

extern "C" int tct_tri_words(int kernel, int nq) {
    if (kernel < TCT_U || kernel > TCT_RH || (nq != 3 && nq != 4)) return 0;
    int w = 0;
#define TCT_W(K, NQ) w = tri_words<K, NQ>()
    if (nq == 3) {
        TCT_TRI_SWITCH(kernel, 3, TCT_W)
    } else {
        TCT_TRI_SWITCH(kernel, 4, TCT_W)
    }
#undef TCT_W
    return w;
}

extern "C" int tct_tri_outputs(int kernel, int nq) {
    if (kernel < TCT_U || kernel > TCT_RH || (nq != 3 && nq != 4)) return 0;
    int w = 0;
#define TCT_W(K, NQ) w = tri_out<K, NQ>()
    if (nq == 3) {
        TCT_TRI_SWITCH(kernel, 3, TCT_W)
    } else {
        TCT_TRI_SWITCH(kernel, 4, TCT_W)
    }
#undef TCT_W
    return w;
}

extern "C" int tct_tri_resident(int kernel, int nq, int prec, int *blocks) {
    TCT_CHECK_ARG(kernel >= TCT_U && kernel <= TCT_RH && (nq == 3 || nq == 4),
                  "tri_resident: kernel %d, rule of %d points", kernel, nq);
    TCT_CHECK_ARG(prec == TCT_F32 || prec == TCT_F64, "tri_resident: precision %d", prec);
    TCT_CHECK_ARG(blocks, "tri_resident: null pointer");
    return prec == TCT_F32 ? far_tri_resident<float>(kernel, nq, blocks)
                           : far_tri_resident<double>(kernel, nq, blocks);
}

extern "C" int tct_tri_pack(const tct_tri_plan *p, const double *obs_pts, const double *obs_ns,
                            const double *src_pts, const double *src_ns, void *stream) {
    if (int e = check_plan(p, "tri_pack")) return e;
    TCT_CHECK_ARG(obs_pts && obs_ns && src_pts && src_ns, "tri_pack: null pointer");
    hipStream_t st = as_stream(stream);
    const unsigned nb = (unsigned)ceil_div(p->n_obs_pad, (int64_t)256);
#define TCT_PACK(K, NQ)                                                                         \
    hipLaunchKernelGGL((tri_pack_obs_kernel<NQ>), dim3(nb), dim3(256), 0, st, p->n_obs,         \
                       p->n_obs_pad, obs_pts, obs_ns, p->obs, p->obs_org);                      \
    hipLaunchKernelGGL((tri_pack_src_kernel<K, NQ>), dim3((unsigned)p->n_tiles), dim3(64), 0,   \
                       st, p->n_src, src_pts, src_ns, p->rec32, p->rec64, p->src_org)
    if (p->nq == 3) {
        TCT_TRI_SWITCH(p->kernel, 3, TCT_PACK)
    } else {
        TCT_TRI_SWITCH(p->kernel, 4, TCT_PACK)
    }
#undef TCT_PACK
    TCT_CHECK_LAUNCH("tri_pack");
    return TCT_OK;
}

extern "C" int tct_tri_gather(const tct_tri_plan *p, int prec, const double *v, void *stream) {
    if (int e = check_plan(p, "tri_gather")) return e;
    TCT_CHECK_ARG(prec == TCT_F32 || prec == TCT_F64, "tri_gather: precision %d", prec);
    TCT_CHECK_ARG(v, "tri_gather: null pointer");
    hipStream_t st = as_stream(stream);
#define TCT_G32(K, NQ) gather_go<K, NQ, float>(*p, p->rec32, v, st)
#define TCT_G64(K, NQ) gather_go<K, NQ, double>(*p, p->rec64, v, st)
    if (p->nq == 3) {
        if (prec == TCT_F32) {
            TCT_TRI_SWITCH(p->kernel, 3, TCT_G32)
        } else {
            TCT_TRI_SWITCH(p->kernel, 3, TCT_G64)
        }
    } else {
        if (prec == TCT_F32) {
            TCT_TRI_SWITCH(p->kernel, 4, TCT_G32)
        } else {
            TCT_TRI_SWITCH(p->kernel, 4, TCT_G64)
        }
    }
#undef TCT_G32
#undef TCT_G64
    TCT_CHECK_LAUNCH("tri_gather");
    return TCT_OK;
}

extern "C" int tct_tri_nbody(int n, const tct_tri_plan *const *plans, int prec, void *stream) {
    TCT_CHECK_ARG(n >= 0 && (n == 0 || plans), "tri_nbody: bad plan list");
    for (int i = 0; i < n; ++i) {
        if (int e = check_plan(plans[i], "tri_nbody")) return e;
        if (int e = check_prec(plans[i], prec, "tri_nbody")) return e;
        const tct_tri_plan &a = *plans[0], &b = *plans[i];
        bool same = a.kernel == b.kernel && a.nq == b.nq && a.params[0] == b.params[0] &&
                    a.params[1] == b.params[1];
        for (int q = 0; q < a.nq; ++q) same = same && a.qw[q] == b.qw[q];
        TCT_CHECK_ARG(same, "tri_nbody: plan %d differs in kernel, rule or constants", i);
    }
    if (n == 0) return TCT_OK;
    return prec == TCT_F32 ? nbody<float>(n, plans, as_stream(stream))
                           : nbody<double>(n, plans, as_stream(stream));
}

extern "C" int tct_tri_scatter(const tct_tri_plan *p, int prec, double *out, void *stream) {
    if (int e = check_plan(p, "tri_scatter")) return e;
    if (int e = check_prec(p, prec, "tri_scatter")) return e;
    TCT_CHECK_ARG(out, "tri_scatter: null pointer");
    hipStream_t st = as_stream(stream);
#define TCT_S(K, NQ) scatter_go<K, NQ>(*p, prec, out, st)
    if (p->nq == 3) {
        TCT_TRI_SWITCH(p->kernel, 3, TCT_S)
    } else {
        TCT_TRI_SWITCH(p->kernel, 4, TCT_S)
    }
#undef TCT_S
    TCT_CHECK_LAUNCH("tri_scatter");
    return TCT_OK;
}

extern "C" int tct_tri_matvec(const tct_tri_plan *p, int prec, const double *v, double *out,
                              void *stream) {
    if (int e = tct_tri_gather(p, prec, v, stream)) return e;
    if (int e = tct_tri_nbody(1, &p, prec, stream)) return e;
    return tct_tri_scatter(p, prec, out, stream);
}
