"""Triangle-to-triangle farfield on the device (far_tri.h): the layout of one
operator and the launches of a matvec.

``TriFarfield`` packs whole triangles instead of single points: a lane of the
N-body holds one observation triangle and walks source triangles, so what is
constant over a flat triangle (normals, surface curls) is used once per
triangle pair.  It serves rules of three points (equal weights) and four
points; other rules keep the point layout of ``farfield.FarfieldEngine``.
"""
import ctypes

import numpy as np
import torch

from . import _native as N
from .farfield import group_extent
from .kernels import kernels as KERNELS

TILE = N.TRI_TILE
LANES = 64
# points of the rules with a triangle form, whose last three weights are equal:
# a lane keeps every point of its triangle, its accumulators and a source
# triangle's record in registers, which seven points exceed (the form with one
# observation point a lane, TriToPtFarfield, has room for seven source points, but
# no Galerkin scatter)
RULE_POINTS = (3, 4)


def supports(qw):
    """Whether a triangle rule with weights ``qw`` has a triangle form."""
    return qw.shape[0] in RULE_POINTS and bool(np.all(qw[-3:] == qw[-1]))


def layout_extent(o_pts, s_pts, nq):
    """Rounding bound of one point stored against two different origins: the
    extents of an observation triangle and of a source tile."""
    return group_extent(o_pts, nq) + group_extent(s_pts, nq * TILE)


def source_chunks(obs_blocks, n_tiles, resident):
    """Source chunks of a launch of obs_blocks x chunks workgroups, of which
    the chip holds ``resident`` at once, four waves each.  A chunk lasts as long
    as its busiest wave, so every wave takes the same number k of tiles and the
    chunks are groups of 4 k (far_tri.h).  k = 1 up to 8,192 such workgroups, 2
    up to 16,384, then 3 while that is at most sixteen rounds of workgroups,
    whose loads and sums overlap others' arithmetic (H FP32, 32,256 triangles:
    7.97 ms in one round, 7.41 in four, 7.18 in sixteen); more beyond, as every
    chunk has its sums to write and an observation block adds the sums of its
    chunks one after another, 512 at most (FP64 H, four points, 100 x 59,700
    triangles: 311 us with 933 chunks, 262 with 467).  k = 1, 2, 3, us: RH FP32,
    4,144 triangles 98.7 99.3 100.6, 6,580 235 224 227, 9,130 425 410 406; FP64 T,
    four points, 306 314 316, 760 749 759, 1436 1418 1413.  Chunks of equal size
    -> this: FP64 H, four points, 1,240 triangles 111 -> 64 (90 over points),
    2,640 236 -> 200; FP64 T, four points, 1,900 116 -> 86; A FP32, 2,640 64 -> 52.
    From the sizes and the compiled kernel alone: the chunks set the summation
    order."""
    groups = -(-n_tiles // 4)
    work = obs_blocks * groups
    k = max(min(3, -(-work // 8192)), -(-work // (16 * max(resident, 1024))), -(-groups // 512))
    return -(-groups // k)


_RESIDENT = {}


def resident_blocks(kid, nq, prec_id):
    """N-body workgroups the chip (256 CUs) holds at once."""
    key = (kid, nq, prec_id)
    if key not in _RESIDENT:
        b = ctypes.c_int(0)
        N.call('tct_tri_resident', kid, nq, prec_id, ctypes.byref(b))
        _RESIDENT[key] = 256 * max(1, b.value)
    return _RESIDENT[key]


class TriFarfield:
    """Device layout + launches of one operator.  ``plan``: the host arrays
    of ``sparse_farfield_op.farfield_plan``."""

    def __init__(self, K_name, params, plan, device):
        K = KERNELS[K_name]
        self.K = K
        self.device = device
        nq = plan['nq']
        qw = np.asarray(plan['q'][1], dtype=np.float64)
        o_pts, s_pts = plan['o_pts'], plan['s_pts']
        self.n_obs, self.n_src = o_pts.shape[0] // nq, s_pts.shape[0] // nq
        if self.n_obs == 0 or self.n_src == 0:
            raise N.TctError('empty point set')
        self.nq = nq
        n_pad = -(-self.n_obs // LANES) * LANES
        n_tiles = -(-self.n_src // TILE)
        self.n_obs_pad, self.n_tiles = n_pad, n_tiles
        self.n_out = N.lib().tct_tri_outputs(K.kid, nq)
        words = N.lib().tct_tri_words(K.kid, nq)
        same = s_pts is o_pts
        # in the types that the kernels read, whatever a caller's plan holds
        up = lambda a: N.upload(a, torch.float64, device)
        up32 = lambda a: N.upload(a, torch.int32, device)
        f64 = dict(dtype=torch.float64, device=device)
        f32 = dict(dtype=torch.float32, device=device)
        obs_of = np.empty(self.n_obs, dtype=np.int32)   # packed position -> triangle
        obs_of[plan['pt_of_tri']] = np.arange(self.n_obs, dtype=np.int32)
        jac = lambda wj: np.ascontiguousarray(wj[nq - 1::nq]) / qw[nq - 1]
        t = {'obs': torch.empty((3 * nq + 3) * n_pad, **f64),
             'obs_org': torch.empty(3 * n_pad, **f64),
             'rec32': torch.empty(n_tiles * TILE * words, **f32),
             'rec64': torch.empty(n_tiles * TILE * words, **f64),
             'src_org': torch.empty(3 * n_tiles, **f64),
             'obs_tri': up32(obs_of), 'src_tri': up32(plan['tri_of_pt'][::nq]),
             'obs_jac': up(jac(plan['o_wj']))}
        t['src_jac'] = t['obs_jac'] if same else up(jac(plan['s_wj']))
        if K.surf_curl_obs:
            t['obs_curl'] = up(plan['curl_obs'])
        if K.surf_curl_src:
            shared = K.surf_curl_obs and plan['curl_src'] is plan['curl_obs']
            t['src_curl'] = t['obs_curl'] if shared else up(plan['curl_src'])
        self._t = t
        extent = plan.get('tri_extent')
        self.group_extent = layout_extent(o_pts, s_pts, nq) if extent is None else float(extent)
        p = N.TriPlan(kernel=K.kid, nq=nq, n_obs=self.n_obs, n_obs_pad=n_pad, n_src=self.n_src,
                      n_tiles=n_tiles, eps2=(8.0 * 2.0 ** -24 * self.group_extent) ** 2,
                      group_extent=self.group_extent)
        p.params[:] = [float(x) for x in params][:2]
        p.qw[:nq] = qw.tolist()
        p.phi[:3 * nq] = np.asarray(plan['phi'], dtype=np.float64).reshape(-1).tolist()
        p.chunks[:] = [source_chunks(n_pad // LANES, n_tiles, resident_blocks(K.kid, nq, i))
                       for i in (N.F32, N.F64)]
        for k, v in t.items():
            setattr(p, k, N.ptr(v))
        self.plan = p
        self._partial = {}
        o, on = up(o_pts), up(plan['o_ns'][::nq])
        s, sn = (o, on) if same else (up(s_pts), up(plan['s_ns'][::nq]))
        N.call('tct_tri_pack', ctypes.addressof(p), N.ptr(o), N.ptr(on), N.ptr(s), N.ptr(sn),
               N.stream_ptr())

    @staticmethod
    def prec_id(prec):
        if prec not in ('f32', 'f64'):
            raise ValueError('precision must be f32 or f64')
        return N.F32 if prec == 'f32' else N.F64

    def partial(self, prec):
        """The partial sums of ``prec`` (allocated at the first use)."""
        pid = self.prec_id(prec)
        buf = self._partial.get(pid)
        if buf is None:
            buf = torch.empty(self.plan.chunks[pid] * self.n_out * self.n_obs_pad,
                              dtype=torch.float64, device=self.device)
            self._partial[pid] = buf
            self.plan.partial[pid] = N.ptr(buf)
        return buf

    def gather(self, v_dev, prec):
        N.call('tct_tri_gather', ctypes.addressof(self.plan), self.prec_id(prec), N.ptr(v_dev),
               N.stream_ptr())

    def run(self, prec):
        """Launch the N-body; returns the partial sums."""
        return run_batched([self], prec)[0]

    def scatter(self, prec, out_dev):
        self.partial(prec)
        N.call('tct_tri_scatter', ctypes.addressof(self.plan), self.prec_id(prec),
               N.ptr(out_dev), N.stream_ptr())

    def matvec(self, v_dev, out_dev, prec):
        pid = self.prec_id(prec)
        if pid not in self._partial:
            self.partial(prec)
        N.call('tct_tri_matvec', ctypes.addressof(self.plan), pid, N.ptr(v_dev), N.ptr(out_dev),
               N.stream_ptr())
        return out_dev

    @property
    def pair_evals(self):
        return self.n_obs * self.n_src * self.nq ** 2


def run_batched(tris, prec='f32'):
    """One launch for the N-bodies of several ``TriFarfield`` (same kernel,
    rule and constants); every one's partial sums get what its own ``run``
    would write.  Returns the partial-sum buffers."""
    outs = [t.partial(prec) for t in tris]
    if tris:
        ptrs = (ctypes.c_void_p * len(tris))(*[ctypes.addressof(t.plan) for t in tris])
        N.call('tct_tri_nbody', len(tris), ctypes.addressof(ptrs), TriFarfield.prec_id(prec),
               N.stream_ptr())
    return outs


class TriToPtFarfield:
    """Device layout + launches of one FP32 triangle-to-point operator.
    ``o_pts``, ``o_ns`` [n, 3] in packing order, ``pt`` the caller's point of
    each; ``s_pts``, ``s_ns`` [n_src * nq, 3] the sources' rule points, whole
    triangles together, ``tri`` and ``jac`` [n_src]; ``q`` the rule, ``phi``
    its basis values [nq, 3]."""

    def __init__(self, K_name, params, o_pts, o_ns, pt, s_pts, s_ns, tri, jac, q, phi, device):
        kid = KERNELS[K_name].kid
        nq = q[1].shape[0]
        if o_pts.shape[0] == 0 or tri.shape[0] == 0:
            raise N.TctError('empty point set')
        n_pad = -(-o_pts.shape[0] // LANES) * LANES
        tile = N.lib().tct_tri_pts_tile(kid, nq)
        n_tiles = -(-tri.shape[0] // tile)
        self.device = device
        up = lambda a: N.upload(a, None, device)
        f64 = dict(dtype=torch.float64, device=device)
        f32 = dict(dtype=torch.float32, device=device)
        words = N.lib().tct_tri_pts_words(kid, nq)
        self.chunks = source_chunks(n_pad // LANES, n_tiles, resident_pts(kid, nq))
        t = {'obs': torch.empty(6 * n_pad, **f32),
             'obs_org': torch.empty(3 * (n_pad // LANES), **f64),
             'rec': torch.empty(n_tiles * tile * words, **f32),
             'src_org': torch.empty(3 * n_tiles, **f64),
             'obs_pt': up(np.ascontiguousarray(pt, dtype=np.int32)),
             'src_tri': up(np.ascontiguousarray(tri, dtype=np.int32)),
             'src_jac': up(np.ascontiguousarray(jac, dtype=np.float64)),
             'partial': torch.empty(self.chunks * 3 * n_pad, **f64)}
        self._t = t
        # rounding bound of one point stored against two different origins
        self.group_extent = group_extent(o_pts, LANES) + group_extent(s_pts, nq * tile)
        p = N.TriPtsPlan(kernel=kid, nq=nq, n_pts=o_pts.shape[0], n_obs_pad=n_pad,
                         n_src=tri.shape[0], n_tiles=n_tiles, chunks=self.chunks,
                         eps2=(8.0 * 2.0 ** -24 * self.group_extent) ** 2)
        p.params[:] = [float(x) for x in params][:2]
        p.qw[:nq] = np.asarray(q[1], dtype=np.float64).tolist()
        p.phi[:3 * nq] = np.asarray(phi, dtype=np.float64).reshape(-1).tolist()
        for k, v in t.items():
            setattr(p, k, N.ptr(v))
        self.plan = p
        dev = [up(np.ascontiguousarray(a)) for a in (o_pts, o_ns, s_pts, s_ns[::nq])]
        N.call('tct_tri_pts_pack', ctypes.addressof(p), *[N.ptr(a) for a in dev],
               N.stream_ptr())

    def matvec(self, v_dev, out_dev):
        N.call('tct_tri_pts_matvec', ctypes.addressof(self.plan), N.ptr(v_dev), N.ptr(out_dev),
               N.stream_ptr())
        return out_dev


def resident_pts(kid, nq):
    """As ``resident_blocks``, of the triangle-to-point N-body."""
    key = ('pts', kid, nq)
    if key not in _RESIDENT:
        b = ctypes.c_int(0)
        N.call('tct_tri_pts_resident', kid, nq, ctypes.byref(b))
        _RESIDENT[key] = 256 * max(1, b.value)
    return _RESIDENT[key]


def pts_supported(K_name, nq):
    """Whether a kernel and a rule of ``nq`` points have the triangle-to-point
    form."""
    return N.lib().tct_tri_pts_words(KERNELS[K_name].kid, nq) > 0
