"""``PairsIntegrator``: the nearfield pair operator, drop-in for
tectosaur/nearfield/pairs_integrator.py:27-93.

Every method integrates a 4-D quadrature rule over a list of triangle pairs
on the device (pairs.hip, FP64) and returns [n, 3, 3, 3, 3] blocks laid out
[b_obs, d_obs, b_src, d_src].  The nearfield is computed in FP64 whatever
``float_type`` says (the reference computes it in float_type with Kahan
summation); results are returned as float64.

The ``*_dev`` variants take and return device tensors, for assembling the
nearfield matrix without host round trips.
"""
import copy
import threading

import numpy as np
import torch

from . import _native as N
from . import triangle_rules
from .quadrature import gauss2d_tri, gauss4d_tri

# pairs per launch: bounds the output buffer of one call (81 doubles/pair)
CALL_SIZE = 1 << 20


_RULES = {}
_RULES_LOCK = threading.Lock()


class DeviceRule(tuple):
    """A 4-D rule on the device, ``(qx [nq, 4], qw [nq])``.
    ``has_equal_params`` says whether some point has equal observation and
    source parameters: on a pair that is one triangle in one frame those
    points are at r = 0, and the kernel's r = 0 test must look for them; a
    rule without such points needs only the r2 == 0 test.  ``side``: the
    triangle rule (q [n, 2], w [n], on the device) whose product with itself
    the rule is, or None."""

    def __new__(cls, qx, qw, has_equal_params, side=None):
        t = super().__new__(cls, (qx, qw))
        t.has_equal_params = bool(has_equal_params)
        t.side = side
        return t


def rule_has_equal_params(qx):
    """Whether some point of a 4-D rule (qx [nq, 4]: obs xhat, obs yhat,
    src xhat, src yhat) has equal observation and source parameters."""
    qx = np.asarray(qx, dtype=np.float64)
    return bool(qx.size) and bool(np.any((qx[:, 0] == qx[:, 2]) & (qx[:, 1] == qx[:, 3])))


def product_pays(kernel, n, n_pairs):
    """Whether a rule that is a product of an n-point triangle rule with
    itself runs as one.  The surface-curl kernels, whose sums are few, always
    (3 x 3 points, RH3 135 -> 106 us for 710,704 pairs); U, T, A and H, with 81
    sums a pair and a wave less per SIMD, from 19 points (U3, 710,704 pairs:
    4 x 4 points 142 -> 167 us, 19 x 19 873 -> 626; 13 x 13, 29,128 pairs: 56 -> 90;
    T3, 19 x 19: 1212 -> 1106), T, A and H with fewer than 28 on 8,192 pairs or
    more (19 x 19 points, 5,000 pairs, T 41 -> 43; 20,000: 100 -> 67).  A rule of
    1,024 points and more in all, which has 64 lanes a pair as it stands and at
    most 16 as a product, only on as many pairs as give every SIMD a wave either
    way (64 x 64 points, 1,000 pairs: U 39 -> 55 us, H 52 -> 97, RT 28 -> 34, RH 31 ->
    28; 5,000: 169 -> 104, 235 -> 185, 82 -> 52, 52 -> 44)."""
    curl = kernel in ('elasticRT3', 'elasticRA3', 'elasticRH3')
    if not curl and (n < 19 or (n < 28 and kernel != 'elasticU3' and n_pairs < 8192)):
        return False
    return n * n < 1024 or n_pairs >= (512 if kernel == 'elasticRH3' else 1536)


def r0_test_mode(q, check0):
    """The check0 argument of tct_pairs_integrate: 0 without the r = 0
    test, 1 for the full test, 2 for r2 == 0 alone (rules known to have no
    point of equal obs and src parameters)."""
    if not check0:
        return 0
    return 1 if getattr(q, 'has_equal_params', True) else 2


class PairsIntegrator:
    def __init__(self, kernel, params, float_type, nq_far, nq_near, pts, tris):
        self.kernel = kernel
        self.kid = N.KERNEL_IDS[kernel]
        self.float_type = float_type
        self.params = N.params_array(params)
        self.device = N.require_device()
        tris = np.asarray(tris)
        if tris.size and (tris.min() < 0 or tris.max() >= np.asarray(pts).shape[0]):
            raise IndexError('triangle vertex index out of range')
        self.gpu_pts = N.upload(np.asarray(pts, dtype=np.float64), None, self.device)
        self.gpu_tris = N.upload(np.asarray(tris, dtype=np.int32), None, self.device)
        self._rules = {}
        self.near_q = self._product_rule('near4d', nq_near)
        self.far_q = self._product_rule('far4d', nq_far)

    def quad_to_gpu(self, q, side=None):
        up = lambda a: N.upload(a, torch.float64, self.device)
        qx = np.asarray(q[0], dtype=np.float64)
        return DeviceRule(up(qx), up(q[1]), rule_has_equal_params(qx),
                          None if side is None else (up(side[0]), up(side[1])))

    def _product_rule(self, name, nq):
        return self._rule((name, nq), lambda: gauss4d_tri(nq, nq), lambda: gauss2d_tri(nq))

    def _rule(self, key, make, side=None):
        if key not in self._rules:
            # rules are pure functions of their orders and read-only on the
            # device: one copy per device shared by every integrator
            dkey = (key, str(self.device))
            q = _RULES.get(dkey)
            if q is None:
                with _RULES_LOCK:
                    q = _RULES.get(dkey)
                    if q is None:
                        q = _RULES[dkey] = self.quad_to_gpu(make(), side and side())
            self._rules[key] = q
        return self._rules[key]

    def with_kernel(self, kernel):
        """An integrator of another kernel on the same mesh and rules."""
        if kernel == self.kernel:
            return self
        o = copy.copy(self)
        o.kernel = kernel
        o.kid = N.KERNEL_IDS[kernel]
        return o

    def product_side(self, q, n_pairs):
        """The triangle rule of a product rule that this kernel runs as one on
        so many pairs, or None."""
        side = getattr(q, 'side', None)
        pays = side is not None and product_pays(self.kernel, side[1].shape[0], n_pairs)
        return side if pays else None

    def pairs_quad_rows(self, q, pairs_dev, check0, rows, out, minus=None, subtract=False):
        """Pair i's block into row rows[i] (int32 device tensor) of ``out``
        [., 81].  minus: a product rule whose integrals of the same pairs are
        subtracted (q must be one too: ``product_side``).  subtract: the
        integrals are subtracted from the rows instead of written."""
        n = pairs_dev.shape[0]
        width = pairs_dev.shape[1]
        side = getattr(q, 'side', None)
        product = self.product_side(q, n) is not None or subtract or minus is not None
        if (minus is not None or subtract) and side is None:
            raise N.TctError('only product rules subtract')
        mq, mw = (None, None) if minus is None else minus.side
        st = N.stream_ptr()
        for s in range(0, n, CALL_SIZE):
            e = min(n, s + CALL_SIZE)
            if product:
                sq, sw = side
                N.call('tct_pairs_product', self.kid, sw.shape[0], N.ptr(sq), N.ptr(sw),
                       sw.shape[0], N.ptr(sq), N.ptr(sw), 0 if mw is None else mw.shape[0],
                       N.ptr(mq), N.ptr(mw), N.ptr(self.gpu_pts), N.ptr(self.gpu_tris), e - s,
                       N.ptr(pairs_dev[s:e]), width, r0_test_mode(q, check0),
                       self.params.ctypes.data, N.ptr(rows[s:e]), int(subtract), N.ptr(out), st)
            else:
                N.call('tct_pairs_integrate_rows', self.kid, q[0].shape[0], N.ptr(q[0]),
                       N.ptr(q[1]), N.ptr(self.gpu_pts), N.ptr(self.gpu_tris), e - s,
                       N.ptr(pairs_dev[s:e]), width, r0_test_mode(q, check0),
                       self.params.ctypes.data, 0, N.ptr(rows[s:e]), N.ptr(out), st)

    def pairs_quad_dev(self, q, pairs_dev, check0, out=None, lanes_per_pair=0):
        """pairs_dev: int32 device tensor [n, 2] or [n, 5]; returns [n, 81]."""
        n = pairs_dev.shape[0]
        width = pairs_dev.shape[1] if pairs_dev.dim() == 2 else 2
        if out is None:
            out = torch.empty((n, 81), dtype=torch.float64, device=self.device)
        st = N.stream_ptr()
        # a rule that is a product runs as one, unless the caller chooses how
        # many lanes share a pair's 4-D rule
        side = self.product_side(q, n) if lanes_per_pair == 0 else None
        for s in range(0, n, CALL_SIZE):
            e = min(n, s + CALL_SIZE)
            if side is not None:
                sq, sw = side
                N.call('tct_pairs_product', self.kid, sw.shape[0], N.ptr(sq), N.ptr(sw),
                       sw.shape[0], N.ptr(sq), N.ptr(sw), 0, None, None, N.ptr(self.gpu_pts),
                       N.ptr(self.gpu_tris), e - s, N.ptr(pairs_dev[s:e]), width,
                       r0_test_mode(q, check0), self.params.ctypes.data, None, 0,
                       N.ptr(out[s:e]), st)
                continue
            N.call('tct_pairs_integrate', self.kid, q[0].shape[0], N.ptr(q[0]), N.ptr(q[1]),
                   N.ptr(self.gpu_pts), N.ptr(self.gpu_tris), e - s, N.ptr(pairs_dev[s:e]),
                   width, r0_test_mode(q, check0), self.params.ctypes.data, lanes_per_pair,
                   N.ptr(out[s:e]), st)
        return out

    def pairs_quad(self, q, pairs_list, check0):
        pairs_list = np.asarray(pairs_list)
        n = pairs_list.shape[0]
        if n == 0:
            return np.empty((0, 3, 3, 3, 3), dtype=np.float64)
        check_pairs(pairs_list, self.gpu_tris.shape[0])
        p = N.upload(pairs_list.astype(np.int32), None, self.device)
        return self.pairs_quad_dev(q, p, check0).cpu().numpy().reshape((n, 3, 3, 3, 3))

    def correction(self, pairs_list, check0):
        return self.pairs_quad(self.far_q, np.asarray(pairs_list)[:, :2], check0)

    def nearfield(self, pairs_list):
        return self.pairs_quad(self.near_q, pairs_list, False)

    def vert_adj(self, nq, pairs_list):
        if isinstance(nq, (int, np.integer)):
            nq = (nq, nq, nq)
        q = self._rule(('va',) + tuple(nq), lambda: triangle_rules.vertex_adj_quad(*nq))
        return self.pairs_quad(q, self._width5(pairs_list), True)

    def coincident(self, nq, pairs_list):
        q = self._rule(('co', nq), lambda: triangle_rules.coincident_quad(nq))
        return self.pairs_quad(q, pairs_list, True)

    def edge_adj(self, nq, pairs_list):
        q = self._rule(('ea', nq), lambda: triangle_rules.edge_adj_quad(nq))
        return self.pairs_quad(q, self._width5(pairs_list), True)

    @staticmethod
    def _width5(pairs_list):
        p = np.asarray(pairs_list).astype(np.int64)
        if p.shape[0] == 0:
            return np.zeros((0, 5), dtype=np.int64)
        if p.shape[1] == 4:  # (obs, src, obs_clicks, src_clicks) with no flip column
            p = np.concatenate([p, np.zeros((p.shape[0], 1), dtype=np.int64)], axis=1)
        return p


def check_pairs(pairs, n_tris):
    """Host-side validation before a launch: the kernel trusts these indices."""
    p = np.asarray(pairs)
    if p.ndim != 2 or p.shape[1] not in (2, 5):
        raise ValueError('pairs must be [n, 2] or [n, 5]')
    if p.shape[0] == 0:
        return
    if p[:, :2].min() < 0 or p[:, :2].max() >= n_tris:
        raise IndexError('pair triangle index out of range [0, %d)' % n_tris)
    if p.shape[1] == 5 and (p[:, 2:4].min() < 0 or p[:, 2:4].max() > 2 or
                            p[:, 4].min() < 0 or p[:, 4].max() > 1):
        raise ValueError('rotation clicks must be 0..2 and flip 0/1')
