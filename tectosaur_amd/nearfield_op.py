"""``RegularizedNearfieldIntegralOp``: the nearfield operator, drop-in for
tectosaur/nearfield/nearfield_op.py:76-168.

Assembly (one-time, per mesh), following nearfield_op.py:95-141:
  * coincident pairs (obs_subset intersect src_subset), integrated with the
    Erichsen-Sauter rule, r2 == 0 points skipped;
  * near pairs |c_i - c_j| <= thr (r_i + r_j) found on the host and split
    by shared vertices into edge-adjacent (rotated so the shared edge is
    local edge 0-1, :44-62), vertex-adjacent (shared vertex rotated to local
    vertex 0) and plain near pairs;
  * each class integrated with K_near and its accurate rule, minus the same
    pairs integrated with K_far and the farfield rule (the farfield operator
    covers every pair with that rule, so the difference corrects it);
  * all blocks placed in one 9x9 BSR matrix on the device (the reference
    keeps four BCOO matrices and applies them on the host).
All integration runs on the device in FP64 (pairs.hip, pairs_product.hip),
sorted pair lists straight into their rows of the matrix.
"""
import ctypes

import numpy as np
import torch

from . import _native as N
from . import find_near_adj
from .pairs_integrator import PairsIntegrator, check_pairs
from .sparse import BSRMatrix, bcoo_to_bsr_dev


def edge_adj_orient(tv0, tv1):
    """Rotation that maps the shared edge to local vertices (0, 1)
    (nearfield_op.py:44-50), vectorised: corners {0,1} -> 0, {1,2} -> 1,
    {0,2} -> 2."""
    lo = np.minimum(tv0, tv1)
    hi = np.maximum(tv0, tv1)
    return np.where(lo == 0, np.where(hi == 2, 2, 0), 1)


def resolve_ea_rotation(tris, ea):
    """(obs, src, obs_clicks, src_clicks, src_flip) per edge-adjacent pair
    (nearfield_op.py:52-62)."""
    ea = np.asarray(ea, dtype=np.int64).reshape((-1, 6))
    oc = edge_adj_orient(ea[:, 2], ea[:, 4])
    sc = edge_adj_orient(ea[:, 3], ea[:, 5])
    t = np.asarray(tris)
    flip = ((t[ea[:, 0], (0 + oc) % 3] != t[ea[:, 1], (1 + sc) % 3]) |
            (t[ea[:, 0], (1 + oc) % 3] != t[ea[:, 1], (0 + sc) % 3]))
    return np.stack([ea[:, 0], ea[:, 1], oc, sc, flip.astype(np.int64)], axis=1)


def _is_identity(subset):
    s = np.asarray(subset)
    return s.ndim == 1 and (s.size == 0 or (s[0] == 0 and s[-1] == s.size - 1 and
                                            bool(np.all(np.diff(s) == 1))))


def to_tri_space(dof_indices, obs_subset, src_subset):
    """Positions in the subsets to triangles; where both subsets are the whole
    mesh, the positions themselves (the same array, not a copy)."""
    di = np.asarray(dof_indices, dtype=np.int64)
    # identity subsets (the whole mesh) map positions to themselves: the
    # array itself where both are
    o_id, s_id = _is_identity(obs_subset), _is_identity(src_subset)
    if o_id and s_id:
        return di
    out = di.copy()
    if not o_id:
        out[:, 0] = obs_subset[di[:, 0]]
    if not s_id:
        out[:, 1] = src_subset[di[:, 1]]
    return out


def to_dof_space(tri_indices, obs_subset, src_subset):
    """Positions of (obs tri, src tri) within the subsets (nearfield_op.py:24-38)."""
    ti = np.asarray(tri_indices, dtype=np.int64).reshape((-1, 2))
    n = int(max(obs_subset.max(initial=-1), src_subset.max(initial=-1))) + 1
    opos = np.full(n, -1, dtype=np.int64)
    spos = np.full(n, -1, dtype=np.int64)
    opos[obs_subset] = np.arange(obs_subset.shape[0])
    spos[src_subset] = np.arange(src_subset.shape[0])
    out = np.stack([opos[ti[:, 0]], spos[ti[:, 1]]], axis=1) if ti.shape[0] else \
        np.zeros((0, 2), dtype=np.int64)
    if (out < 0).any():
        raise ValueError('pair outside the obs/src subsets')
    return out


def nearfield_plan(pts, tris, obs_subset, src_subset, near_threshold, finder='host'):
    """Pair classification: coincident, edge-adjacent (rotated),
    vertex-adjacent and near pairs, in triangle and DOF space
    (nearfield_op.py:95-114).  finder 'host' searches with the C++ finder
    (no device work, safe on worker threads); 'device' with the device
    finder and classifier (the same pairs, in the same order)."""
    pts = np.asarray(pts, dtype=np.float64)
    tris = np.asarray(tris, dtype=np.int64)
    obs_subset = np.asarray(obs_subset, dtype=np.int64)
    src_subset = np.asarray(src_subset, dtype=np.int64)
    co_tris = np.intersect1d(obs_subset, src_subset)
    co_indices = np.stack([co_tris, co_tris], axis=1)
    co_dofs = to_dof_space(co_indices, obs_subset, src_subset)
    if finder == 'device':
        import torch
        ta, tb = tris[obs_subset], tris[src_subset]
        close = find_near_adj.find_near_pairs_dev(
            *find_near_adj.get_tri_centroids_rs(pts, ta),
            *find_near_adj.get_tri_centroids_rs(pts, tb), near_threshold)
        d = lambda a: torch.as_tensor(np.ascontiguousarray(a), device=close.device)
        near_dofs, va_dofs, ea_dofs = (x.cpu().numpy() for x in
                                       find_near_adj.split_adjacent_close_dev(close, d(ta), d(tb)))
    elif finder == 'host':
        close = find_near_adj.find_close_or_touching(pts, tris[obs_subset], pts,
                                                     tris[src_subset], near_threshold)
        near_dofs, va_dofs, ea_dofs = find_near_adj.split_adjacent_close(
            close, tris[obs_subset], tris[src_subset])
    else:
        raise ValueError("finder must be 'host' or 'device'")
    near = to_tri_space(near_dofs, obs_subset, src_subset)
    va = to_tri_space(va_dofs, obs_subset, src_subset)
    va = np.concatenate([va, np.zeros((va.shape[0], 1), dtype=np.int64)], axis=1)
    ea = resolve_ea_rotation(tris, to_tri_space(ea_dofs, obs_subset, src_subset))
    return dict(co=(co_indices, co_dofs), ea=(ea, ea_dofs[:, :2]), va=(va, va_dofs[:, :2]),
                near=(near, near_dofs))


def check_places(dofs, shape):
    """The blocks (dofs [n, 2], n > 0) must lie in a matrix of ``shape``: its
    product trusts the columns and the rows of blocks."""
    d = np.asarray(dofs)
    for k, what in ((0, 'row'), (1, 'column')):
        if d[:, k].min() < 0 or d[:, k].max() >= shape[k] // 9:
            raise IndexError('block %s out of range [0, %d)' % (what, shape[k] // 9))


class RegularizedNearfieldIntegralOp:
    def __init__(self, pts, tris, obs_subset, src_subset, nq_coincident, nq_edge_adj,
                 nq_vert_adjacent, nq_far, nq_near, near_threshold, K_near_name, K_far_name,
                 params, float_type, keep_classes=False, plan=None, keep_uncorrected=True):
        pts = np.asarray(pts, dtype=np.float64)
        tris = np.asarray(tris, dtype=np.int64)
        obs_subset = np.asarray(obs_subset, dtype=np.int64)
        src_subset = np.asarray(src_subset, dtype=np.int64)
        self.shape = (obs_subset.shape[0] * 9, src_subset.shape[0] * 9)
        self.device = N.require_device()
        dev = self.device
        pairs_int = PairsIntegrator(K_near_name, params, float_type, nq_far, nq_near, pts, tris)
        corr_int = pairs_int.with_kernel(K_far_name)
        if plan is None:
            plan = nearfield_plan(pts, tris, obs_subset, src_subset, near_threshold)

        from . import triangle_rules
        from .quadrature import gauss4d_tri
        nqv = nq_vert_adjacent if not isinstance(nq_vert_adjacent, (int, np.integer)) else \
            (nq_vert_adjacent,) * 3
        rules = {
            'co': pairs_int._rule(('co', nq_coincident),
                                  lambda: triangle_rules.coincident_quad(nq_coincident)),
            'ea': pairs_int._rule(('ea', nq_edge_adj),
                                  lambda: triangle_rules.edge_adj_quad(nq_edge_adj)),
            'va': pairs_int._rule(('va',) + tuple(nqv),
                                  lambda: triangle_rules.vertex_adj_quad(*nqv)),
            'near': pairs_int.near_q,
        }
        far_q = corr_int.far_q
        classes = (('co',) + plan['co'] + (True, True),
                   ('ea',) + plan['ea'] + (True, False),
                   ('va',) + plan['va'] + (True, False),
                   ('near',) + plan['near'] + (False, False))
        self.counts = {name: int(prs.shape[0]) for name, prs, _, _, _ in classes}
        self.classes = {}
        self.n_pairs = sum(self.counts.values())
        if not keep_classes and self._assemble_rows(classes, rules, far_q, pairs_int, corr_int,
                                                    tris.shape[0], keep_uncorrected):
            return
        rows, cols, corrected, uncorrected = [], [], [], []
        for name, prs, dofs, check0, corr_check0 in classes:
            if prs.shape[0] == 0:
                continue
            check_pairs(prs, tris.shape[0])
            check_places(dofs, self.shape)
            p_dev = N.upload(prs.astype(np.int32), None, dev)
            acc = pairs_int.pairs_quad_dev(rules[name], p_dev, check0)
            corr = corr_int.pairs_quad_dev(far_q, p_dev[:, :2].contiguous(), corr_check0)
            diff = torch.empty_like(acc)
            N.call('tct_sub_f64', acc.numel(), N.ptr(acc), N.ptr(corr), N.ptr(diff),
                   N.stream_ptr())
            rows.append(N.upload(dofs[:, 0], None, dev))
            cols.append(N.upload(dofs[:, 1], None, dev))
            corrected.append(diff)
            if keep_uncorrected:
                uncorrected.append(acc)
            if keep_classes:
                self.classes[name] = (prs, dofs, acc, corr)
            del corr
        if rows:
            r = torch.cat(rows)
            c = torch.cat(cols)
            self.mat = bcoo_to_bsr_dev(r, c, torch.cat(corrected), self.shape)
            self.mat_no_correction = (bcoo_to_bsr_dev(r, c, torch.cat(uncorrected), self.shape)
                                      if keep_uncorrected else None)
        else:
            z = torch.zeros((0, 81), dtype=torch.float64, device=dev)
            e = torch.zeros(0, dtype=torch.int64, device=dev)
            self.mat = bcoo_to_bsr_dev(e, e, z, self.shape)
            self.mat_no_correction = self.mat

    def _assemble_rows(self, classes, rules, far_q, pairs_int, corr_int, n_tris,
                       keep_uncorrected):
        """The matrix with every block integrated straight into its place.

        Each class comes sorted by (obs, src) from the finder, so a block's
        place is its rank in the merge of at most four sorted lists
        (tct_bsr_merge), and the integrators write there: no list of accurate
        blocks, list of corrections, difference, concatenation and reordering,
        each a pass over 648 bytes a pair.  Where both kernels are the same and
        the accurate rule is a product rule the correction is part of the
        same pass; otherwise it is subtracted in place.  Returns False,
        having done nothing, for lists that are not sorted (or dofs outside
        the matrix), which the general way below takes."""
        dev = self.device
        nr, nc = self.shape[0] // 9, self.shape[1] // 9
        # (name, pairs, dofs or None where they are the pairs', tests)
        work = []
        for name, prs, dofs, check0, corr_check0 in classes:
            if prs.shape[0] == 0:
                continue
            prs = np.ascontiguousarray(prs, dtype=np.int64)
            dofs = np.asarray(dofs, dtype=np.int64)
            if dofs.shape != (prs.shape[0], 2) or prs.shape[1] not in (2, 5):
                return False
            if dofs.strides[1] != 8 or dofs.strides[0] % 8 or dofs.strides[0] < 16:
                dofs = np.ascontiguousarray(dofs)
            same = ctypes.c_int(dofs is prs)
            if not same.value:
                N.call('tct_pairs_same', prs.shape[0], prs.shape[1], N.ptr(prs), N.ptr(dofs),
                       dofs.strides[0] // 8, ctypes.byref(same))
            work.append((name, prs, None if same.value else dofs, check0, corr_check0))
        if not work:
            return False
        # pairs, and dofs where they are others, as int32 in one pinned
        # buffer: one conversion pass, one copy
        n = [c[1].shape[0] for c in work]
        width = [c[1].shape[1] for c in work]
        own = [c[2] is not None for c in work]
        size = [k * (w + 2 * o) for k, w, o in zip(n, width, own)]
        off = np.concatenate([[0], np.cumsum(size)]).astype(np.int64)
        host = torch.empty(int(off[-1]), dtype=torch.int32, pin_memory=True)
        flag = ctypes.c_int(0)
        for (_, prs, dofs, _, _), o, k, w in zip(work, off, n, width):
            at = host.data_ptr() + 4 * int(o)
            d = dofs is not None
            rc = N.lib().tct_pairs_pack(
                k, w, N.ptr(prs), n_tris, N.ptr(dofs), dofs.strides[0] // 8 if d else 0, nr, nc,
                at, at + 4 * k * w if d else None, ctypes.byref(flag))
            if rc != 0 or not flag.value:
                check_pairs(prs, n_tris)      # raises for a bad pair
                return False
        buf = host.to(dev, non_blocking=True)
        total = sum(n)
        rank = torch.empty(total, dtype=torch.int32, device=dev)
        indices = torch.empty(total, dtype=torch.int32, device=dev)
        indptr = torch.empty(nr + 1, dtype=torch.int32, device=dev)
        start = np.concatenate([[0], np.cumsum(n)[:-1]]).astype(np.int64)
        ptrs = lambda base, offs: (ctypes.c_void_p * len(n))(*[base + 4 * int(i) for i in offs])
        dof_off = [o + (k * w if d else 0) for o, k, w, d in zip(off, n, width, own)]
        N.call('tct_bsr_merge', len(n), (ctypes.c_int64 * len(n))(*n),
               ptrs(N.ptr(buf), dof_off),
               (ctypes.c_int * len(n))(*[2 if d else w for w, d in zip(width, own)]), nr,
               ptrs(N.ptr(rank), start), N.ptr(indices), N.ptr(indptr), N.stream_ptr())
        data = torch.empty((total, 81), dtype=torch.float64, device=dev)
        same = corr_int is pairs_int
        plain = None
        lists = []
        for (name, _, _, check0, corr_check0), o, k, w, s in zip(work, off, n, width, start):
            p_dev = buf[int(o):int(o) + k * w].view(k, w)
            r_dev = rank[int(s):int(s) + k]
            q = rules[name]
            fused = (same and not keep_uncorrected and w == 2 and check0 == corr_check0 and
                     pairs_int.product_side(q, k) is not None)
            pairs_int.pairs_quad_rows(q, p_dev, check0, r_dev, data,
                                      minus=far_q if fused else None)
            if not fused:
                lists.append((p_dev, r_dev, corr_check0))
        if keep_uncorrected:
            plain = data.clone()
        for p_dev, r_dev, corr_check0 in lists:
            # the correction takes the triangles in their own frames
            corr_int.pairs_quad_rows(far_q, p_dev[:, :2].contiguous(), corr_check0, r_dev, data,
                                     subtract=True)
        self.mat = BSRMatrix(indptr, indices, data, self.shape)
        self.mat_no_correction = (BSRMatrix(indptr, indices, plain, self.shape)
                                  if keep_uncorrected else None)
        return True

    def dot_dev(self, x, out=None, accumulate=False, prec='f64'):
        """prec other than 'f64' uses the FP32 copy of the blocks when one
        exists (``use_f32_inner``)."""
        return self.mat.dot_dev(x, out, accumulate, prec)

    def use_f32_inner(self):
        """Keep an FP32 copy of the corrected blocks for inexact (inner)
        matvecs of mixed-precision solves; FP64 products are unchanged."""
        self.mat.make_f32()
        return self

    def dot(self, v):
        return self.mat.dot(v)

    def nearfield_no_correction_dot(self, v):
        return self.mat_no_correction.dot(v)

    def to_dense(self):
        return self.mat.to_dense()

    def no_correction_to_dense(self):
        return self.mat_no_correction.to_dense()

    def full_scipy_mat(self):
        return self.mat.to_scipy()

    def full_scipy_mat_no_correction(self):
        return self.mat_no_correction.to_scipy()
