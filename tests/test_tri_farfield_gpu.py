"""The triangle-to-triangle N-body (rules of three and four points) at the
edges of its layout: fewer observation triangles than a wave's 64 lanes, one
more, source counts around a tile of 16 and around the four tiles that the
waves of a workgroup take at a time.

Tolerances as the farfield's: FP64 1e-12, FP32 1e-5 relative L2 against the
long-double oracle."""
import numpy as np
import pytest
import torch

from tectosaur_amd import mesh
from tectosaur_amd.quadrature import gauss2d_tri

pytestmark = pytest.mark.gpu
KS = ['elasticU3', 'elasticT3', 'elasticA3', 'elasticH3', 'elasticRT3', 'elasticRA3',
      'elasticRH3']
TOL = {'f32': 1e-5, 'f64': 1e-12}


def _mesh(n):
    pts, tris = mesh.make_rect(n, n + 2, [[-1, 0, 1], [-1, 0, -1], [1, 0, -1], [1, 0, 1]])
    return pts + 0.03 * np.random.default_rng(n).normal(size=pts.shape), tris


def _rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize('n_obs,n_src', [(1, 1), (1, 80), (63, 15), (64, 16), (65, 17), (3, 63),
                                         (130, 65), (200, 200)])
@pytest.mark.parametrize('nq', [1, 2])
@pytest.mark.parametrize('K', KS)
def test_layout_edges(oracle, K, nq, n_obs, n_src):
    from tectosaur_amd.sparse_farfield_op import TriToTriDirectFarfieldOp
    pts, tris = _mesh(12)
    n = tris.shape[0]
    obs = np.arange(n_obs)
    src = np.arange(n - n_src, n)          # overlaps the observers when large
    v = np.random.default_rng(1).normal(size=n_src * 9)
    qx, qw = gauss2d_tri(nq)
    ref = oracle.farfield_tris(K, qx, qw, pts, tris[obs], tris[src], v, [3e10, 0.25])
    for prec, ft in (('f32', np.float32), ('f64', np.float64)):
        op = TriToTriDirectFarfieldOp(nq, K, [3e10, 0.25], pts, tris, ft, obs, src)
        assert op.tri is not None
        assert _rel(op.dot(v), ref) <= TOL[prec], prec


@pytest.mark.parametrize('prec', ['f32', 'f64'])
@pytest.mark.parametrize('K', KS)
def test_every_chunk_count_gives_the_sum(K, prec):
    # one chunk, chunks of less than a tile per wave, one tile per chunk
    from tectosaur_amd.sparse_farfield_op import TriToTriDirectFarfieldOp
    pts, tris = _mesh(14)
    n = tris.shape[0]
    op = TriToTriDirectFarfieldOp(1, K, [1.0, 0.25], pts, tris, np.float32, np.arange(n),
                                  np.arange(n))
    v = torch.as_tensor(np.random.default_rng(2).normal(size=n * 9), device='cuda')
    base = op.dot_dev(v, prec=prec).clone()
    t, pid = op.tri, op.tri.prec_id(prec)
    for c in (1, 2, 5, t.n_tiles):
        t.plan.chunks[pid] = c
        t._partial.clear()
        y = op.dot_dev(v, prec=prec)
        assert float((y - base).norm() / base.norm()) <= (1e-6 if prec == 'f32' else 1e-14), c


@pytest.mark.parametrize('prec', ['f32', 'f64'])
@pytest.mark.parametrize('K', ['elasticH3', 'elasticRH3', 'elasticU3'])
def test_batched_equals_single_and_the_whole_matvec(K, prec):
    # problems of several sizes in one table (more than one launch's worth)
    # have the bits of their own launches, and gather + N-body + scatter
    # those of the matvec call
    from tectosaur_amd import tri_farfield
    from tectosaur_amd.sparse_farfield_op import TriToTriDirectFarfieldOp
    ops, vs = [], []
    for k, nx in enumerate((5, 9, 14, 12, 7) * 4):
        pts, tris = _mesh(nx)
        n = tris.shape[0]
        obs = np.arange(n) if k % 3 else np.arange(n // 2, n)
        op = TriToTriDirectFarfieldOp(1, K, [3e10, 0.25], pts, tris, np.float32, obs,
                                      np.arange(n))
        v = torch.as_tensor(np.random.default_rng(k).normal(size=op.shape[1]), device='cuda')
        op.nbody_gather(v, prec)
        ops.append(op)
        vs.append(v)
    single = [op.tri.run(prec).clone() for op in ops]
    outs = tri_farfield.run_batched([op.tri for op in ops], prec)
    for a, b in zip(single, outs):
        assert torch.equal(a, b)
    for op, v in zip(ops, vs):
        y = torch.empty(op.shape[0], dtype=torch.float64, device='cuda')
        op.nbody_scatter(prec, y)
        assert torch.equal(y, op.dot_dev(v, prec=prec))


def test_other_rules_keep_the_point_layout():
    from tectosaur_amd import _native as N
    from tectosaur_amd.sparse_farfield_op import TriToTriDirectFarfieldOp
    pts, tris = _mesh(5)
    n = np.arange(tris.shape[0])
    args = ('elasticH3', [1.0, 0.25], pts, tris, np.float32, n, n)
    assert TriToTriDirectFarfieldOp(3, *args).tri is None            # seven points
    assert TriToTriDirectFarfieldOp(1, *args, tile_cfg=N.TileCfg(64, 1, 1, 0)).tri is None
    p = N.TriPlan(kernel=6, nq=7)
    import ctypes
    assert N.lib().tct_tri_gather(ctypes.addressof(p), 0, 1, None) < 0
    assert b'7 points' in N.lib().tct_last_error()
