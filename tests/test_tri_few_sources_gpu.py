"""Few source triangles against many observers: the waves of a workgroup share
the triangles of one or two tiles (far_tri.h, far_tri_pts.hip)."""
import numpy as np
import pytest
import torch

from tectosaur_amd import mesh

pytestmark = pytest.mark.gpu
PARAMS = [3e10, 0.25]
TOL = {'f32': 1e-5, 'f64': 1e-12}      # the farfield's, relative L2


def _mesh(nx, ny):
    pts, tris = mesh.make_rect(nx, ny, [[-1, 0, 1], [-1, 0, -1], [1, 0, -1], [1, 0, 1]])
    return pts + 0.02 * np.random.default_rng(nx).normal(size=pts.shape) / nx, tris


def _over_points(op, v, prec):
    op.engine
    op._gather(v, prec)
    op.engine.run(prec)
    y = torch.empty(op.shape[0], dtype=torch.float64, device='cuda')
    op._scatter(prec, y)
    return y


# one tile in four parts, two in two, three and four with one wave each
@pytest.mark.parametrize('n_src', [1, 2, 3, 4, 5, 16, 17, 19, 31, 32, 33, 48, 49, 64])
@pytest.mark.parametrize('prec,K,nq', [('f32', 'elasticH3', 1), ('f32', 'elasticRA3', 2),
                                       ('f64', 'elasticT3', 2), ('f64', 'elasticRH3', 1)])
def test_shared_tiles_give_the_sum(n_src, prec, K, nq):
    from tectosaur_amd.sparse_farfield_op import TriToTriDirectFarfieldOp
    pts, tris = _mesh(17, 15)
    n = tris.shape[0]
    op = TriToTriDirectFarfieldOp(nq, K, PARAMS, pts, tris, np.float32 if prec == 'f32' else
                                  np.float64, np.arange(150), np.arange(n - n_src, n))
    v = torch.as_tensor(np.random.default_rng(n_src).standard_normal(9 * n_src), device='cuda')
    ref = _over_points(op, v, 'f64')
    for chunks in range(1, op.tri.n_tiles + 1):
        op.tri.plan.chunks[op.tri.prec_id(prec)] = chunks
        op.tri._partial.clear()
        y = op.dot_dev(v)
        assert float((y - ref).norm()) <= TOL[prec] * float(ref.norm()), chunks


def _time(f):
    best = float('inf')
    for _ in range(10):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(10):
            f()
        b.record()
        b.synchronize()
        best = min(best, a.elapsed_time(b))
    return best


def test_few_sources_are_no_slower_than_over_points():
    # 0.7 of the point form's time; 2.0 with one wave of four at work
    from tectosaur_amd.sparse_farfield_op import TriToTriDirectFarfieldOp
    pts, tris = _mesh(200, 151)
    n = tris.shape[0]
    op = TriToTriDirectFarfieldOp(2, 'elasticH3', PARAMS, pts, tris, np.float64, np.arange(n),
                                  np.arange(9))
    v = torch.ones(81, dtype=torch.float64, device='cuda')
    y = torch.empty(op.shape[0], dtype=torch.float64, device='cuda')
    over_points = lambda: (op._gather(v, 'f64'), op.engine.run('f64'), op._scatter('f64', y))
    over_points()
    assert _time(lambda: op.dot_dev(v, y)) <= 1.3 * _time(over_points)
