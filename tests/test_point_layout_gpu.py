"""The point layout of operators that run over whole triangles: its arrays are
there as on every operator, whoever asks first and on whichever stream, and an
operator that will need it has it from the start."""
import threading

import numpy as np
import pytest
import torch

from tectosaur_amd import mesh

pytestmark = pytest.mark.gpu
PARAMS = [3e10, 0.25]


def _tri(K='elasticRH3', **kw):
    from tectosaur_amd.sparse_farfield_op import TriToTriDirectFarfieldOp
    pts, tris = mesh.make_rect(9, 8, [[-1, 0, 1], [-1, 0, -1], [1, 0, -1], [1, 0, 1]])
    n = np.arange(tris.shape[0])
    return TriToTriDirectFarfieldOp(1, K, PARAMS, pts, tris, np.float32, n, n, **kw)


def _pts(precisions):
    from tectosaur_amd.interior import TriToPtDirectFarfieldOp
    pts, tris = mesh.make_rect(9, 8, [[-1, 0, 1], [-1, 0, -1], [1, 0, -1], [1, 0, 1]])
    obs = np.random.default_rng(0).uniform(0.2, 1, (90, 3))
    return TriToPtDirectFarfieldOp(obs, np.tile([0, 0, 1.0], (90, 1)), (pts, tris), 'elasticT3',
                                   2, PARAMS, np.float32, precisions=precisions)


@pytest.mark.parametrize('name', ['tri_of_pt', 'pt_of_tri', 'qphi', 'wj_src', 'wj_obs',
                                  'curl_src', 'curl_obs'])
def test_arrays_of_a_new_triangle_operator(name):
    from tectosaur_amd import _native as N
    op, points = _tri(), _tri(tile_cfg=N.TileCfg(64, 1, 1, 0))
    assert op.tri is not None and points.tri is None
    assert torch.equal(getattr(op, name), getattr(points, name))


@pytest.mark.parametrize('name', ['tri_of_pt', 'qphi', 'wj_src', 'po_dev'])
def test_arrays_of_a_new_point_operator(name):
    op, both = _pts(('f32',)), _pts(('f32', 'f64'))
    assert op.tri is not None
    assert torch.equal(getattr(op, name), getattr(both, name))


def test_an_unknown_attribute_is_one():
    with pytest.raises(AttributeError):
        _tri().no_such
    with pytest.raises(AttributeError):
        _tri('elasticU3').curl_obs


def test_threads_build_it_once(monkeypatch):
    from tectosaur_amd.sparse_farfield_op import TriToTriDirectFarfieldOp as Op
    op, made, make = _tri(), [], Op._make_points
    monkeypatch.setattr(Op, '_make_points', lambda self: (made.append(1), make(self))[1])
    got, gate = [], threading.Barrier(8)

    def ask():
        gate.wait()
        with torch.cuda.stream(torch.cuda.Stream()):
            got.append(op.engine)
    ts = [threading.Thread(target=ask) for _ in range(8)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert len(made) == 1 and len(got) == 8 and all(e is op.engine for e in got)


def test_built_on_one_stream_and_used_on_another():
    op = _tri()
    v = torch.as_tensor(np.random.default_rng(1).standard_normal(op.shape[1]), device='cuda')
    ref = op.dot_dev(v, prec='f64')
    torch.cuda.synchronize()
    with torch.cuda.stream(torch.cuda.Stream()):
        torch.cuda._sleep(20_000_000)      # the builder's stream is behind
        op.engine
    y = torch.empty_like(ref)
    op._gather(v, 'f64')
    op.engine.run('f64')
    op._scatter('f64', y)
    assert float((y - ref).norm()) <= 1e-12 * float(ref.norm())


def test_first_fp64_product_in_a_graph():
    # an operator of both precisions has both layouts from the start
    op = _pts(('f32', 'f64'))
    v = torch.as_tensor(np.random.default_rng(2).standard_normal(op.shape[1]), device='cuda')
    y = torch.zeros(op.shape[0], dtype=torch.float64, device='cuda')
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        op.dot_dev(v, y, 'f64')
    for k in range(3):
        v.mul_(1.5)
        y.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, op.dot_dev(v, prec='f64'))


def test_no_build_during_a_capture():
    from tectosaur_amd import _native as N
    op = _pts(('f32',))
    v = torch.ones(op.shape[1], dtype=torch.float64, device='cuda')
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        w = v * 2
        with pytest.raises(N.TctError, match='capture'):
            op.dot_dev(v, prec='f64')
    g.replay()
    torch.cuda.synchronize()
    assert bool((w == 2).all())
    assert op.dot_dev(v, prec='f64').shape[0] == op.shape[0]
