"""Batched N-bodies over a list of both layouts, points and whole triangles."""
import numpy as np
import pytest
import torch

from tectosaur_amd import mesh

pytestmark = pytest.mark.gpu


def _op(nq, K='elasticH3', params=(3e10, 0.25), n=6):
    from tectosaur_amd.sparse_farfield_op import TriToTriDirectFarfieldOp
    pts, tris = mesh.make_rect(n, n + 2, [[-1, 0, 1], [1, 0, 1], [1, 0.3, -1], [-1, -0.2, -1]])
    idx = np.arange(tris.shape[0])
    op = TriToTriDirectFarfieldOp(nq, K, list(params), pts, tris, np.float32, idx, idx)
    v = torch.as_tensor(np.random.default_rng(n).normal(size=op.shape[1]), device='cuda')
    op.nbody_gather(v, 'f32')
    return op


def test_a_list_of_both_layouts_and_rules():
    from tectosaur_amd.farfield import run_batched
    ops = [_op(nq, n=n) for nq, n in ((3, 9), (1, 6), (2, 8), (3, 5), (1, 12), (2, 7))]
    assert [op.tri is None for op in ops] == [True, False, False, True, False, False]
    single = [op.nbody_engine.run('f32').clone() for op in ops]
    for a, b in zip(single, run_batched([op.nbody_engine for op in ops])):
        assert torch.equal(a, b)
    for a, b in zip(single, run_batched([op.nbody_engine for op in ops], block=128)):
        assert torch.equal(a, b)


@pytest.mark.parametrize('nqs', [(1, 3), (3, 1), (1, 2), (1, 1), (3, 3)])
def test_differing_operators_are_refused(nqs):
    from tectosaur_amd import _native as N
    from tectosaur_amd.farfield import run_batched
    a = _op(nqs[0])
    for b in (_op(nqs[1], K='elasticT3'), _op(nqs[1], params=(3e10, 0.3))):
        with pytest.raises(N.TctError):
            run_batched([a.nbody_engine, b.nbody_engine])


@pytest.mark.parametrize('nq', [1, 3])
@pytest.mark.parametrize('shape', [(100, 1), (256, 3)])
def test_bad_launch_shapes_are_refused(nq, shape):
    from tectosaur_amd import _native as N
    from tectosaur_amd.farfield import run_batched
    with pytest.raises(N.TctError):
        run_batched([_op(nq).nbody_engine], *shape)
