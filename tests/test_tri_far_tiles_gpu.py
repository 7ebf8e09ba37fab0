"""Far tiles of the triangle N-body run without the r2 test: on a mesh whose
triangles differ ten- or a thousandfold in size, with many tiles on both sides of the
separation, they give the same bits as the test on every tile (every operation
of the two bodies is written out), and in FP64 the sums of the point form with
its test on every tile.  (FP32 resolves no mesh of this grading to the
farfield's 1e-5 in either form: H reaches 2e-4 and 3e-4 with triangles a
thousandfold smaller than others.)"""
import numpy as np
import pytest
import torch

from tectosaur_amd import mesh

pytestmark = pytest.mark.gpu
KS = ['elasticU3', 'elasticT3', 'elasticA3', 'elasticH3', 'elasticRT3', 'elasticRA3',
      'elasticRH3']
TOL = 1e-12      # the FP64 farfield's, relative L2


def _graded(p):
    pts, tris = mesh.make_rect(80, 76, [[-1, 0, 1], [-1, 0, -1], [1, 0, -1], [1, 0, 1]])
    x, z = pts[:, 0], pts[:, 2]
    return np.stack([x * np.abs(x) ** p, 0.05 * x * x * z, z * np.abs(z) ** p], axis=1), tris


@pytest.mark.parametrize('grading', [0.5, 1.5])
@pytest.mark.parametrize('prec', ['f32', 'f64'])
@pytest.mark.parametrize('nq', [1, 2])
@pytest.mark.parametrize('K', KS)
def test_far_tiles_need_no_test(K, nq, prec, grading):
    from tectosaur_amd import _native as N
    from tectosaur_amd.sparse_farfield_op import TriToTriDirectFarfieldOp
    pts, tris = _graded(grading)
    n = tris.shape[0]
    ft = np.float32 if prec == 'f32' else np.float64
    args = (nq, K, [1.0, 0.25], pts, tris, ft, np.arange(n), np.arange(n))
    op = TriToTriDirectFarfieldOp(*args)
    t = op.tri
    # thousands of tiles closer and farther than the separation
    c = pts[tris].mean(1)
    tiles = c[t._t['src_tri'].cpu().numpy()][:n // 16 * 16].reshape((-1, 16, 3)).mean(1)
    far = np.linalg.norm(tiles[:, None] - c[None, ::7], axis=2) > t.group_extent
    assert 0.03 < far.mean() < 0.97
    v = torch.as_tensor(np.random.default_rng(3).standard_normal(9 * n), device='cuda')
    out = []
    for flags in (0, 1):
        t.plan.flags = flags
        out.append(op.dot_dev(v).clone())
    assert bool(torch.isfinite(out[0]).all())
    assert torch.equal(out[0], out[1])
    if prec == 'f32':
        return
    over_points = TriToTriDirectFarfieldOp(*args, tile_cfg=N.TileCfg(128, 1, 4, 1))
    ref = over_points.dot_dev(v, prec='f64')
    assert float((out[0] - ref).norm()) <= TOL * float(ref.norm())
