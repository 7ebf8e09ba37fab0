"""Triangle-to-point farfield in FP32 (far_tri_pts.hip) against the FP64 point
N-body of the same operator, at the edges of its tiles (16 triangles), waves
(64 points) and rules, and at a point that lies on a source point."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

PARAMS = [1.0, 0.25]


def _problem(n_obs, n_src, seed):
    """Triangles of size 0.3 scattered in a 4 x 4 x 1 box, points in a layer
    0.5 to 1.5 above it."""
    rng = np.random.default_rng(seed)
    c = rng.uniform(0, 1, (n_src, 1, 3)) * [4, 4, 1]
    pts = (c + rng.uniform(-0.15, 0.15, (n_src, 3, 3))).reshape((-1, 3))
    tris = np.arange(3 * n_src).reshape((-1, 3))
    obs = rng.uniform(0, 1, (n_obs, 3)) * [4, 4, 1] + [0, 0, 1.65]
    ns = rng.standard_normal((n_obs, 3))
    return pts, tris, obs, ns / np.linalg.norm(ns, axis=1)[:, None], rng


# distances are 0.35 and more in a box of 4, so D carries about 12 FP32
# roundings' worth of relative error, r^-5 five times that: 4e-6 of a pair, of
# sums whose terms' sizes add to several times the largest output
TOL = 5e-5


@pytest.mark.parametrize('K', ['elasticU3', 'elasticT3', 'elasticA3', 'elasticH3'])
@pytest.mark.parametrize('nq', [1, 2, 3])
@pytest.mark.parametrize('n_obs,n_src', [(1, 1), (63, 15), (64, 16), (65, 17), (130, 64),
                                         (1000, 65), (7, 300)])
def test_points_match_fp64(K, nq, n_obs, n_src):
    from tectosaur_amd.interior import TriToPtDirectFarfieldOp
    pts, tris, obs, ns, rng = _problem(n_obs, n_src, 10 * n_obs + n_src)
    op = TriToPtDirectFarfieldOp(obs, ns, (pts, tris), K, nq, PARAMS, np.float32,
                                 precisions=('f32', 'f64'))
    assert (op.tri is None) == (K == 'elasticH3' and nq == 3)
    v = torch.as_tensor(rng.standard_normal(9 * n_src), device='cuda')
    ref = op.dot_dev(v, prec='f64')
    out = op.dot_dev(v)
    assert float((out - ref).abs().max()) <= TOL * float(ref.abs().max())
    # the same bits again, and into a caller's tensors of other forms
    again = torch.full((n_obs * 3,), float('nan'), dtype=torch.float64, device='cuda')
    assert op.dot_dev(v, again) is again and torch.equal(again, out)
    wide = torch.zeros(2 * 3 * n_obs, dtype=torch.float64, device='cuda')
    op.dot_dev(v, wide[::2])
    assert torch.equal(wide[::2], out) and not bool(wide[1::2].any())
    more = torch.zeros(3 * n_obs + 3, dtype=torch.float64, device='cuda')
    op.dot_dev(v, more)
    assert torch.equal(more[:3 * n_obs], out) and not bool(more[3 * n_obs:].any())
    with pytest.raises((RuntimeError, IndexError)):
        op.dot_dev(v, torch.zeros(3 * n_obs, dtype=torch.float32, device='cuda'))


@pytest.mark.parametrize('K', ['elasticU3', 'elasticH3'])
def test_point_on_a_source_point_is_skipped(K):
    from tectosaur_amd.interior import TriToPtDirectFarfieldOp
    from tectosaur_amd.quadrature import gauss2d_tri
    pts, tris, obs, ns, rng = _problem(70, 40, 5)
    q = gauss2d_tri(2)[0][2]
    t = pts[tris[23]]
    obs[11] = (1 - q[0] - q[1]) * t[0] + q[0] * t[1] + q[1] * t[2]
    op = TriToPtDirectFarfieldOp(obs, ns, (pts, tris), K, 2, PARAMS, np.float32,
                                 precisions=('f32', 'f64'))
    v = torch.zeros(9 * 40, dtype=torch.float64, device='cuda')
    v[9 * 30:] = torch.as_tensor(rng.standard_normal(90), device='cuda')
    far = op.dot_dev(v)[33:36].clone()
    # strengths on the point's own triangle add its other points' terms only
    v[9 * 23:9 * 24] = 1.0
    own = op.dot_dev(v)[33:36]
    assert bool(torch.isfinite(own).all()) and bool(torch.isfinite(far).all())
    ref = op.dot_dev(v, prec='f64')[33:36]
    # 0.06 between the rule's points where D was 0.35 above: six times TOL
    assert float((own - ref).abs().max()) <= 6 * TOL * float(ref.abs().max())


def test_forms_without_it_run_over_points():
    from tectosaur_amd import _native as N
    from tectosaur_amd.interior import TriToPtDirectFarfieldOp
    pts, tris, obs, ns, rng = _problem(20, 9, 1)
    args = (obs, ns, (pts, tris))
    assert TriToPtDirectFarfieldOp(*args, 'elasticRT3', 2, PARAMS, np.float32).tri is None
    assert TriToPtDirectFarfieldOp(*args, 'elasticH3', 3, PARAMS, np.float32).tri is None
    assert TriToPtDirectFarfieldOp(*args, 'elasticT3', 4, PARAMS, np.float32).tri is None
    assert TriToPtDirectFarfieldOp(*args, 'elasticT3', 2, PARAMS, np.float64).tri is None
    import ctypes
    p = N.TriPtsPlan(kernel=0, nq=13)
    assert N.lib().tct_tri_pts_matvec(ctypes.addressof(p), 1, 1, None) < 0
    assert b'13 points' in N.lib().tct_last_error()
