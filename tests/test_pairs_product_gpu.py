"""Product rules of the pair integrator and the way the outputs leave it:
pair counts around a wave's 64 lanes and the 8 or 16 pairs staged at a time,
rules whose points do not fill the lanes' groups, rotated and flipped pairs,
and the r = 0 test on coincident triangles.

Tolerance as the nearfield's: 1e-10 of each block's largest entry against the
long-double oracle."""
import numpy as np
import pytest
import torch

from tectosaur_amd import mesh
from tectosaur_amd.quadrature import gauss2d_tri, gauss4d_tri

pytestmark = pytest.mark.gpu
ALLK = ['elasticU3', 'elasticT3', 'elasticA3', 'elasticH3', 'elasticRT3', 'elasticRA3',
        'elasticRH3']
PARAMS = [3e10, 0.25]


def _mesh():
    pts, tris = mesh.make_icosphere([0, 0, 0], 1.0, 2)
    return pts + 0.01 * np.random.default_rng(3).normal(size=pts.shape), tris


def _far_pairs(tris, n, seed):
    """Pairs of triangles that share no vertex."""
    rng = np.random.default_rng(seed)
    p = rng.integers(0, tris.shape[0], (4 * n + 64, 2))
    touch = (tris[p[:, 0]][:, :, None] == tris[p[:, 1]][:, None, :]).any((1, 2))
    return p[~touch][:n]


def _close(got, want):
    got, want = got.reshape(-1, 81), want.reshape(-1, 81)
    scale = np.abs(want).max(axis=1, keepdims=True)
    return (np.abs(got - want) / scale).max()


@pytest.mark.parametrize('n,order', [(1, 1), (7, 2), (9, 3), (63, 1), (65, 2), (17, 4), (257, 1),
                                     (5, 5), (3, 6)])
@pytest.mark.parametrize('K', ALLK)
def test_product_rule_vs_oracle(oracle, K, n, order):
    from tectosaur_amd import _native as N
    from tectosaur_amd.pairs_integrator import PairsIntegrator
    pts, tris = _mesh()
    prs = _far_pairs(tris, n, n)
    q = gauss4d_tri(order, order)
    want = oracle.pairs_integrate(K, q[0], q[1], pts, tris, prs, False, PARAMS)
    pi = PairsIntegrator(K, PARAMS, np.float64, order, order, pts, tris)
    assert _close(pi.nearfield(prs), want) <= 1e-10
    # the product form by itself too, where the integrator takes the other
    side = [torch.as_tensor(a, device='cuda') for a in gauss2d_tri(order)]
    p = torch.as_tensor(prs.astype(np.int32), device='cuda')
    out = torch.full((n + 1, 81), 7.0, dtype=torch.float64, device='cuda')
    m = side[1].shape[0]
    N.call('tct_pairs_product', pi.kid, m, N.ptr(side[0]), N.ptr(side[1]), m, N.ptr(side[0]),
           N.ptr(side[1]), 0, None, None, N.ptr(pi.gpu_pts), N.ptr(pi.gpu_tris), n, N.ptr(p), 2, 0,
           pi.params.ctypes.data, None, 0, N.ptr(out), N.stream_ptr())
    out = out.cpu().numpy()
    assert _close(out[:n], want) <= 1e-10
    assert np.all(out[n] == 7.0)      # nothing past the last pair


@pytest.mark.parametrize('order', [1, 2, 3])
@pytest.mark.parametrize('K', ALLK)
def test_product_rule_coincident_rotated_flipped(oracle, K, order):
    from tectosaur_amd.pairs_integrator import PairsIntegrator
    pts, tris = _mesh()
    q = gauss4d_tri(order, order)
    pi = PairsIntegrator(K, PARAMS, np.float64, order, order, pts, tris)
    co = np.stack([np.arange(70)] * 2, axis=1)
    want = oracle.pairs_integrate(K, q[0], q[1], pts, tris, co, True, PARAMS)
    assert _close(pi.correction(co, True), want) <= 1e-10
    prs = _far_pairs(tris, 36, 5)
    k = np.arange(36)
    five = np.concatenate([prs, np.stack([k % 3, k // 3 % 3, k // 9 % 2], axis=1)], axis=1)
    want = oracle.pairs_integrate(K, q[0], q[1], pts, tris, five, False, PARAMS)
    assert _close(pi.pairs_quad(pi.near_q, five, False), want) <= 1e-10


@pytest.mark.parametrize('K', ['elasticRH3', 'elasticRT3', 'elasticRA3', 'elasticU3'])
def test_product_rule_many_pairs(K):
    # enough pairs for one lane a pair; the general 4-D rule is the reference
    from tectosaur_amd.pairs_integrator import PairsIntegrator
    pts, tris = _mesh()
    prs = np.repeat(_far_pairs(tris, 4001, 9), 40, axis=0)
    pi = PairsIntegrator(K, PARAMS, np.float64, 1, 3, pts, tris)
    p = torch.as_tensor(prs.astype(np.int32), device='cuda')
    got = pi.pairs_quad_dev(pi.near_q, p, False).cpu().numpy()
    want = pi.pairs_quad_dev(pi.near_q, p, False, lanes_per_pair=1).cpu().numpy()
    assert _close(got, want) <= 1e-10


@pytest.mark.parametrize('kernels', [('elasticRH3', 'elasticRH3'), ('elasticRH3', 'elasticH3'),
                                     ('elasticRT3', 'elasticRT3'), ('elasticU3', 'elasticU3')])
@pytest.mark.parametrize('which', ['whole', 'subset', 'keep', 'unsorted'])
def test_blocks_integrated_into_place_equal_the_lists(kernels, which):
    # the matrix assembled in place against the one from lists of accurate
    # blocks and corrections (keep_classes), for the whole mesh, subsets whose
    # dofs are not the triangles, the uncorrected matrix beside it, and a plan
    # that is not sorted (general way)
    from tectosaur_amd.nearfield_op import RegularizedNearfieldIntegralOp, nearfield_plan
    pts, tris = _mesh()
    n = tris.shape[0]
    obs, src = (np.arange(40, 170), np.arange(10, 200)) if which == 'subset' else \
        (np.arange(n), np.arange(n))
    plan = nearfield_plan(pts, tris, obs, src, 2.0)
    if which == 'unsorted':
        k = np.random.default_rng(0).permutation(plan['near'][0].shape[0])
        plan['near'] = tuple(a[k] for a in plan['near'])
    args = (pts, tris, obs, src, 3, 3, 3, 1, 3, 2.0) + kernels + (PARAMS, np.float64)
    keep = which == 'keep'
    a = RegularizedNearfieldIntegralOp(*args, plan=plan, keep_uncorrected=keep)
    b = RegularizedNearfieldIntegralOp(*args, plan=plan, keep_uncorrected=keep, keep_classes=True)
    assert a.counts == b.counts and a.n_pairs == b.n_pairs
    for x, y in ((a.mat, b.mat), (a.mat_no_correction, b.mat_no_correction))[:1 + keep]:
        assert torch.equal(x.indptr, y.indptr) and torch.equal(x.indices, y.indices)
        scale = y.data.abs().amax(1, keepdim=True)
        assert float(((x.data - y.data).abs() / scale).max()) <= 1e-10
    assert keep or a.mat_no_correction is None


def test_bad_plans_are_refused():
    from tectosaur_amd.nearfield_op import RegularizedNearfieldIntegralOp, nearfield_plan
    pts, tris = _mesh()
    idx = np.arange(tris.shape[0])
    for col, val, err in ((0, -1, IndexError), (1, tris.shape[0], IndexError),
                          (2, 3, ValueError), (4, 2, ValueError)):
        plan = nearfield_plan(pts, tris, idx, idx, 2.0)
        prs = plan['ea'][0].copy()
        prs[7, col] = val
        plan['ea'] = (prs, plan['ea'][1])
        with pytest.raises(err):
            RegularizedNearfieldIntegralOp(pts, tris, idx, idx, 3, 3, 3, 1, 3, 2.0, 'elasticRH3',
                                           'elasticRH3', PARAMS, np.float64, plan=plan)
