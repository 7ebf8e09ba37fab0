"""Group extents of point layouts: full and short groups, groups of a triangle's
points and of a tile's, and points that are NaN (left out, as where a grid of
observation points is masked)."""
import numpy as np
import pytest

from tectosaur_amd.farfield import group_extent


def _plain(p, group):
    best = 0.0
    for s in range(0, p.shape[0], group):
        q = p[s:s + group]
        q = q[~np.isnan(q).any(axis=1)]
        if q.size:
            best = max(best, np.linalg.norm(q - q.mean(axis=0), axis=1).max())
    return best


@pytest.mark.parametrize('group', [3, 4, 7, 48, 63, 64])
@pytest.mark.parametrize('n', [1, 2, 3, 4, 63, 64, 65, 200, 1001])
@pytest.mark.parametrize('nan', [False, True])
def test_against_a_plain_loop(group, n, nan):
    rng = np.random.default_rng(n)
    p = rng.standard_normal((n, 3)) * 10 + 100
    if nan and n > 2:
        p[rng.integers(0, n, max(1, n // 20))] = np.nan
        if np.isnan(p).all():
            return
    assert group_extent(p, group) == pytest.approx(_plain(p, group), rel=1e-13, abs=1e-12)


def test_no_points():
    assert group_extent(np.zeros((0, 3))) == 0.0


@pytest.mark.gpu
@pytest.mark.parametrize('K,nq', [('elasticT3', 3), ('elasticU3', 2), ('elasticH3', 1)])
def test_masked_observation_points(K, nq):
    import torch
    from tectosaur_amd import mesh
    from tectosaur_amd.interior import TriToPtDirectFarfieldOp
    pts, tris = mesh.make_rect(9, 8, [[-1, 0, 1], [-1, 0, -1], [1, 0, -1], [1, 0, 1]])
    obs = np.random.default_rng(0).uniform(0.3, 1, (200, 3))
    ns = np.tile([0.0, 0.0, 1.0], (200, 1))
    v = torch.as_tensor(np.random.default_rng(1).standard_normal(9 * tris.shape[0]),
                        device='cuda')
    args = ((pts, tris), K, nq, [1.0, 0.25], np.float32)
    whole = TriToPtDirectFarfieldOp(obs, ns, *args)
    assert whole.tri is not None
    ref = whole.dot_dev(v).reshape(-1, 3)
    obs = obs.copy()
    obs[70] = np.nan
    y = TriToPtDirectFarfieldOp(obs, ns, *args).dot_dev(v).reshape(-1, 3)
    # NaN at the point and at most at those packed with it
    bad = torch.isnan(y).any(1)
    assert bool(bad[70]) and int(bad.sum()) <= 64
    # in another packing: two FP32 roundings of distances of 0.3 and more
    assert float((y - ref)[~bad].abs().max()) <= 5e-5 * float(ref.abs().max())
