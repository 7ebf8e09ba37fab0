"""Pair integrals on few pairs: counts around the goes in which a wave's outputs
leave it (16 pairs), the counts from which a rule runs in another form or with
other lanes, and the time of a large rule on a few pairs."""
import numpy as np
import pytest
import torch

from tectosaur_amd import mesh

pytestmark = pytest.mark.gpu
ALLK = ['elasticU3', 'elasticT3', 'elasticA3', 'elasticH3', 'elasticRT3', 'elasticRA3',
        'elasticRH3']
TOL = 1e-10      # the nearfield's, of each block's largest entry


def _setup(K, nq_far, nq_near):
    from tectosaur_amd.pairs_integrator import PairsIntegrator
    pts, tris = mesh.make_icosphere([0, 0, 0], 1.0, 3)
    pts = pts + 0.003 * np.random.default_rng(3).normal(size=pts.shape)
    return PairsIntegrator(K, [1.0, 0.25], np.float64, nq_far, nq_near, pts, tris), tris


def _pairs(tris, n):
    rng = np.random.default_rng(n)
    p = rng.integers(0, tris.shape[0], (2 * n + 64, 2))
    touch = (tris[p[:, 0]][:, :, None] == tris[p[:, 1]][:, None, :]).any((1, 2))
    return torch.as_tensor(p[~touch][:n].astype(np.int32), device='cuda')


@pytest.mark.parametrize('K', ALLK)
@pytest.mark.parametrize('n', [1, 15, 16, 17, 63, 64, 65, 255, 257, 1000])
def test_few_pairs_of_a_small_rule(K, n):
    pi, tris = _setup(K, 2, 2)
    p = _pairs(tris, n)
    ref = pi.pairs_quad_dev(pi.far_q, p, True, lanes_per_pair=16)
    scale = ref.abs().amax(1, keepdim=True)
    for lanes in (0, 1, 4, 64):
        out = pi.pairs_quad_dev(pi.far_q, p, True, lanes_per_pair=lanes)
        assert float(((out - ref).abs() / scale).max()) <= TOL, lanes
    # into rows of a larger array, and subtracted from them
    rows = torch.as_tensor(np.random.default_rng(1).permutation(3 * n)[:n].astype(np.int32),
                           device='cuda')
    big = torch.full((3 * n, 81), 2.0, dtype=torch.float64, device='cuda')
    pi.pairs_quad_rows(pi.far_q, p, True, rows, big)
    assert float(((big[rows.long()] - ref).abs() / scale).max()) <= TOL
    pi.pairs_quad_rows(pi.far_q, p, True, rows, big, subtract=True)
    assert float((big[rows.long()].abs() / scale).max()) <= 2 * TOL
    rest = torch.ones(3 * n, dtype=torch.bool, device='cuda')
    rest[rows.long()] = False
    assert bool((big[rest] == 2.0).all())


@pytest.mark.parametrize('K', ALLK)
@pytest.mark.parametrize('n', [1, 511, 512, 1535, 1536])
def test_few_pairs_of_a_large_rule(K, n):
    pi, tris = _setup(K, 2, 8)
    p = _pairs(tris, n)
    ref = pi.pairs_quad_dev(pi.near_q, p, False, lanes_per_pair=16)
    scale = ref.abs().amax(1, keepdim=True)
    out = pi.pairs_quad_dev(pi.near_q, p, False)
    assert float(((out - ref).abs() / scale).max()) <= TOL


@pytest.mark.parametrize('n', [8191, 8192, 16383, 16384])
@pytest.mark.parametrize('K,nq', [('elasticT3', 5), ('elasticH3', 2), ('elasticU3', 2)])
def test_counts_where_the_form_changes(K, nq, n):
    pi, tris = _setup(K, 2, nq)
    p = _pairs(tris, n)
    ref = pi.pairs_quad_dev(pi.near_q, p, False, lanes_per_pair=16)
    scale = ref.abs().amax(1, keepdim=True)
    out = pi.pairs_quad_dev(pi.near_q, p, False)
    assert float(((out - ref).abs() / scale).max()) <= TOL


@pytest.mark.parametrize('K', ['elasticU3', 'elasticT3', 'elasticH3', 'elasticRT3'])
def test_a_large_rule_on_few_pairs_has_a_wave_a_pair(K):
    # a product rule shares a pair among at most 16 lanes, 1.2 to 1.9 times the
    # time of the 64 of the rule as it stands when a few pairs are all there is
    pi, tris = _setup(K, 2, 8)
    p = _pairs(tris, 60)
    out = torch.empty((60, 81), dtype=torch.float64, device='cuda')

    def best(lanes):
        t = float('inf')
        for _ in range(10):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(10):
                pi.pairs_quad_dev(pi.near_q, p, False, out, lanes_per_pair=lanes)
            b.record()
            b.synchronize()
            t = min(t, a.elapsed_time(b))
        return t
    assert best(0) <= 1.15 * best(64)
