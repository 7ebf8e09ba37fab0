"""Two upward levels in one launch (tct_tree_m2m_pair) against two launches of
tct_tree_m2m, over level sizes with one to four children a node."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

C = {0: 4, 4: 13, 5: 4, 6: 12}   # channels of U, RT, RA, RH


@pytest.mark.parametrize('kid', sorted(C))
@pytest.mark.parametrize('order', [2, 3, 4])
@pytest.mark.parametrize('n_child', [1, 2, 3, 4, 5, 7, 8, 9, 70])
def test_pair_equals_two_levels(kid, order, n_child):
    from tectosaur_amd import _native as N
    rng = np.random.default_rng(n_child)
    terms = (order + 1) * (order + 2) * (order + 3) // 6
    n_par = -(-n_child // 2)
    n_g = -(-n_par // 2)
    c_off = 3
    p_off = c_off + n_child + 2
    g_off = p_off + n_par + 1
    n = g_off + n_g
    cr = np.concatenate([rng.uniform(-1, 1, (n, 3)), rng.uniform(0.5, 2, (n, 1))], axis=1)
    cr = torch.as_tensor(cr, device='cuda')
    for prec, dt, tol in ((N.F64, torch.float64, 1e-13), (N.F32, torch.float32, 3e-7)):
        m0 = torch.full((n, C[kid] * terms), 7.0, dtype=dt, device='cuda')
        m0[c_off:c_off + n_child] = torch.as_tensor(
            rng.standard_normal((n_child, C[kid] * terms)), device='cuda').to(dt)
        two, one = m0.clone(), m0.clone()
        N.call('tct_tree_m2m', kid, prec, order, p_off, n_par, c_off, n_child, N.ptr(cr),
               N.ptr(two), N.stream_ptr())
        N.call('tct_tree_m2m', kid, prec, order, g_off, n_g, p_off, n_par, N.ptr(cr), N.ptr(two),
               N.stream_ptr())
        N.call('tct_tree_m2m_pair', kid, prec, order, g_off, n_g, p_off, n_par, c_off, n_child,
               N.ptr(cr), N.ptr(one), N.stream_ptr())
        # FP64 sums of at most 280 products in another order (their sizes add
        # to a few hundred times the largest moment at most for a shift over
        # radius of 4, order 4: 1e-16 of that), rounded once to FP32
        scale = float(two.abs().max())
        assert float((one - two).abs().max()) <= tol * scale
        used = torch.zeros(n, dtype=torch.bool, device='cuda')
        used[p_off:p_off + n_par] = used[g_off:] = True
        assert torch.equal(one[~used], m0[~used])


def test_pair_refuses_other_orders():
    from tectosaur_amd import _native as N
    buf = torch.zeros(4096, dtype=torch.float64, device='cuda')
    p = N.ptr(buf)
    for order in (0, 1, 5, 8):
        rc = N.lib().tct_tree_m2m_pair(6, N.F64, order, 3, 1, 2, 1, 0, 2, p, p, N.stream_ptr())
        assert rc < 0 and b'order' in N.lib().tct_last_error()
