"""CGS2 with its columns in registers (krylov.hip once_kernel) at the edges of
its forms: the columns a lane holds, the last tile, the basis size and the
problem size where another form takes over, and a scratch sized for the
walking form only.  The reference is torch FP64 of the same formula."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

# columns a lane holds: 2, 4, 8, 16, 26, 38, 50 by eight waves; past 130,048
# points the column sums are a launch of their own; past 400 columns they are
# walked
CASES = [(1, 1), (1, 63), (8, 64), (16, 65), (17, 1000), (32, 8370), (33, 8370), (64, 16384),
         (65, 16385), (128, 130048), (129, 130049), (5, 130049), (208, 131073), (209, 140001),
         (304, 4097), (305, 200000), (400, 130049), (400, 2049), (401, 2049), (401, 130049)]


@pytest.mark.parametrize('m,n', CASES)
def test_cgs2_forms_match_torch(m, n):
    from tectosaur_amd import _native as N
    g = torch.Generator(device='cuda').manual_seed(m + n)
    ld = n + 3   # odd rows: columns start at every alignment a double has
    V = torch.zeros((m, ld), dtype=torch.float64, device='cuda')
    V[:, :n] = torch.randn((m, n), generator=g, dtype=torch.float64, device='cuda') / n ** 0.5
    V[:, n:] = float('nan')   # what lies between the rows is never used
    w0 = torch.randn(n, generator=g, dtype=torch.float64, device='cuda')
    Vn = V[:, :n]
    h1 = Vn @ w0
    wr = w0 - Vn.t() @ h1
    h2 = Vn @ wr
    wr = wr - Vn.t() @ h2
    ref = torch.cat([h1 + h2, torch.linalg.vector_norm(wr).reshape(1)])
    nd = ctypes.c_int64(0)
    N.call('tct_krylov_scratch', m, n, ctypes.byref(nd))
    walk = 2 * min(max(-(-n // 1024), 1), 1024) * m + 2 * m
    assert walk <= nd.value
    outs = []
    for size in (nd.value, walk, None):
        guard = 64
        scratch = torch.full(((size or 0) + guard,), 7.0, dtype=torch.float64, device='cuda')
        w = w0.clone()
        h = torch.empty(m + 1, dtype=torch.float64, device='cuda')
        vn = torch.empty(n, dtype=torch.float64, device='cuda')
        if size is None:
            N.call('tct_cgs2_noalloc', m, n, ld, N.ptr(V), N.ptr(w), N.ptr(h), N.ptr(vn), None,
                   N.stream_ptr())
        else:
            N.call('tct_cgs2', m, n, ld, N.ptr(V), N.ptr(w), N.ptr(h), N.ptr(scratch), size,
                   N.ptr(vn), None, N.stream_ptr())
            assert bool((scratch[size:] == 7.0).all())
        # a sum of n products rounds by about sqrt(n) 1e-16 |v| |w| (6e-14 of
        # |w| at the largest n); 1e-12 of the scale leaves a margin
        scale = float(torch.cat([ref, w0]).abs().max()) + float(w0.norm())
        assert torch.allclose(h, ref, rtol=0, atol=1e-12 * scale)
        assert torch.allclose(w, wr, rtol=0, atol=1e-12 * scale)
        assert torch.equal(vn, w / h[m])
        outs.append((w, h))
    # the static scratch takes the same form as a full one: same bits
    assert torch.equal(outs[0][0], outs[2][0]) and torch.equal(outs[0][1], outs[2][1])
    short = torch.empty(walk, dtype=torch.float64, device='cuda')
    with pytest.raises(N.TctError, match='scratch'):
        N.call('tct_cgs2', m, n, ld, N.ptr(V), N.ptr(w0), N.ptr(outs[0][1]), N.ptr(short),
               walk - 1, None, None, N.stream_ptr())
