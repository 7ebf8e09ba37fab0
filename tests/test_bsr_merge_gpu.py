"""Block lists merged into block rows (tct_bsr_merge): equal places within and
across lists, empty lists, rows without blocks, strides of pairs with frames."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('sizes', [(5,), (0, 7), (64, 1), (300, 0, 257), (40, 40, 40, 40),
                                   (1, 2000, 3, 511)])
@pytest.mark.parametrize('n_rows', [1, 3, 90])
def test_merge_is_a_stable_sort_of_the_lists(sizes, n_rows):
    from tectosaur_amd import _native as N
    rng = np.random.default_rng(sum(sizes) + n_rows)
    strides = [2 if k % 2 else 5 for k in range(len(sizes))]
    lists, dev, ranks = [], [], []
    for n, s in zip(sizes, strides):
        # rows and columns from a few values: many equal places
        d = np.stack([rng.integers(0, n_rows, n), rng.integers(0, 4, n)], axis=1)
        if n_rows > 3:
            d[:, 0] -= d[:, 0] % 3          # rows without blocks
        d = d[np.lexsort((d[:, 1], d[:, 0]))].astype(np.int32)
        wide = np.full((n, s), 7, dtype=np.int32)
        wide[:, :2] = d
        lists.append(d)
        dev.append(torch.as_tensor(wide, device='cuda'))
        ranks.append(torch.full((max(n, 1),), -1, dtype=torch.int32, device='cuda'))
    total = sum(sizes)
    indices = torch.full((max(total, 1),), -1, dtype=torch.int32, device='cuda')
    indptr = torch.full((n_rows + 1,), -1, dtype=torch.int32, device='cuda')
    k = len(sizes)
    N.call('tct_bsr_merge', k, (ctypes.c_int64 * k)(*sizes),
           (ctypes.c_void_p * k)(*[N.ptr(d) for d in dev]), (ctypes.c_int * k)(*strides), n_rows,
           (ctypes.c_void_p * k)(*[N.ptr(r) for r in ranks]), N.ptr(indices), N.ptr(indptr),
           N.stream_ptr())
    every = np.concatenate(lists)
    order = np.lexsort((every[:, 1], every[:, 0]))      # stable: earlier lists first
    place = np.empty(total, dtype=np.int64)
    place[order] = np.arange(total)
    at = 0
    for n, r in zip(sizes, ranks):
        assert np.array_equal(r.cpu().numpy()[:n], place[at:at + n])
        at += n
    assert np.array_equal(indices.cpu().numpy()[:total], every[order, 1])
    assert np.array_equal(indptr.cpu().numpy(),
                          np.searchsorted(every[order, 0], np.arange(n_rows + 1)))
