"""tct_bsr39_spmv against numpy: row lengths around its eight lanes a row, rows
past a workgroup's, setting and adding."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('lens', [[0], [1], [7, 8, 9, 0, 16, 17, 63, 64, 65], [0] * 11 + [3],
                                  list(range(40))])
@pytest.mark.parametrize('accumulate', [0, 1])
def test_bsr39_matches_numpy(lens, accumulate):
    from tectosaur_amd import _native as N
    rng = np.random.default_rng(len(lens))
    n, nnz, cols = len(lens), sum(lens), 29
    indptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    idx = rng.integers(0, cols, max(nnz, 1)).astype(np.int32)
    data = rng.standard_normal((max(nnz, 1), 3, 9))
    x, y0 = rng.standard_normal(9 * cols), rng.standard_normal(3 * n)
    ref, size = np.zeros((n, 3)), np.zeros((n, 3))
    for i in range(n):
        for k in range(indptr[i], indptr[i + 1]):
            xv = x[9 * idx[k]:9 * idx[k] + 9]
            ref[i] += data[k] @ xv
            size[i] += np.abs(data[k]) @ np.abs(xv)
    ref, size = ref.reshape(-1) + accumulate * y0, size.reshape(-1) + accumulate * np.abs(y0)
    d = [torch.as_tensor(a, device='cuda') for a in (indptr, idx, data, x)]
    y = torch.as_tensor(y0, device='cuda').clone()
    N.call('tct_bsr39_spmv', n, *[N.ptr(a) for a in d], N.ptr(y), accumulate, N.stream_ptr())
    # at most 9 * 65 + 4 products and sums a row, each rounding 1.1e-16
    assert np.all(np.abs(y.cpu().numpy() - ref) <= 600 * 1.2e-16 * size + 1e-300)
