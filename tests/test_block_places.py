"""The places of nearfield blocks are checked against the matrix they go to,
also where they are the triangle pairs themselves."""
import ctypes

import numpy as np
import pytest

from tectosaur_amd import _native as N
from tectosaur_amd import mesh
from tectosaur_amd.nearfield_op import check_places


def _pack(pairs, n_tris, n_rows, n_cols, dofs=None):
    pairs = np.ascontiguousarray(pairs, dtype=np.int64)
    n, w = pairs.shape
    out = np.empty((n, w), dtype=np.int32)
    d32 = np.empty((n, 2), dtype=np.int32)
    flag = ctypes.c_int(-1)
    if dofs is not None:
        dofs = np.ascontiguousarray(dofs, dtype=np.int64)
    rc = N.lib().tct_pairs_pack(n, w, N.ptr(pairs), n_tris, N.ptr(dofs), 0 if dofs is None else 2,
                                n_rows, n_cols, N.ptr(out), None if dofs is None else N.ptr(d32),
                                ctypes.byref(flag))
    return rc, flag.value


@pytest.mark.parametrize('n', [3, 40000])      # serial and parallel loop
@pytest.mark.parametrize('width', [2, 5])
@pytest.mark.parametrize('own', [False, True])
def test_places_outside_the_matrix_are_refused(n, width, own):
    pairs = np.zeros((n, width), dtype=np.int64)
    pairs[:, 0] = np.arange(n) // 4
    pairs[:, 1] = np.arange(n) % 4
    rows, cols = int(pairs[-1, 0]) + 1, 4
    dofs = pairs[:, :2] if own else None
    assert _pack(pairs, 50000, rows, cols, dofs) == (0, 1)
    assert _pack(pairs, 50000, rows - 1 if rows > 1 else 0, cols, dofs)[0] < 0
    assert _pack(pairs, 50000, rows, int(pairs[:, 1].max()), dofs)[0] < 0


def test_check_places():
    d = np.array([[0, 3], [2, 1]])
    check_places(d, (27, 36))
    for shape in ((18, 36), (27, 27)):
        with pytest.raises(IndexError):
            check_places(d, shape)
    with pytest.raises(IndexError):
        check_places(d - [[0, 2]], (27, 36))


@pytest.mark.gpu
@pytest.mark.parametrize('keep', [False, True])     # in place, and the lists' way
@pytest.mark.parametrize('side', [0, 1])
def test_a_plan_of_more_triangles_than_the_subset_is_refused(side, keep):
    from tectosaur_amd.nearfield_op import RegularizedNearfieldIntegralOp, nearfield_plan
    pts, tris = mesh.make_icosphere([0, 0, 0], 1.0, 2)
    whole = np.arange(tris.shape[0])
    plan = nearfield_plan(pts, tris, whole, whole, 2.0)      # dofs equal pairs
    sub = [whole, whole]
    sub[side] = whole[:tris.shape[0] // 2]
    with pytest.raises(IndexError):
        RegularizedNearfieldIntegralOp(pts, tris, sub[0], sub[1], 3, 3, 3, 1, 3, 2.0,
                                       'elasticRH3', 'elasticRH3', [3e10, 0.25], np.float64,
                                       plan=plan, keep_classes=keep)
