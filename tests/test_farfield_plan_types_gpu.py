"""A farfield plan whose arrays have other types than farfield_plan's (index
arrays of 64 bits, points of 32, read-only arrays, as a file may give them) makes
the operator that its values describe."""
import numpy as np
import pytest
import torch

from tectosaur_amd import mesh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('nq', [1, 3])          # whole triangles, points
@pytest.mark.parametrize('K', ['elasticU3', 'elasticRH3'])
def test_plan_of_other_types(K, nq):
    from tectosaur_amd.sparse_farfield_op import TriToTriDirectFarfieldOp, farfield_plan
    pts, tris = mesh.make_rect(9, 8, [[-1, 0, 1], [-1, 0, -1], [1, 0, -1], [1, 0, 1]])
    n = np.arange(tris.shape[0])
    args = (nq, K, [1.0, 0.25], pts, tris, np.float64, n, n)
    plan = farfield_plan(nq, pts, tris, n, n, K == 'elasticRH3')
    v = np.random.default_rng(0).standard_normal(9 * n.size)
    ref = TriToTriDirectFarfieldOp(*args, plan=plan).dot(v)
    wide = dict(plan)
    for k in ('tri_of_pt', 'pt_of_tri'):
        wide[k] = plan[k].astype(np.int64)
    assert np.array_equal(TriToTriDirectFarfieldOp(*args, plan=wide).dot(v), ref)
    for k in ('o_pts', 's_pts', 'o_ns', 's_ns', 'o_wj', 's_wj'):
        wide[k] = plan[k].astype(np.float32)
    y = TriToTriDirectFarfieldOp(*args, plan=wide).dot(v)
    # points rounded to 1e-7 of their size, an eighth and more apart: r^-3 moves
    # by a few 1e-6 of a pair's term
    assert np.linalg.norm(y - ref) <= 1e-4 * np.linalg.norm(ref)


@pytest.mark.parametrize('K', ['elasticU3', 'elasticRH3'])
def test_plan_without_the_triangle_extent(K):
    # a plan made before it held one
    from tectosaur_amd.sparse_farfield_op import TriToTriDirectFarfieldOp, farfield_plan
    pts, tris = mesh.make_rect(9, 8, [[-1, 0, 1], [-1, 0, -1], [1, 0, -1], [1, 0, 1]])
    n = np.arange(tris.shape[0])
    args = (1, K, [1.0, 0.25], pts, tris, np.float32, n, n)
    plan = farfield_plan(1, pts, tris, n, n, K == 'elasticRH3')
    a = TriToTriDirectFarfieldOp(*args, plan=plan)
    del plan['tri_extent']
    b = TriToTriDirectFarfieldOp(*args, plan=plan)
    assert a.tri.group_extent == b.tri.group_extent > 0
    v = np.random.default_rng(0).standard_normal(9 * n.size)
    assert np.array_equal(a.dot(v), b.dot(v))
