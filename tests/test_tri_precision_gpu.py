"""FP32 rounding of the forms over whole triangles against that of the point
form: both against FP64, on the same mesh, strengths and points.

The forms round the same quantities; where tiles, frames and sums of a triangle
form are no larger than the point form's, so are its errors, up to the scatter
of a median over thousands of outputs (about 1%) and of which roundings happen
to meet.  Bound: 1.1 times the point form's error."""
import numpy as np
import pytest
import torch

from tectosaur_amd import mesh

pytestmark = pytest.mark.gpu
PARAMS = [3e10, 0.25]
BOUND = 1.1


def _fault(nx, nz):
    """A fault of 2 km with vertices a little off the grid, in its plane and
    (0.2 m) out of it."""
    h = 2000.0 / nx
    w = h * nz
    pts, tris = mesh.make_rect(nx + 1, nz + 1, [[-1000, 0, 0], [1000, 0, 0], [1000, 0, -w],
                                                [-1000, 0, -w]])
    off = np.random.default_rng(nx * nz).uniform(-0.01 * h, 0.01 * h, pts.shape)
    return pts + off * [1, 0.3, 1], tris


def _errors(y, ref):
    return torch.linalg.vector_norm((y - ref).reshape(-1, 3), dim=1)


def _points_form(op, v, prec):
    e = op.engine
    e.gather_tris(v, op.tri_of_pt, op.qphi, op.wj_src, op.nq, prec)
    e.run(prec)
    e.reduce_pts(prec, op._packed)
    y = torch.empty_like(op._packed)
    y.index_copy_(0, op.po_dev, op._packed)
    return y


@pytest.mark.parametrize('K,nq', [('elasticU3', 1), ('elasticT3', 1), ('elasticA3', 1),
                                  ('elasticH3', 1), ('elasticU3', 2), ('elasticT3', 2),
                                  ('elasticA3', 2), ('elasticH3', 2), ('elasticU3', 3),
                                  ('elasticT3', 3), ('elasticA3', 3)])
def test_points_beside_the_surface(K, nq):
    from tectosaur_amd.interior import TriToPtDirectFarfieldOp
    pts, tris = _fault(32, 32)
    xs = np.linspace(-3000, 3000, 100)
    X, Y = np.meshgrid(xs, xs)
    rng = np.random.default_rng(7)
    obs = np.stack([X.ravel(), Y.ravel(), np.full(X.size, -520.0)], axis=1)
    obs += rng.uniform(-5, 5, obs.shape)
    ns = np.tile([0.0, 0.0, 1.0], (obs.shape[0], 1))
    op = TriToPtDirectFarfieldOp(obs, ns, (pts, tris), K, nq, PARAMS, np.float32,
                                 precisions=('f32', 'f64'))
    assert op.tri is not None
    v = torch.as_tensor(rng.standard_normal(9 * tris.shape[0]), device='cuda')
    ref = _points_form(op, v, 'f64')
    tri = _errors(op.dot_dev(v).reshape(-1, 3), ref)
    point = _errors(_points_form(op, v, 'f32'), ref)
    assert float(tri.median()) <= BOUND * float(point.median())
    # ... and the 200 points next to the fault's plane
    near = torch.as_tensor(np.argsort(np.abs(obs[:, 1]))[:200], device='cuda')
    assert float(tri[near].median()) <= BOUND * float(point[near].median())


@pytest.mark.parametrize('nq', [1, 2])
@pytest.mark.parametrize('K', ['elasticU3', 'elasticT3', 'elasticA3', 'elasticH3', 'elasticRT3',
                               'elasticRA3', 'elasticRH3'])
def test_triangles_of_curved_meshes(K, nq):
    # mean of the logarithm over meshes of several sizes and orientations: on
    # one mesh alone a tile that reaches across a fold of the Z-curve in one form
    # and not in the other decides
    from tectosaur_amd.sparse_farfield_op import TriToTriDirectFarfieldOp
    l2, med = [], []
    for seed in range(8):
        rng = np.random.default_rng(seed)
        pts, tris = mesh.make_rect(int(rng.integers(40, 75)), int(rng.integers(40, 75)),
                                   [[-1, 0, 1], [-1, 0, -1], [1, 0, -1], [1, 0, 1]])
        x, z = pts[:, 0], pts[:, 2]
        turn = np.linalg.qr(rng.standard_normal((3, 3)))[0]
        pts = np.stack([x, 0.05 * x * x * z, z], axis=1) @ turn + rng.uniform(-1, 1, 3)
        n = np.arange(tris.shape[0])
        op = TriToTriDirectFarfieldOp(nq, K, PARAMS, pts, tris, np.float32, n, n)
        assert op.tri is not None
        v = torch.as_tensor(rng.standard_normal(9 * n.size), device='cuda')
        op.engine
        out = []
        for prec in ('f32', 'f64'):
            op._gather(v, prec)
            op.engine.run(prec)
            y = torch.empty(op.shape[0], dtype=torch.float64, device='cuda')
            op._scatter(prec, y)
            out.append(y)
        point, ref = _errors(out[0], out[1]), out[1]
        tri = _errors(op.dot_dev(v, prec='f32'), ref)
        l2.append(float(tri.norm() / point.norm()))
        med.append(float(tri.median() / point.median()))
    assert np.exp(np.mean(np.log(l2))) <= BOUND
    assert np.exp(np.mean(np.log(med))) <= BOUND
