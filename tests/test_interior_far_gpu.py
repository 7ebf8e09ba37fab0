"""Interior points none of which is close to the surface: the farfield alone."""
import numpy as np
import pytest

from tectosaur_amd import mesh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('ft', [np.float32, np.float64])
def test_no_close_pair(ft):
    from tectosaur_amd.interior import InteriorOp, TriToPtDirectFarfieldOp
    pts, tris = mesh.make_rect(6, 5, [[-1, 0, 1], [-1, 0, -1], [1, 0, -1], [1, 0, 1]])
    obs = np.random.default_rng(0).uniform(20, 30, (70, 3))
    ns = np.tile([0.0, 0.0, 1.0], (70, 1))
    v = np.random.default_rng(1).standard_normal(9 * tris.shape[0])
    op = InteriorOp(obs, ns, (pts, tris), 'elasticT3', 4.0, 8, 2, 8, [1.0, 0.25], ft)
    assert op.n_blocks == 0
    far = TriToPtDirectFarfieldOp(obs, ns, (pts, tris), 'elasticT3', 2, [1.0, 0.25], ft)
    assert np.array_equal(op.dot(v), far.dot(v))
