"""The source chunks of the triangle N-bodies: every wave of a launch's fullest
chunk with the same number of tiles, and a bounded number of chunks."""
import numpy as np
import pytest

from tectosaur_amd.tri_farfield import source_chunks


def _tiles(n_tiles, chunks):
    """Tiles of each chunk, as far_tri.h makes them: whole groups of four."""
    groups = -(-n_tiles // 4)
    assert chunks <= groups
    edge = [min(n_tiles, 4 * (groups * c // chunks)) for c in range(chunks + 1)]
    return np.diff(edge)


@pytest.mark.parametrize('resident', [256, 512, 1024, 2048])
def test_waves_take_equal_tiles(resident):
    rng = np.random.default_rng(resident)
    for _ in range(400):
        ob, nt = (int(x) for x in np.exp(rng.uniform(0, np.log([3000, 12000]))).astype(int))
        c = source_chunks(ob, nt, resident)
        assert 1 <= c <= min(512, -(-nt // 4))
        t = _tiles(nt, c)
        k = -(-int(t.max()) // 4)
        # chunks end between groups of four tiles (the last where the tiles do)
        assert t.sum() == nt and t.min() >= 1 and np.all(t[:-1] % 4 == 0)
        # one tile a wave unless that is more than 8,192 workgroups or 512 chunks
        groups = -(-nt // 4)
        if groups <= 512 and ob * groups <= 8192:
            assert k == 1 and c == groups


@pytest.mark.parametrize('n_tris', [1064, 1240, 1408])
def test_no_wave_waits_for_another_with_one_workgroup_a_cu(n_tris):
    # FP64 H with four points, one workgroup a CU: as many rounds of
    # workgroups as one tile a wave needs, never one with twice the tiles
    ob, nt = -(-n_tris // 64), -(-n_tris // 16)
    c = source_chunks(ob, nt, 256)
    k = -(-int(_tiles(nt, c).max()) // 4)
    assert -(-ob * c // 256) * k <= -(-ob * -(-nt // 4) // 256)
