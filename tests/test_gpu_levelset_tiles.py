"""The level-set sweeps' tiling: 15 x 15 columns per workgroup, chunks of 4 steps along
x, tiles waiting for their lower neighbours. Grids at and around those sizes, long and
thin ones along each axis, and several tiles per axis, bit for bit against the CPU
restatement."""
import numpy as np
import pytest

import meshes as M
from oracle import oracle as O

pytestmark = pytest.mark.gpu

SIZES = [(2, 2, 2), (3, 16, 17), (4, 17, 16), (5, 31, 32), (17, 2, 47), (18, 46, 2), (67, 5, 3), (3, 4, 70), (2, 71, 16),
         (33, 32, 31), (40, 62, 47)]


@pytest.mark.parametrize("n", SIZES, ids=["x".join(map(str, s)) for s in SIZES])
def test_tile_edges_bitwise(gpu, n):
    from atac.sdfmesh import level_set
    V, F = M.torus(1.0, 0.35, 20, 11)
    ext = np.array([3.1, 3.0, 1.2])
    d = tuple(float(e / max(k - 1, 1)) for e, k in zip(ext, n))
    origin = (-1.55, -1.5, -0.6)
    ref = O.make_level_set3(V.astype(np.float32), F, origin, d, n, 1)
    got = level_set(V, F, origin, d, n, 1)
    assert np.array_equal(np.asarray(got).view(np.uint32), np.asarray(ref).view(np.uint32))


def test_more_lines_than_one_launch_holds(gpu):
    """2^26 x lines and more, a wavefront each: the signs of a box in the last corner of a flat grid are those
    of a small grid around it (coordinates of small whole numbers: the same distances)."""
    from atac.sdfmesh import level_set
    V, F = M.box(3.25)
    big, small = (1, 8200, 8200), (1, 20, 20)
    at = lambda n, off: (0.0, float(off - n[1]), float(off - n[2]))   # the box 10 nodes before the end
    got = level_set(V, F, at(big, 10), (1.0, 1.0, 1.0), big, 1)
    ref = level_set(V, F, at(small, 10), (1.0, 1.0, 1.0), small, 1)
    corner = got[-20:, -20:]
    assert np.array_equal(corner < 0, ref < 0) and (ref < 0).sum() == 49
    near = np.abs(ref) < 2.0
    assert np.array_equal(corner[near], ref[near])
    assert (got < 0).sum() == 49
