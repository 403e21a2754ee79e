"""The BVH's pruned search against all triangles, on the host in the kernel's arithmetic:
the same squared distance to the bit, and among equally near triangles the smallest face,
on meshes with many of them (finely split flat faces) and at points on them (vertices,
lattices), where an entry dropped a few FP32 steps too early shows."""
import numpy as np
import pytest

from hostcheck import hostcheck as H
from meshes import split_box, torus

BOX = (0.5, 0.5, 0.5)
SLAB = (0.37, 0.61, 0.83)


def _points(V, kind, n):
    lo, hi = V.min(0), V.max(0)
    rng = np.random.default_rng(17)
    if kind == "random":
        return rng.uniform(lo, hi, (n, 3))
    if kind == "near":     # close to the surface: box distances of nearly nothing
        p = V[rng.integers(len(V), size=n)] + rng.normal(size=(n, 3)) * 10.0 ** rng.uniform(-12, -2, (n, 1))
        return np.clip(p, lo, hi)
    if kind == "vertices":
        return V
    k = rng.integers(0, 97, (n, 3))
    return lo + (hi - lo) * k / 96.0


@pytest.mark.parametrize("kind", ["random", "near", "vertices", "lattice"])
@pytest.mark.parametrize("mesh", ["box", "slab", "torus", "one", "nine"])
def test_search_equals_all_triangles(mesh, kind):
    V, F = {"box": lambda: split_box(BOX, 16), "slab": lambda: split_box(SLAB, 13), "torus": lambda: torus(1.0, 0.35, 64, 33),
            "one": lambda: (np.eye(3), np.array([[0, 1, 2]])),
            "nine": lambda: (np.random.default_rng(2).normal(size=(27, 3)), np.arange(27).reshape(9, 3))}[mesh]()
    d2, f, bd2, bf, deepest = H.mesh_closest(V, F, _points(V, kind, 4000))
    assert np.array_equal(d2, bd2), (int((d2 != bd2).sum()), np.abs(d2 - bd2).max())
    assert np.array_equal(f, bf), int((f != bf).sum())
    assert deepest <= 80


def test_far_and_large_coordinates():
    """Squared distances past FP32's and near FP64's range: the keys stay ordered bounds."""
    V, F = split_box(BOX, 4)
    x = np.random.default_rng(5).normal(size=(300, 3))
    for scale in (1e-30, 1e18, 1e25, 1e150):
        d2, f, bd2, bf, _ = H.mesh_closest(V * scale, F, x * scale)
        assert np.array_equal(d2, bd2) and np.array_equal(f, bf), scale
