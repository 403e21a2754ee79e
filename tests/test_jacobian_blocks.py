"""Km and Dm from the summed 3x3 blocks (contact_jac, jac_entry: what the batched
derivative evaluation computes) against the 24 tangents of contact_jvp, both in FP64
on the host, over the friction branches, both bodies moving and posed anywhere, and
points within the finite-difference step of cell faces (the slow path)."""
import numpy as np
import pytest

from atac import workloads as W
from atac.batch import make_instance
from hostcheck import hostcheck as H

# both sides round a few hundred FP64 operations per contact; the slow path's
# Hessian diagonal (up to 1 / 1e-5 of the slope jump) cancels up to 1e3 of it
TOL = 1e-11


@pytest.mark.parametrize("mu,kt,twist", [(0.3, 1e3, 0.1), (0.0, 1e3, 0.1), (0.3, 1e5, 2.0), (0.3, 0.0, 0.5)],
                         ids=["mixed", "frictionless", "dynamic", "kt0"])
def test_blocks_match_tangents(mu, kt, twist):
    w = W.peg_in_hole(n_points=1500, n_poses=6)
    g = w.grids[0]
    rng = np.random.default_rng(31)
    pts = W.round_points_f32(w.point_sets[0])
    seen = np.zeros(3, dtype=np.int64)
    for i, ins in enumerate(w.instances):
        E2 = W.pose(W.random_rotation(rng), rng.uniform(-2, 2, 3))
        if i == 0:   # the body frames aligned with the grid: points on cell faces
            E2, ins.E1 = np.eye(4), W.pose(np.eye(3), [0.05, 0.0, 0.025])
            pts[:200, 2] = np.round(pts[:200, 2] / 0.05) * 0.05 - 0.025
            pts = W.round_points_f32(pts)
        inst = make_instance(0, 0, 0, E2 @ ins.E1, rng.normal(0, twist, 6), E2, rng.normal(0, twist, 6), 0.01, 1e4, kt,
                             mu, 10.0, 1.3, 0.7)
        ref = H.eval_instance(g, pts, inst, deriv=True, precise=True)
        Km, Dm, counts, _ = H.jacobian_blocks(g, pts, inst)
        assert counts.sum() == ref["n_active"] > 0
        seen += counts
        for a, b in ((Km, ref["Km"]), (Dm, ref["Dm"])):
            assert np.abs(a - b).max() <= TOL * np.abs(b).max(), (i, np.abs(a - b).max() / np.abs(b).max())
    assert seen[2] > 0
    if (mu, kt) == (0.3, 1e5):
        assert seen[1] > 0
    if mu == 0.0 or kt == 0.0:
        assert seen[1] == 0


@pytest.mark.parametrize("defect", ["fp64", "products", "drift", "fp32", "scaled", "sheared"])
def test_poses_as_given(defect):
    """Km and Dm are the derivative of the wrench with the pose matrices as they are given, also
    where these are no rotations to FP64: poses from FP32 data, drifted or deformed ones."""
    w = W.peg_in_hole(n_points=1500, n_poses=6)
    rng = np.random.default_rng(7)
    pts = W.round_points_f32(w.point_sets[0])
    change = {"fp64": lambda R: R, "fp32": lambda R: R.astype(np.float32).astype(np.float64), "scaled": lambda R: 1.001 * R,
              "drift": lambda R: R @ (np.eye(3) + 2.0 ** -48 * rng.uniform(-1, 1, (3, 3))),
              "sheared": lambda R: R @ (np.eye(3) + 1e-3 * np.eye(3, k=1))}
    seen = 0
    for ins in w.instances:
        E2 = W.pose(W.random_rotation(rng), rng.uniform(-2, 2, 3))
        if defect == "products":
            for _ in range(50):
                E2 = E2 @ W.pose(W.random_rotation(rng), np.zeros(3))
        E1 = E2 @ ins.E1
        if defect in change:
            E1[:3, :3], E2[:3, :3] = change[defect](E1[:3, :3]), change[defect](E2[:3, :3])
        inst = make_instance(0, 0, 0, E1, rng.normal(0, 0.3, 6), E2, rng.normal(0, 0.3, 6), 0.01, 1e4, 1e3, 0.3, 10.0)
        ref = H.eval_instance(w.grids[0], pts, inst, deriv=True, precise=True)
        Km, Dm, counts, rigid = H.jacobian_blocks(w.grids[0], pts, inst)
        seen += counts.sum()
        off = max(np.abs(E[:3, :3].T @ E[:3, :3] - np.eye(3)).max() for E in (E1, E2))
        if defect in ("fp64", "products"):
            assert rigid, off
        if defect in ("fp32", "scaled", "sheared"):
            assert not rigid
        for a, b in ((Km, ref["Km"]), (Dm, ref["Dm"])):
            assert np.abs(a - b).max() <= TOL * np.abs(b).max(), (off, np.abs(a - b).max() / max(np.abs(b).max(), 1e-300))
    assert seen > 100
