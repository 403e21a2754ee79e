"""Km and Dm on the GPU where the pose matrices are no rotations to FP64 (poses from FP32
data, deformed ones): the derivative of the wrench with the matrices as they are given,
by every route an evaluation can take, for batches that mix them with exact rotations."""
import ctypes as C

import numpy as np
import pytest
import torch

from atac import _lib as L
from atac import workloads as W
from atac.batch import ContactBatch, DeviceGrid, DevicePoints, make_instance
from atac.bvh import BVHMesh
from hostcheck import hostcheck as H

pytestmark = pytest.mark.gpu

# FP64: both sides round a few hundred operations per contact, contracted differently;
# FP32: those of the FP32 terms (2^-24, some 100 of them, cancelling by up to 100)
TOL = {True: 1e-11, False: 1e-3}


def _scene(n_points):
    """Instances whose poses are rotations and FP32 or sheared ones in turn, without friction (no branch
    that a rounding can switch), and their host Km, Dm."""
    w = W.peg_in_hole(n_points=n_points, n_poses=8)
    rng = np.random.default_rng(41)
    pts = W.round_points_f32(w.point_sets[0])
    made = []
    for k, ins in enumerate(w.instances):
        E2 = W.pose(W.random_rotation(rng), rng.uniform(-2, 2, 3))
        E1 = E2 @ ins.E1
        exact = (E1.copy(), E2.copy())
        if k % 4 == 1:
            E1, E2 = E1.astype(np.float32).astype(np.float64), E2.astype(np.float32).astype(np.float64)
        elif k % 4 == 3:
            E1[:3, :3] = E1[:3, :3] @ (np.eye(3) + 1e-4 * np.eye(3, k=1))
        rest = (rng.normal(0, 0.3, 6), rng.normal(0, 0.3, 6))
        make = lambda A, B: make_instance(0, 0, 0, A, rest[0], B, rest[1], 0.01, 1e4, 1e3, 0.0, 10.0)
        made.append((make(*exact), make(E1, E2)))
    return w, pts, [m[0] for m in made], [m[1] for m in made]


@pytest.mark.parametrize("precise", [True, False], ids=["precise", "fp32"])
@pytest.mark.parametrize("route", ["instance", "pipeline", "replay", "replay_pipeline", "torch_graph", "torch_graph_pipeline", "host",
                                   "host_graph"])
def test_poses_as_given(gpu, route, precise):
    n_points = 5000 if route == "host_graph" else 1800
    w, pts, exact, given = _scene(n_points)
    ref = [H.eval_instance(w.grids[0], pts, i, deriv=True, precise=precise) for i in given]
    tuning = {"max_active": -1} if "pipeline" in route else None
    g = w.grids[0]
    grid = DeviceGrid(g.values, g.min_box, g.max_box, g.dxyz)
    b = ContactBatch([grid], [DevicePoints(w.point_sets[0])], given, tuning=tuning)
    out = b.alloc_outputs(deriv=True)
    if "replay" in route:
        b.set_instances(exact)
        b.graph_capture(out, deriv=True, precise=precise)
        b.graph_launch()
        for poses in (given, exact, given):
            b.set_instances(poses)
            b.graph_launch()
        torch.cuda.synchronize()
    elif "torch_graph" in route:   # captured with rotations only
        b.set_instances(exact)
        b.eval(deriv=True, precise=precise, out=out)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            b.eval(deriv=True, precise=precise, out=out)
        for poses in (exact, given):
            b.set_instances(poses)
            graph.replay()
        torch.cuda.synchronize()
    elif "host" in route:
        res = {k: np.empty(v.shape, dtype=np.int32 if k == "n_active" else np.float64) for k, v in out.items()}
        at = lambda k: res[k].ctypes.data_as(C.c_void_p)
        L.check(L.lib().atac_batch_eval_instances_host(b.handle, b.instances, b.n, b.flags(deriv=True, precise=precise),
                                                       at("fm"), at("Km"), at("Dm"), at("dfm_dp6"), at("n_active")))
        out = {k: torch.tensor(v) for k, v in res.items()}
    else:
        b.eval(deriv=True, precise=precise, out=out)
    seen = 0
    for i, r in enumerate(ref):
        assert int(out["n_active"][i]) == r["n_active"]
        # (a finite difference across cells magnifies a last-bit difference 1e10 times)
        if r["slow"][r["active"]].any() or r["n_active"] == 0:
            continue
        seen += i % 2
        for key in ("Km", "Dm"):
            p, q = out[key][i].cpu().numpy(), r[key]
            assert np.abs(p - q).max() <= TOL[precise] * np.abs(q).max(), (i, key, np.abs(p - q).max() / np.abs(q).max())
    assert seen > 0


@pytest.mark.parametrize("n", [300, 40000])
def test_bvh_poses_as_given(gpu, n):
    """Central differences of the BVH wrench at poses sheared by 1e-2: the block sums would be off by as much."""
    V, F = W.icosphere(1.0, levels=2)
    rng = np.random.default_rng(3)
    u = rng.normal(size=(n, 3))
    xi = 0.3 * u / np.linalg.norm(u, axis=1, keepdims=True)
    E1, E2 = W.pose(W.random_rotation(rng), [1.05, 0.1, -0.05]), W.pose(W.random_rotation(rng), rng.uniform(-1, 1, 3))
    E1 = E2 @ E1
    E1[:3, :3] = E1[:3, :3] @ (np.eye(3) + 1e-2 * np.eye(3, k=1))
    E2[:3, :3] = E2[:3, :3] @ (np.eye(3) + 1e-2 * np.eye(3, k=-1))
    phi = [rng.normal(0, 0.2, 6), rng.normal(0, 0.2, 6)]
    m = BVHMesh(V, F)
    f = lambda A, B, p, q, **kw: m.force(xi, A, p, B, q, 0.01, 1e4, 1e3, 0.0, 10.0, **kw)
    got = f(E1, E2, *phi, deriv=True)
    assert got["n_active"] > 10
    for k in range(12):   # the wrench is linear in the twists: exact up to FP64
        h = np.zeros(12)
        h[k] = 0.5
        p, q = (f(E1, E2, phi[0] + s * h[:6], phi[1] + s * h[6:])["fm"] for s in (1.0, -1.0))
        assert np.abs(got["Dm"][:, k] - (p - q)).max() <= 1e-9 * np.abs(got["Dm"]).max(), k
    zero = f(E1, E2, *phi, deriv=True, p6=True)
    assert np.array_equal(zero["Km"], got["Km"]) and np.isfinite(zero["dfm_dp6"]).all()
