"""Contacts whose finite-difference stencil leaves their cell: a face of points on a cell
plane, where every contact takes the slow path."""
import numpy as np
import pytest
import torch

from atac.batch import ContactBatch, DeviceGrid, DevicePoints, make_instance

pytestmark = pytest.mark.gpu

N = 64
H = 2.0 / (N - 1)
AXIS = -1.0 + H * np.arange(N)
PLANE = float(np.float32(AXIS[30]))   # of nodes, below the face z = 0


def _batch(sizes, tuning=None):
    """A half space z < 0 and point sets of these sizes on the node plane."""
    z = np.ascontiguousarray(np.broadcast_to(AXIS[:, None, None], (N, N, N)).astype(np.float32))
    grid = DeviceGrid(z, np.full(3, -1.0), np.full(3, -1.0 + H * (N - 1)), np.full(3, H))
    rng = np.random.default_rng(5)
    sets = []
    for s in sizes:
        p = rng.uniform(-0.9, 0.9, (s, 3))
        p[:, 2] = PLANE
        sets.append(p)
    return ContactBatch([grid], [DevicePoints(np.concatenate(sets), np.cumsum([0] + list(sizes)).astype(np.int64))],
                        _poses(len(sizes), 0.0), tuning=tuning)


def _poses(n, lift):
    """Aligned with the grid, raised by `lift` cells."""
    rng = np.random.default_rng(6)
    E1 = np.eye(4)
    E1[2, 3] = lift * H
    return [make_instance(0, 0, i, E1, rng.normal(0, 0.1, 6), np.eye(4), np.zeros(6), 0.01, 1e4, 1e3, 0.3, 10.0)
            for i in range(n)]


@pytest.mark.parametrize("precise", [False, True], ids=["fp32", "precise"])
def test_more_than_the_slow_list_holds(gpu, precise):
    """The pipeline's slow list holds 4,096 contacts here: an evaluation with 6,000 is reported as overflowed, in
    NaN and n_active -1, whatever the pass that follows detection; the next one with fewer is right again."""
    b = _batch([2000, 2000, 2000], tuning={"max_active": -1})
    g = torch.ones((3, 12), dtype=torch.float64, device="cuda")
    for kw in ({}, {"p6": True}, {"deriv": True}):
        out = b.eval(precise=precise, **kw)
        grads = b.vjp(g)
        torch.cuda.synchronize()
        assert (out["n_active"] == -1).all() and b.workspace()["overflowed"]
        assert all(torch.isnan(v).all() for k, v in (*out.items(), *grads.items()) if k != "n_active")
    out, grads = b.eval_vjp(g, precise=precise)
    assert (out["n_active"] == -1).all() and torch.isnan(out["fm"]).all() and torch.isnan(grads["g_q1"]).all()
    b.set_instances(_poses(3, 0.4))   # off the plane: no slow contact
    out = b.eval(precise=precise, deriv=True)
    torch.cuda.synchronize()
    assert (out["n_active"] == 2000).all() and not b.workspace()["overflowed"]
    assert all(torch.isfinite(v).all() for v in out.values())


@pytest.mark.parametrize("precise", [False, True], ids=["fp32", "precise"])
@pytest.mark.parametrize("n", [1, 3, 127, 128, 129, 511, 512, 513, 640, 641, 2048, 3072])
def test_one_workgroup_equals_the_pipeline(gpu, n, precise):
    """Instances of slow contacts alone, around the numbers that one workgroup takes together: the samples have
    the pipeline's bits, the sums its order (terms of a few ulp: FP32 2^-24, FP64 2^-53, cancelling by up to 1e3)."""
    tol = 1e-12 if precise else 1e-4
    g = torch.tensor(np.random.default_rng(n).normal(size=(2, 12)), device="cuda")
    for kw in ({}, {"p6": True}, {"deriv": True}):
        res = []
        for tuning in (None, {"max_active": -1}):
            b = _batch([n, min(n, 1000)], tuning=tuning)
            out = b.eval(precise=precise, **kw)
            res.append({**out, **b.vjp(g)})
        torch.cuda.synchronize()
        assert res[0]["n_active"].tolist() == [n, min(n, 1000)]
        for k in res[0]:
            p, q = res[0][k].double(), res[1][k].double()
            assert torch.isfinite(p).all() and (p - q).abs().max() <= tol * q.abs().max(), k


def test_default_values_written_out(gpu):
    """A plan with the default values written out, or a plan's own values given back, is the default plan: small
    instances run in one workgroup, which holds 6,000 slow contacts where the pipeline's list overflows."""
    b = _batch([2000, 2000, 2000])
    info = b.info()
    own = {k: info[k] for k in ("tile_points", "detect_block", "blocks_per_cu", "order", "points_per_lane", "max_active", "group_cull")}
    for tuning in (None, {}, {"tile_points": 4096, "order": 1, "points_per_lane": 4}, {"group_cull": 1}, own):
        assert _batch([2000, 2000, 2000], tuning=tuning).eval()["n_active"].tolist() == [2000, 2000, 2000], tuning
        b.retune(tuning or {})
        assert b.eval()["n_active"].tolist() == [2000, 2000, 2000], tuning
    for tuning in ({"order": 4}, {"points_per_lane": 2}, {"detect_block": 64}, {"blocks_per_cu": 1}, {"max_active": 6000},
                   {"group_cull": -1}, {"tile_points": 2048}, {"tile_points": 8192}):
        b.retune(tuning)
        assert b.eval()["n_active"].tolist() == [-1, -1, -1], tuning


def test_autotune_times_the_default_plan():
    from atac.autotune import DEFAULT_CANDIDATES
    assert DEFAULT_CANDIDATES[0] == {}
