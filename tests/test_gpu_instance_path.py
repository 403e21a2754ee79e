"""Small batches run one workgroup per instance; a plan with a tuning runs the pipeline
of passes. Both give the same contacts, records and sums, at point counts around the
edges of the steps (64 points), the work items (256 contacts) and the range."""
import numpy as np
import pytest

from atac import workloads as W
from atac.batch import batch_from_workload

pytestmark = pytest.mark.gpu

SIZES = [0, 1, 63, 64, 65, 255, 256, 257, 1023, 1025, 2047, 2048]
SIZES_WRENCH = SIZES + [2049, 4095, 4096, 4097, 8191, 8192]
# the sums run in one order; a contact's terms are rounded alike up to the compiler's
# choice of fused multiply-adds: a few ulp of the largest term (FP32 2^-24, FP64 2^-53,
# times some 10 operations and a cancellation of up to 100 between the terms)
TOL = {False: 1e-4, True: 1e-12}


def _workload(sizes, pose_spread):
    """Every size at two poses: a peg that touches all round, and a face of points on
    the grid's cell planes (the slow path)."""
    w = W.peg_in_hole(n_points=max(max(sizes), 1), n_poses=2 * len(sizes))
    pts = W.round_points_f32(w.point_sets[0])
    pts[::7, 2] = np.round(pts[::7, 2] / 0.05) * 0.05 - 0.025
    w.point_sets = [pts[:s] for s in sizes]
    for k, ins in enumerate(w.instances):
        ins.points = k // 2
        if k % 2:
            ins.E1 = W.pose(np.eye(3), [pose_spread, 0.0, 0.025])
    return w


def _compare(w, kw):
    import torch
    a, b = batch_from_workload(w), batch_from_workload(w, tuning={"max_active": -1})
    g = torch.tensor(np.random.default_rng(3).normal(size=(a.n, 12)), device="cuda")
    res = []
    for x in (a, b):
        out = x.eval(**kw)
        grad = x.vjp(g)
        torch.cuda.synchronize()
        res.append((out, grad, x.workspace(), [x.active_ids(i) for i in range(x.n)]))
    tol = TOL[bool(kw.get("precise"))]
    for u, v in ((res[0][0], res[1][0]), (res[0][1], res[1][1])):
        assert set(u) == set(v)
        for k in u:
            p, q = u[k].cpu().numpy(), v[k].cpu().numpy()
            if k == "n_active":
                assert np.array_equal(p, q)
            else:
                assert np.isfinite(p).all() and np.abs(p - q).max() <= tol * max(np.abs(q).max(), 1e-300), k
    assert res[0][2]["used"] == res[1][2]["used"] > 0 and not res[0][2]["overflowed"]
    for p, q in zip(res[0][3], res[1][3]):
        assert np.array_equal(p, q)


@pytest.mark.parametrize("precise", [False, True], ids=["fp32", "precise"])
@pytest.mark.parametrize("kw", [{}, {"p6": True}, {"deriv": True, "p6": True}], ids=["wrench", "p6", "jacobian"])
def test_equals_the_pipeline(gpu, kw, precise):
    _compare(_workload(SIZES if kw else SIZES_WRENCH, 0.05), dict(kw, precise=precise))


@pytest.mark.parametrize("sizes", [[2049], [8193], [40] * 129, [40] * 257], ids=["2049", "8193", "258", "514"])
def test_around_the_rule(gpu, sizes):
    """One point more than the range, and batches on either side of an instance (two) per CU."""
    _compare(_workload(sizes, 0.05), {"deriv": True, "p6": True})
    _compare(_workload(sizes, 0.05), {})


def test_captured_and_replayed(gpu):
    """The path inside a captured graph: replays give what the eager call gave."""
    import torch
    b = batch_from_workload(_workload(SIZES, 0.05))
    want = {k: v.clone() for k, v in b.eval(deriv=True, p6=True).items()}
    out = b.alloc_outputs(deriv=True, p6=True)
    b.graph_capture(out, deriv=True, p6=True)
    for _ in range(3):
        for v in out.values():
            v.zero_()
        b.graph_launch()
        torch.cuda.synchronize()
        b.eval(p6=True)
        torch.cuda.synchronize()
        for k in want:
            assert torch.equal(out[k], want[k]), k


def test_several_tiles(gpu):
    """Instances of more than one tile, beside small and empty ones: the tiles' workgroups finish in any order, and
    every launch, replay and host call gives the same bits; the next launch starts from clear counts."""
    import ctypes as C

    import torch

    from atac import _lib as L
    sizes = [4097, 0, 8192, 100, 6240, 4096, 8191, 5000]
    w = _workload(sizes, 0.05)
    b, ref = batch_from_workload(w), batch_from_workload(w, tuning={"max_active": -1})
    g = torch.tensor(np.random.default_rng(3).normal(size=(b.n, 12)), device="cuda")
    for precise in (False, True):
        want, grads = b.eval(precise=precise), b.vjp(g)
        other, ograds = ref.eval(precise=precise), ref.vjp(g)
        out = b.alloc_outputs()
        for k, v in {**want, **grads}.items():
            q = {**other, **ograds}[k].double()
            assert (v - q).abs().max() <= (0 if k == "n_active" else TOL[precise]) * q.abs().max(), k
        for _ in range(50):
            b.eval(precise=precise, out=out)
            assert torch.equal(out["fm"], want["fm"]) and torch.equal(out["n_active"], want["n_active"])
        b.graph_capture(out, precise=precise)
        for _ in range(3):
            out["fm"].zero_()
            b.graph_launch()
            assert torch.equal(out["fm"], want["fm"])
        fm, na = np.zeros((b.n, 12)), np.zeros(b.n, dtype=np.int32)
        for _ in range(20):
            fm[:] = 0.0
            L.check(L.lib().atac_batch_eval_instances_host(b.handle, b.instances, b.n, b.flags(precise=precise),
                                                           fm.ctypes.data_as(C.c_void_p), None, None, None,
                                                           na.ctypes.data_as(C.c_void_p)))
            assert np.array_equal(fm, want["fm"].cpu().numpy()) and np.array_equal(na, want["n_active"].cpu().numpy())
        again = b.vjp(g)
        assert all(torch.equal(again[k], grads[k]) for k in grads)
        for i in (0, 4, 14):
            assert np.array_equal(b.active_ids(i), ref.active_ids(i))


def test_one_workgroup_for_several_tiles(gpu):
    """More tiles than three for two CUs: a workgroup takes all tiles of its instance."""
    _compare(_workload([4100, 8192] * 50, 0.05), {})
