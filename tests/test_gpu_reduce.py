"""The per-instance sums over many tiles and items: tilings with a tile list shorter and
longer than a wavefront, and rows that fill the groups of lanes unevenly, give the sums of
one large tile (for the wrench, the scale column, the adjoint and the fused pass)."""
import numpy as np
import pytest

from atac import workloads as W
from atac.batch import batch_from_workload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [300, 16384, 16640, 33000])
def test_sums_do_not_depend_on_the_tiling(gpu, n):
    """256-point tiles: 2 to 129 of them. FP64 contact arithmetic, so the results differ by the order
    of the sums alone: 2^-53 times the number of terms (3e4) of a result's scale, the terms cancelling up to 1e3."""
    import torch
    w = W.peg_in_hole(n_points=n, n_poses=6)
    g = torch.tensor(np.random.default_rng(n).normal(size=(6, 12)), device="cuda")
    res = []
    for tile in (256, 8192):
        b = batch_from_workload(w, tuning={"tile_points": tile})
        out, grad = b.eval(p6=True, precise=True), b.vjp(g)
        plain = b.eval(precise=True)["fm"]
        f_out, f_grad = b.eval_vjp(g, precise=True)
        torch.cuda.synchronize()
        assert torch.equal(f_out["n_active"], out["n_active"])
        res.append([out["n_active"].double(), out["fm"], out["dfm_dp6"], plain, f_out["fm"], *grad.values(), *f_grad.values()])
    assert torch.equal(res[0][0], res[1][0]) and (n < 1000 or res[0][0].max() > 0)
    for p, q in zip(res[0], res[1]):
        assert torch.isfinite(p).all() and (p - q).abs().max() <= 1e-9 * q.abs().max().clamp(min=1e-300)


@pytest.mark.parametrize("precise", [False, True], ids=["fp32", "precise"])
def test_items_by_wavefront_and_by_workgroup(gpu, precise):
    """2,600 tiles (a wavefront per work item) against 120 (a workgroup per item). FP64 as above; FP32: a
    contact's terms are rounded alike, a lane's sums of up to four differ by 2^-24, the terms cancelling up to 1e2."""
    import torch
    w = W.peg_in_hole(n_points=16640, n_poses=40)
    g = torch.tensor(np.random.default_rng(5).normal(size=(40, 12)), device="cuda")
    res = []
    for tile in (256, 8192):
        b = batch_from_workload(w, tuning={"tile_points": tile})
        out, grad = b.eval(p6=True, precise=precise), b.vjp(g)
        plain = b.eval(precise=precise)["fm"]
        f_out, f_grad = b.eval_vjp(g, precise=precise)
        torch.cuda.synchronize()
        res.append([out["fm"], out["dfm_dp6"], plain, f_out["fm"], *grad.values(), *f_grad.values()])
    for p, q in zip(*res):
        assert torch.isfinite(p).all() and (p - q).abs().max() <= (1e-9 if precise else 1e-5) * q.abs().max()
