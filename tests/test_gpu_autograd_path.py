"""The device route of contact_wrench (poses read by a kernel, pose gradients solved by
one) against the general route that tensors of another layout, type or place take."""
import numpy as np
import pytest
import torch

from atac import workloads as W
from atac.autograd import contact_wrench, se3_exp, tangent_pairing_matrix
from atac.batch import batch_from_workload

pytestmark = pytest.mark.gpu


def _inputs(w):
    f = lambda k: torch.tensor(np.stack([getattr(i, k) for i in w.instances]), dtype=torch.float64, device="cuda")
    return [f(k) for k in ("E1", "E2", "phi1", "phi2", "kn", "kt")]


# other forms of the same values; index: which inputs
FORMS = {"strided": lambda t: torch.stack([t, t], -1)[..., 0], "cpu": lambda t: t.cpu(),
         "neg": lambda t: torch._neg_view(-t), "rows": lambda t: t.reshape(t.shape[0], -1) if t.dim() == 3 else t}


@pytest.mark.parametrize("form", list(FORMS))
@pytest.mark.parametrize("n", [1, 2, 33])
def test_routes_agree(gpu, form, n):
    """Forward, instances kept and gradients: the same values reach the same kernels, so equal
    bits; the pose gradients are solved in another order (FP64, condition of a pose: below 1e2)."""
    w = W.peg_in_hole(n_points=700, n_poses=33)
    w.instances = w.instances[1:1 + n] if n < 33 else w.instances   # (pose 0 touches nothing)
    g = torch.tensor(np.random.default_rng(n).normal(size=(n, 12)), device="cuda")
    res = []
    for change in (lambda t: t, FORMS[form]):
        b = batch_from_workload(w)
        x = [change(t).detach() for t in _inputs(w)]
        for t in x[2:] if form == "rows" and len(res) else x:
            t.requires_grad_()
        fm = contact_wrench(b, *x)
        if form == "cpu" and len(res):   # the gradients are on the device: a forward pass only
            grads = [None] * 6
        elif form == "rows" and len(res):   # (a pose's gradient needs n x 4 x 4)
            grads = [None, None, *torch.autograd.grad(fm, x[2:], g)]
        else:
            grads = list(torch.autograd.grad(fm, x, g))
        res.append((fm.detach(), grads, bytes(b.instances)))
    assert torch.equal(res[0][0], res[1][0]) and res[0][2] == res[1][2]
    assert res[0][0].abs().max() > 0
    for k, (p, q) in enumerate(zip(res[0][1], res[1][1])):
        if q is None:
            continue
        q = q.to(p.device)
        assert torch.equal(p, q) if k >= 2 else (p - q).abs().max() <= 1e-12 * q.abs().max().clamp(min=1e-300)


@pytest.mark.parametrize("n", [1, 31, 32, 33, 64])
def test_pose_gradients(gpu, n):
    """Rigid and general matrices (row exchanges needed), and one that has no inverse."""
    b = batch_from_workload(W.peg_in_hole(n_points=8, n_poses=n))
    rng = np.random.default_rng(n)
    E1 = se3_exp(torch.tensor(rng.normal(0, 1, (n, 6)))).cuda()
    E2 = torch.tensor(rng.normal(0, 1, (n, 4, 4)) + 4 * np.eye(4)[[1, 0, 3, 2]], device="cuda")
    g1, g2 = (torch.tensor(rng.normal(0, 1, (n, 6)), device="cuda") for _ in range(2))
    got1, got2, bad = b.pose_gradients(E1, g1, E2, g2)
    assert bad == 0
    for got, E, g in ((got1, E1, g1), (got2, E2, g2)):
        want = tangent_pairing_matrix(E, g)
        cond = float(torch.linalg.cond(E).max())
        assert (got - want).abs().max() <= 64 * 2.0 ** -52 * cond * want.abs().max()
    only, none, bad = b.pose_gradients(E1, g1, None, None)
    assert none is None and torch.equal(only, got1) and bad == 0
    E2[n - 1, 3] = 0.0
    assert b.pose_gradients(E1, g1, E2, g2)[2] == 1


def test_singular_pose_raises(gpu):
    w = W.peg_in_hole(n_points=100, n_poses=2)
    b = batch_from_workload(w)
    x = _inputs(w)
    x[0][1, 3] = 0.0   # the last row is not read by the evaluation
    x = [t.requires_grad_() for t in x]
    fm = contact_wrench(b, *x)
    with pytest.raises(torch.linalg.LinAlgError):
        fm.sum().backward()
    x[0] = x[0].detach()   # its gradient is not asked for
    torch.autograd.grad(contact_wrench(b, *x).sum(), x[1:])


def test_second_derivative_keeps_its_graph(gpu):
    w = W.peg_in_hole(n_points=300, n_poses=2)
    b = batch_from_workload(w)
    x = [t.requires_grad_() for t in _inputs(w)]
    gE, = torch.autograd.grad(contact_wrench(b, *x).sum(), x[:1], create_graph=True)
    assert gE.requires_grad and torch.isfinite(torch.autograd.grad(gE.sum(), x[0])[0]).all()


def _same_rows(E): E[2] = E[0]
def _same_columns(E): E[:, 2] = E[:, 0]
def _sum_of_rows(E): E[2] = E[0] + E[1]
def _ones(E): E[:] = 1.0
def _flat(E): E[:3, :3] = np.outer(E[:3, 0], E[0, :3])
def _near(E): E[2] = E[0] * (1 + 1e-15)
def _nan(E): E[3, 3] = np.nan
def _tall(E): E[:3, 3] = [1e9, -2e9, 3e8]


@pytest.mark.parametrize("change", [_same_rows, _same_columns, _sum_of_rows, _ones, _flat, _near, _nan, _tall])
def test_poses_without_an_inverse(gpu, change):
    """What torch refuses to invert is refused, also where the elimination leaves a rounding in place of a zero;
    what torch inverts gives torch's gradient."""
    w = W.peg_in_hole(n_points=100, n_poses=6)
    b = batch_from_workload(w)
    rng = np.random.default_rng(9)
    for k in range(6):
        x = _inputs(w)
        E = np.eye(4)
        E[:3, :3], E[:3, 3] = W.random_rotation(rng), rng.uniform(-2, 2, 3)
        change(E)
        x[1][k] = torch.tensor(E, device="cuda")
        x = [t.requires_grad_() for t in x]
        g = torch.tensor(rng.normal(size=(6, 12)), device="cuda")
        fm = contact_wrench(b, *x)
        try:
            torch.linalg.inv(x[1].detach())
        except torch.linalg.LinAlgError:
            with pytest.raises(torch.linalg.LinAlgError):
                torch.autograd.grad(fm, x, g)
            continue
        got = torch.autograd.grad(fm, x, g)[1]
        want = tangent_pairing_matrix(x[1].detach(), b.vjp(g)["g_q2"])
        ok = torch.isfinite(want)
        assert torch.equal(ok, torch.isfinite(got))
        # FP64, a condition of up to 1e19 (tall): of each pose's largest entry
        scale = torch.where(ok, want, 0).abs().amax((1, 2), keepdim=True).clamp(min=1e-300)
        tol = 1e-12 if change is not _tall else 1e-6
        assert (torch.where(ok, got - want, 0).abs() <= tol * scale).all(), (k, change.__name__)
