"""fit_loss on device tensors (its own kernels) against the same loss written as tensor
operations on the CPU: sizes around the workgroup, one atom, one replica, a million values;
tensors that the kernels do not take (strides, single precision) take the general path.
Sums of up to 3 M squares in FP64: 1e-13 relative; the residuals' gradients are the same
few roundings, 1e-15 of their largest."""
import pytest

pytestmark = pytest.mark.gpu


def _case(atoms, reps, dtype, seed=3):
    import torch
    g = torch.Generator().manual_seed(seed)
    F, Ft = (torch.randn((atoms, 3), generator=g, dtype=torch.float64).to(dtype) for _ in range(2))
    E, Et = (100.0 * torch.randn(reps, generator=g, dtype=torch.float64).to(dtype) for _ in range(2))
    n = torch.randint(1, 900, (reps,), generator=g).to(dtype)
    return F, E, Ft, Et, n


def _loss(F, E, Ft, Et, n, w):
    return ((F - Ft) ** 2).mean() + w * (((E - Et) / n) ** 2).mean()


@pytest.mark.parametrize("atoms,reps,w", [(1, 1, 0.1), (85, 64, 0.1), (86, 257, 2), (1000, 3, 0.0), (43691, 1, 0.1),
                                          (3, 70000, 0.5), (1000003, 1, 0.1)])
def test_fit_loss_device(atoms, reps, w):
    import torch
    from exastamp_amd.fitting import fit_loss
    case = _case(atoms, reps, torch.float64)
    out = []
    for dev, f in (("cpu", _loss), ("cuda", fit_loss)):
        F, E, Ft, Et, n = (t.to(dev, copy=True) for t in case)
        F, E = F.requires_grad_(), E.requires_grad_()
        args = (F, E, Ft, Et, n, w)
        L = f(*args)
        (3.0 * L).backward()
        out.append((L.detach().cpu(), F.grad.cpu(), E.grad.cpu()))
    (L0, F0, E0), (L1, F1, E1) = out
    assert L1.shape == L0.shape and abs(L1 - L0) <= 1e-13 * abs(L0)
    for a, b in ((F1, F0), (E1, E0)):
        assert a.shape == b.shape and (a - b).abs().max() <= 1e-15 * b.abs().max()


@pytest.mark.parametrize("how", ["strided", "float32", "create_graph"])
def test_fit_loss_general_path(how):
    import torch
    from exastamp_amd.fitting import fit_loss
    dtype = torch.float32 if how == "float32" else torch.float64
    case = _case(90, 5, dtype)
    F0, E0, Ft0, Et0, n0 = (t.double() for t in case)
    F0.requires_grad_(), E0.requires_grad_()
    _loss(F0, E0, Ft0, Et0, n0, 0.1).backward()
    F, E, Ft, Et, n = (t.cuda() for t in case)
    if how == "strided":
        F = F.t().contiguous().t()
    F.requires_grad_(), E.requires_grad_()
    L = fit_loss(F, E, Ft, Et, n, 0.1)
    gF, gE = torch.autograd.grad(L, (F, E), create_graph=how == "create_graph")
    tol = 1e-6 if how == "float32" else 1e-15
    for a, b in ((gF, F0.grad), (gE, E0.grad)):
        assert a.dtype == dtype and (a.detach().cpu().double() - b).abs().max() <= tol * b.abs().max()
