"""fit_loss on device tensors whose memory does not hold their values, against the same
loss written as tensor operations on the CPU.  Sums of at most 300 squares in FP64: 1e-14
relative; the gradients are a few roundings, 1e-15 of their largest."""
import pytest

pytestmark = pytest.mark.gpu


def _inputs(reps):
    import torch
    g = torch.Generator().manual_seed(11)
    F, Ft = (torch.randn((100, 3), generator=g, dtype=torch.float64) for _ in range(2))
    E, Et = (100.0 * torch.randn(reps, generator=g, dtype=torch.float64) for _ in range(2))
    return F, E, Ft, Et, torch.randint(1, 900, (reps,), generator=g).double()


def _loss(F, E, Ft, Et, n, w):
    return ((F - Ft) ** 2).mean() + w * (((E - Et) / n) ** 2).mean()


def _negated(t):
    """t, as a view that negates memory holding -t"""
    import torch
    v = torch._neg_view(-t)
    assert v.is_neg() and v.is_contiguous() and torch.equal(v, t)
    return v


@pytest.mark.parametrize("which", ["F", "E", "Ft", "Et", "n"])
def test_fit_loss_negated_views(which):
    import torch
    from exastamp_amd.fitting import fit_loss
    case = _inputs(reps=4)
    ref = [t.clone().requires_grad_(k < 2) for k, t in enumerate(case)]
    L0 = _loss(*ref, 0.1)
    L0.backward()
    args = [t.cuda().requires_grad_(k < 2) for k, t in enumerate(case)]
    used = [_negated(t) if name == which else t for name, t in zip(("F", "E", "Ft", "Et", "n"), args)]
    L = fit_loss(*used, 0.1)
    L.backward()
    assert abs(L.item() - L0.item()) <= 1e-14 * abs(L0.item())
    for a, b in zip(args[:2], ref[:2]):
        assert (a.grad.cpu() - b.grad).abs().max() <= 1e-15 * b.grad.abs().max()


def test_fit_loss_imaginary_part_of_a_conjugate():
    import torch
    from exastamp_amd.fitting import fit_loss
    F, E, Ft, _, n = (t.cuda() for t in _inputs(reps=1))
    Et = torch.tensor([1.0 + 200.0j], dtype=torch.complex128, device="cuda").conj().imag
    assert Et.is_neg() and Et.item() == -200.0
    L, L0 = fit_loss(F, E, Ft, Et, n, 0.1).item(), _loss(F, E, Ft, torch.full_like(E, -200.0), n, 0.1).item()
    assert abs(L - L0) <= 1e-14 * abs(L0)


def test_fit_loss_batched_backward():
    """Several incoming gradients at once: the gradient that reaches the node is a batched
    tensor, which has no address."""
    import torch
    from exastamp_amd.fitting import fit_loss
    case = _inputs(reps=4)
    scales = torch.tensor([1.0, -2.5, 0.0], dtype=torch.float64)
    ref = [t.clone().requires_grad_(k < 2) for k, t in enumerate(case)]
    gF0, gE0 = torch.autograd.grad(_loss(*ref, 0.1), ref[:2])
    args = [t.cuda().requires_grad_(k < 2) for k, t in enumerate(case)]
    gF, gE = torch.autograd.grad(fit_loss(*args, 0.1), args[:2], scales.cuda(), is_grads_batched=True)
    for g, g0 in ((gF, gF0), (gE, gE0)):
        want = torch.stack([s * g0 for s in scales])
        assert g.shape == want.shape and (g.cpu() - want).abs().max() <= 2e-15 * want.abs().max()


@pytest.mark.parametrize("which", ["Ft", "Et"])
def test_fit_loss_zero_tensors(which):
    """Autograd's tensors of zeros, which have no memory"""
    import torch
    from exastamp_amd.fitting import fit_loss
    case = dict(zip(("F", "E", "Ft", "Et", "n"), _inputs(reps=4)))
    case[which] = torch.zeros_like(case[which])
    L0 = _loss(*case.values(), 0.1).item()
    used = {k: t.cuda() for k, t in case.items()}
    used[which] = torch._efficientzerotensor(case[which].shape, dtype=torch.float64, device="cuda")
    L = fit_loss(*used.values(), 0.1).item()
    assert abs(L - L0) <= 1e-14 * abs(L0)
