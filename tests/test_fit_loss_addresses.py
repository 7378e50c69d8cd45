"""Which tensors the fitting loss reads by address."""


def test_fit_loss_addresses():
    """What the loss's kernels read by address: memory that holds the values (on the CPU
    here; the kernels take device tensors only)."""
    import torch
    from exastamp_amd.fitting import _addresses
    a, b = torch.arange(6.0, dtype=torch.float64).view(2, 3), torch.ones((), dtype=torch.float64)
    assert _addresses(a, b, a[1]) == [a.data_ptr(), b.data_ptr(), a.data_ptr() + 24]
    for other in (a.t(), a.float(), a[:0], a.to_sparse(), torch.nn.Parameter(a), a.to("meta"),
                  torch._neg_view(a), torch.ones(1, dtype=torch.complex128).conj().imag,
                  torch._efficientzerotensor((), dtype=torch.float64)):
        assert _addresses(a, other) is None
    seen = []

    class Spy(torch.autograd.Function):
        @staticmethod
        def forward(ctx, x):
            return 2.0 * x

        @staticmethod
        def backward(ctx, g):
            seen.append(_addresses(a, g))
            return 2.0 * g

    x = b.clone().requires_grad_()
    torch.autograd.grad(Spy.apply(x), x, torch.ones(4, dtype=torch.float64), is_grads_batched=True)
    torch.func.vmap(lambda v: seen.append(_addresses(a, v)) or v)(a)
    torch.func.grad(lambda v: (seen.append(_addresses(a, v)), v.sum())[1])(a)
    assert seen == [None, None, None]
