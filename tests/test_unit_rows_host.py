"""A differentiated backward of the row normalisation against F.normalize on the host: first and second
derivatives, rows below eps, at zero and not finite."""
import types

import pytest
import torch
import torch.nn.functional as F


@pytest.mark.parametrize("scale", [1.0, 1e-11, 5e-13, 1e-14, 0.0, float("nan")])
def test_differentiated_backward(scale):
    from verace_amd.hip_kernels import UnitRowsFunction
    g = torch.Generator().manual_seed(1)
    x = (F.normalize(torch.randn(3, 16, generator=g, dtype=torch.double), dim=-1) * scale).requires_grad_()
    dy = torch.randn(3, 16, generator=g, dtype=torch.double, requires_grad=True)
    w = torch.randn(3, 16, generator=g, dtype=torch.double)
    hooks = []
    hook = x.register_hook(hooks.append)   # runs on the result, in the engine, not in here
    dx, none = UnitRowsFunction.backward(types.SimpleNamespace(saved_tensors=(x,)), dy)
    hook.remove()
    assert not hooks
    ref, = torch.autograd.grad(F.normalize(x, p=2, dim=-1), x, dy, create_graph=True)
    assert none is None
    torch.testing.assert_close(dx, ref, rtol=1e-9, atol=0.0, equal_nan=True)
    for a, b in zip(torch.autograd.grad(dx, (x, dy), w, allow_unused=True),
                    torch.autograd.grad(ref, (x, dy), w, allow_unused=True)):
        a, b = (torch.zeros_like(x) if t is None else t for t in (a, b))
        torch.testing.assert_close(a, b, rtol=1e-7, atol=1e-9 * float(b.detach().abs().nan_to_num().max()), equal_nan=True)
