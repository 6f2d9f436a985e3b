"""GPU parity of the fused row normalisation (csrc/unit_rows.hip) with F.normalize, forward and
backward, against fp64: fp32 4e-6 of the row's scale (a sum of up to 1024 squares, a square root, a
division and, backward, a second sum), bf16 results one rounding, 2^-8."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


def _close(got, ref, bar):
    err = (got.double() - ref).norm(dim=-1)
    assert bool((err <= bar * ref.norm(dim=-1).clamp_min(1e-20)).all()), float((err / ref.norm(dim=-1).clamp_min(1e-20)).max())


@pytest.mark.parametrize("rows,D", [(1, 1), (5, 3), (33, 64), (130, 128), (7, 130), (3, 257), (2, 1024)])
@pytest.mark.parametrize("dtype,autocast", [(torch.float32, False), (torch.bfloat16, False),
                                            (torch.bfloat16, True), (torch.float16, True)])
def test_unit_rows(device, rows, D, dtype, autocast):
    from verace_amd.hip_kernels import UnitRowsFunction, unit_rows
    g = torch.Generator(device).manual_seed(D)
    x = (3 * torch.randn(rows, D, generator=g, device=device)).to(dtype).requires_grad_()
    with torch.autocast("cuda", dtype=torch.bfloat16, enabled=autocast):
        y = unit_rows(x)
        ref_type = F.normalize(x, p=2, dim=-1).dtype
    assert y.dtype == ref_type and type(y.grad_fn).__name__ == UnitRowsFunction.__name__ + "Backward"
    dy = torch.randn(rows, D, generator=g, device=device).to(y.dtype)
    dx, = torch.autograd.grad(y, x, dy)
    x64 = x.detach().double().requires_grad_()
    y64 = F.normalize(x64, p=2, dim=-1)
    dx64, = torch.autograd.grad(y64, x64, dy.double())
    _close(y, y64.detach(), 4e-6 if y.dtype == torch.float32 else 2.0 ** -8)
    # the tangential part can be small against the gradient it is left of (all of it at D = 1)
    bar = (4e-6 if dtype == torch.float32 else 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11)
    scale = (dy.double().norm(dim=-1) / x64.norm(dim=-1)).detach()
    assert bool(((dx.double() - dx64).norm(dim=-1) <= bar * scale).all())


def test_unit_rows_special_rows(device):
    """Zero rows, rows below eps, NaN and infinite elements: as F.normalize, both ways."""
    from verace_amd.hip_kernels import unit_rows
    x = torch.randn(5, 8, device=device)
    x[0] = 0.0
    x[1] *= 1e-14
    x[2, 3] = float("nan")
    x[3, 1] = float("inf")
    a, b = x.clone().requires_grad_(), x.clone().requires_grad_()
    dy = torch.randn(5, 8, device=device)
    ya, yb = unit_rows(a), F.normalize(b, p=2, dim=-1)
    ga, gb = torch.autograd.grad(ya, a, dy)[0], torch.autograd.grad(yb, b, dy)[0]
    assert torch.allclose(ya, yb, rtol=1e-5, atol=1e-6, equal_nan=True)
    for r in (0, 1, 4):
        assert torch.allclose(ga[r], gb[r], rtol=1e-4, atol=1e-5 * float(gb[r].abs().max()))
    assert torch.isnan(ga[2]).all()


def test_unit_rows_double_backward(device):
    from verace_amd.hip_kernels import unit_rows
    x = torch.randn(4, 16, device=device, requires_grad=True)
    w = torch.randn(4, 16, device=device)
    out = []
    for f in (unit_rows, lambda t: F.normalize(t, p=2, dim=-1)):
        g, = torch.autograd.grad((f(x) * w).sum(), x, create_graph=True)
        out.append(torch.autograd.grad(g.pow(2).sum(), x)[0])
    assert torch.allclose(out[0], out[1], rtol=1e-4, atol=1e-5)


def test_unit_rows_observed(device):
    """A function mode, a trace and a compiler see F.normalize's ops, in the CHAM projections too."""
    from torch.overrides import TorchFunctionMode
    from verace_amd import ContinuousHolographicMemory
    from verace_amd.hip_kernels import unit_rows
    seen = []

    class Watch(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))
    x = torch.randn(3, 8, device=device)
    ref = F.normalize(x, p=2, dim=-1)
    m = ContinuousHolographicMemory(16, 32).to(device)
    with torch.no_grad(), Watch():
        y = unit_rows(x)
        m.project(torch.randn(1, 2, 16, device=device))
    assert seen.count(F.normalize) == 4 and torch.equal(y, ref)
    traced = torch.jit.trace(unit_rows, x)
    assert "PythonOp" not in str(traced.graph) and torch.equal(traced(2 * x), F.normalize(2 * x, p=2, dim=-1))
    assert torch.equal(torch.compile(unit_rows, backend="eager", fullgraph=True)(x), ref)


def test_replaced_project_runs_in_training(device):
    """A subclass's or an instance's own ``project(x, active_mask)`` is called as in inference."""
    from verace_amd import SSSDAttention
    calls = []

    class Own(SSSDAttention):
        def project(self, x, active_mask=None):
            calls.append(active_mask)
            return super().project(x, active_mask)
    torch.manual_seed(0)
    a, b = Own(64, 2, 16).to(device), SSSDAttention(64, 2, 16).to(device)
    b.load_state_dict(a.state_dict())
    x = torch.randn(2, 5, 64, device=device, requires_grad=True)
    mask = torch.ones(2, 5, device=device, dtype=torch.bool)
    ya, yb = a(x, active_mask=mask)[0], b(x, active_mask=mask)[0]
    assert len(calls) == 1 and calls[0] is mask and torch.allclose(ya, yb, rtol=1e-4, atol=1e-5)
    plain = b.project
    b.project = lambda x, active_mask=None: calls.append(b) or plain(x, active_mask)
    b(x)[0].sum().backward()
    assert calls[-1] is b and bool(x.grad.isfinite().all())
