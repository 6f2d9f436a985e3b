"""GPU parity of the fused element-wise layer steps (csrc/layer_ops.hip) against the torch ops
they replace, evaluated in fp64 on the same inputs, at the edges of their ranges; and that
everything the kernels must not take (grad mode, hooks, subclasses, odd shapes) runs the torch ops.

Bars per element: fp32 2e-6 of the value's scale (a few roundings of expf / tanhf / a sum of up to
1024 terms); bf16 / fp16: one rounding of the result (2^-8 / 2^-11) per step that the kernel rounds
(one for the activation and the coefficients; norm, add and norm: up to four)."""
import pytest
import torch
import torch.nn as nn

pytestmark = pytest.mark.gpu

EPS = {torch.float32: 2e-6, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}
DTYPES = [torch.float32, torch.bfloat16, torch.float16]


def _close(got, ref, bar):
    err = (got.double().cpu() - ref.cpu()).abs()
    assert bool((err <= bar * (ref.cpu().abs() + ref.cpu().pow(2).mean().sqrt())).all()), float(err.max())


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n,f", [(1, 8), (3, 264), (65, 2048)])
def test_situ_glu(device, dtype, n, f):
    from verace_amd.layer_ops import situ_glu
    g = torch.Generator(device).manual_seed(n)
    a, b = (10 * torch.randn(n, f, generator=g, device=device).to(dtype) for _ in range(2))
    with torch.no_grad():
        y = situ_glu(a, b, 4.0, 25.0)
    x, z = a.double(), b.double()
    ref = (4.0 * torch.tanh(x / 4.0) * torch.sigmoid(x)) * (25.0 * torch.tanh(z / 25.0))
    _close(y, ref, EPS[dtype])


def _coef_ref(logits, sig, vproj, k):
    n, C = logits.shape
    # equal logits by lowest index, as torch.topk gives them here
    order = torch.argsort(logits.double(), dim=-1, descending=True, stable=True)[:, :k]
    w = torch.full(logits.shape, float("-inf"), dtype=torch.double, device=logits.device)
    w = torch.softmax(w.scatter(-1, order, logits.double().gather(-1, order)), -1)
    r = vproj.shape[1] // C
    return (vproj.double().view(n, C, r) * torch.sigmoid(sig.double()).view(n, C, r) * w.unsqueeze(-1)).view(n, -1)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n,C,r,k", [(1, 64, 32, 8), (5, 64, 32, 8), (9, 16, 8, 8), (7, 3, 16, 3), (66, 40, 8, 1)])
def test_mcmoe_coef(device, dtype, n, C, r, k):
    from verace_amd.layer_ops import mcmoe_coef
    g = torch.Generator(device).manual_seed(n + C)
    # logits on a coarse grid, so that ties at the boundary of the top k are common
    logits = (torch.randn(n, C, generator=g, device=device) * 2).round().to(dtype) / 2
    sig, v = (torch.randn(n, C * r, generator=g, device=device).to(dtype) for _ in range(2))
    with torch.no_grad():
        y = mcmoe_coef(logits, sig, v, k)
        top = torch.zeros(n, C, device=device).scatter(1, torch.topk(logits, k, dim=-1)[1], 1.0)
    _close(y, _coef_ref(logits, sig, v, k), EPS[dtype])
    # the same components as torch.topk keeps (which of equal logits it keeps is its own choice: the
    # lowest indices at the model's 64 components, not always at other counts)
    kept = (y.view(n, C, r) != 0).any(-1).float()
    if C == 64:
        assert torch.equal(kept, top)
    inf = torch.full_like(logits, float("-inf"))
    assert torch.equal(torch.where(kept.bool(), logits, inf).sort(-1)[0], torch.where(top.bool(), logits, inf).sort(-1)[0])


def test_mcmoe_coef_nonfinite_logits(device):
    """NaN and infinite logits give NaN exactly where the torch ops do."""
    from verace_amd.layer_ops import mcmoe_coef
    logits = torch.randn(4, 16, device=device)
    logits[0, 3] = float("nan")
    logits[1, 5] = float("inf")
    logits[2] = float("-inf")
    sig, v = torch.randn(4, 128, device=device), torch.randn(4, 128, device=device)
    with torch.no_grad():
        y = mcmoe_coef(logits, sig, v, 4)
    with torch.enable_grad():   # the torch ops
        ref = mcmoe_coef(logits, sig, v, 4)
    assert torch.equal(torch.isnan(y), torch.isnan(ref))
    assert torch.isnan(y[:3]).all() and torch.isfinite(y[3]).all()


@pytest.mark.parametrize("dtype", DTYPES)
def test_mcmoe_coef_nonfinite_off_the_top_k(device, dtype):
    """Infinite and NaN projections and sigmas of components off the top k give NaN, as the torch
    ops' product with a weight of 0 does, in their own place alone."""
    from verace_amd.layer_ops import mcmoe_coef
    n, C, r, inf = 3, 16, 8, float("inf")
    logits = torch.arange(C, device=device).flip(0).expand(n, C).to(dtype).contiguous()   # 0 .. 3 kept
    sig, v = torch.zeros(n, C * r, device=device, dtype=dtype), torch.ones(n, C * r, device=device, dtype=dtype)
    v[0, 2 * r], v[0, 9 * r + 1], v[1, 15 * r + 7] = inf, -inf, float("nan")
    sig[1, 8 * r], sig[2, 5 * r + 2], sig[2, 6 * r], sig[2, 7 * r] = float("nan"), float("nan"), inf, -inf
    with torch.no_grad():
        y = mcmoe_coef(logits, sig, v, 4)
    with torch.enable_grad():   # the torch ops
        ref = mcmoe_coef(logits, sig, v, 4)
    assert int(torch.isnan(ref).sum()) == 4
    assert torch.equal(torch.isnan(y), torch.isnan(ref)) and torch.equal(torch.isinf(y), torch.isinf(ref))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rows,d", [(1, 8), (3, 1024), (67, 1032), (2, 4096)])
@pytest.mark.parametrize("which", ["norm", "add_norm", "norm_add_norm", "norm_add_add"])
def test_norm_add(device, dtype, rows, d, which):
    from verace_amd.layer_ops import norm_add
    g = torch.Generator(device).manual_seed(d)
    a, b, c = (torch.randn(rows, d, generator=g, device=device).to(dtype) for _ in range(3))
    n1, n2 = (nn.RMSNorm(d, eps=1e-6, device=device, dtype=dtype) for _ in range(2))
    for n in (n1, n2):
        n.weight.data = (1 + 0.1 * torch.randn(d, generator=g, device=device)).to(dtype)
    args = dict(norm=(a, None, None, None, n2), add_norm=(a, None, None, b, n2),
                norm_add_norm=(a, n1, None, b, n2), norm_add_add=(a, n1, c, b, None))[which]

    def norm64(x, n):
        return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + 1e-6) * n.weight.double()
    ref = a.double() if args[1] is None else norm64(a.double(), n1)
    for t in (args[2], args[3]):
        ref = ref if t is None else ref + t.double()
    with torch.no_grad():
        s, out = norm_add(*args)
    _close(s, ref, 3 * EPS[dtype])
    if args[4] is None:
        assert out is None
    else:
        _close(out, norm64(ref, n2), 4 * EPS[dtype])


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("b,s,d", [(1, 1, 8), (3, 5, 1024), (64, 1, 1032)])
def test_halting_updates_match_torch(device, dtype, b, s, d):
    """Loops of steps in all three modes against the torch ops in the same type, tokens halting at
    different steps (probabilities 0.1 .. 0.8 a step).  The halting probability's dot product may round
    the other way, so the accumulators are compared at one rounding a step and tokens within that of
    the threshold are left out."""
    from verace_amd import AdaptiveCognitiveDepthEngine
    torch.manual_seed(d)
    eng = AdaptiveCognitiveDepthEngine(d, 0.9).to(device, dtype)
    with torch.no_grad():
        eng.w_halting.weight.copy_(torch.randn(1, d) * 2 / d ** 0.5)
        eng.w_halting.bias.fill_(-0.5)
        x = torch.randn(b, s, d, device=device).to(dtype)
        layers = [_Shift(device, dtype, d, i) for i in range(6)]
        eng_ref = _TorchEngine(eng, d).to(device, dtype)
        got = eng.run(layers, x, 6, 2, step_states=_States(6), static_control=True)
        ref = eng_ref.run(layers, x, 6, 2, step_states=_States(6), static_control=True)
    near = ((got[1].float() - ref[1].float()).abs() > 0.5)   # a token that halted a step apart
    assert float(near.float().mean()) <= 0.05
    keep = ~near
    bar = 12 * EPS[dtype]
    assert float((got[1] - ref[1]).float().abs()[keep].max()) <= bar * 6
    assert float((got[0] - ref[0]).float().abs()[keep].max()) <= bar * float(ref[0].float().abs().max())
    assert 0 < int((ref[1] < 6).sum()) or b * s == 1


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("where", ["bias", "weight", "token", "infinite token", "infinite weight"])
def test_halting_updates_nonfinite(device, dtype, where):
    """NaN and infinite halting inputs and tokens: final states, depths and activity are NaN exactly
    where the torch ops make them so, whether the token is active, halts or has halted."""
    from verace_amd import AdaptiveCognitiveDepthEngine
    torch.manual_seed(3)
    d = 64
    eng = AdaptiveCognitiveDepthEngine(d, 0.9).to(device, dtype)
    with torch.no_grad():
        eng.w_halting.weight.copy_(torch.randn(1, d) / d ** 0.5)
        x = torch.randn(4, 3, d, device=device).to(dtype)
        bad = float("inf") if where.startswith("infinite") else float("nan")
        if where == "bias":
            eng.w_halting.bias.fill_(bad)
        elif where.endswith("weight"):
            eng.w_halting.weight[0, 5] = bad
        else:
            x[1, 2, 7] = bad
        layers = [_Shift(device, dtype, d, i) for i in range(4)]
        eng_ref = _TorchEngine(eng, d).to(device, dtype)
        got = eng.run(layers, x, 4, 1, step_states=_States(4), static_control=True)
        ref = eng_ref.run(layers, x, 4, 1, step_states=_States(4), static_control=True)
    for a, b in zip(got[:2], ref[:2]):
        assert torch.equal(torch.isnan(a), torch.isnan(b)) and torch.equal(torch.isinf(a), torch.isinf(b))
    if where in ("bias", "weight"):
        assert torch.isnan(ref[1]).all()


class _Shift(nn.Module):
    def __init__(self, device, dtype, d, i):
        super().__init__()
        g = torch.Generator().manual_seed(i)
        self.v = torch.randn(d, generator=g).to(device, dtype)

    def step_(self, h, st, mask):
        return h * 0.9 + 0.3 * self.v


class _States:
    def __init__(self, n):
        self.layers = [None] * n


def _TorchEngine(eng, d):
    from verace_amd import AdaptiveCognitiveDepthEngine

    class Sub(AdaptiveCognitiveDepthEngine):   # a subclass takes the torch ops
        pass
    e = Sub(d, eng.energy_threshold)
    e.load_state_dict(eng.state_dict())
    return e


def test_fused_steps_stand_aside(device):
    """Hooks fire, replaced sub-modules run and gradients flow as without the kernels."""
    from verace_amd import ManifoldContinuousMoE, SiTUGLU
    from verace_amd.layer_ops import fusable, norm_add
    m = ManifoldContinuousMoE(64, rank=8, num_components=16).to(device)
    x = torch.randn(2, 3, 64, device=device)
    with torch.no_grad():
        y = m(x)
    assert torch.allclose(y, m(x).detach(), rtol=1e-5, atol=1e-5)   # grad mode: torch ops
    m(x).sum().backward()
    assert all(p.grad is not None for p in m.parameters())
    seen = []
    m.norm.register_forward_hook(lambda *a: seen.append("norm"))
    m.base_situ_glu.register_forward_hook(lambda *a: seen.append("glu"))
    with torch.no_grad():
        assert torch.allclose(m(x), y, rtol=1e-5, atol=1e-5)
    assert seen == ["glu", "norm"]

    class Twice(SiTUGLU):
        def forward(self, t):
            return 2 * super().forward(t)
    t = Twice(64, 128).to(device)
    t.load_state_dict(m.base_situ_glu.state_dict())
    with torch.no_grad():
        assert torch.equal(t(x), 2 * SiTUGLU.forward(m.base_situ_glu, x))
        odd = torch.randn(3, 7, device=device)
        s, _ = norm_add(odd, b=odd)
        assert torch.equal(s, odd + odd)
        assert not fusable(x.cpu())
        with torch.autocast("cuda", dtype=torch.bfloat16):
            assert not fusable(x)
        assert torch.func.vmap(lambda v: norm_add(v, b=v)[0])(x).shape == x.shape


def test_fused_steps_keep_to_the_current_device(device, monkeypatch):
    """With another device current, as in a program of several, no kernel is launched."""
    from verace_amd import ManifoldContinuousMoE, _lib
    from verace_amd.hip_kernels import unit_rows
    m = ManifoldContinuousMoE(64, rank=8, num_components=16).to(device)
    x = torch.randn(2, 3, 64, device=device)
    with torch.no_grad():
        ref = m(x)
        monkeypatch.setattr(torch._C, "_cuda_getDevice", lambda: 1)
        monkeypatch.setattr(_lib, "load", lambda: pytest.fail("a kernel's entry point was loaded"))
        assert torch.allclose(m(x), ref, rtol=1e-5, atol=1e-5)
        assert torch.allclose(unit_rows(x).norm(dim=-1), torch.ones(2, 3, device=device), atol=1e-5)


@pytest.mark.parametrize("dtype", DTYPES)
def test_nonfinite_rows(device, dtype):
    """The activation and the norms are NaN and infinite exactly where the torch ops are."""
    from verace_amd.layer_ops import norm_add, situ_glu
    inf, nan, big = float("inf"), float("nan"), torch.finfo(dtype).max
    g = torch.Generator(device).manual_seed(1)
    a, b, c = (torch.randn(8, 64, generator=g, device=device).to(dtype) for _ in range(3))
    for t, vals in ((a, (inf, nan, big, -inf)), (b, (-inf, 1.0, big, inf)), (c, (0.0, 0.0, big, nan))):
        for r, x in enumerate(vals):
            t[r, 3 * r] = x
    n1, n2 = (nn.RMSNorm(64, device=device, dtype=dtype) for _ in range(2))

    def ops():
        return (situ_glu(a, b, 4.0, 25.0), situ_glu(b, c, 4.0, 25.0), *norm_add(a, b=b, norm2=n2),
                *norm_add(a, n1, b=b, norm2=n2), norm_add(a, n1, c, b)[0])
    with torch.no_grad():
        got = ops()
    with torch.enable_grad():
        ref = ops()
    for i, (x, y) in enumerate(zip(got, ref)):
        assert torch.equal(torch.isnan(x), torch.isnan(y)) and torch.equal(torch.isinf(x), torch.isinf(y)), i
    assert any(bool(torch.isnan(y).any()) for y in ref)
