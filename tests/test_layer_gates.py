"""What the fused layer steps may take, checked on the host with fake device tensors: parameters that
the torch ops refuse, convert or broadcast (another shape, type, device or tensor class) must reach those
ops, as the kernels read them as they stand.  (No case here may run on a device: a kernel given a
shorter weight would read past it.)"""
import pytest
import torch
import torch.nn as nn
from torch._subclasses.fake_tensor import FakeTensor, FakeTensorMode

from verace_amd import layer_ops

pytestmark = pytest.mark.filterwarnings("ignore:Accessing the data pointer of FakeTensor")

D = 64


@pytest.fixture
def mode(monkeypatch):
    """Fake tensors on cuda devices count as plain, aligned device tensors."""
    monkeypatch.setattr(layer_ops, "fusable", lambda x: True)
    monkeypatch.setattr(layer_ops, "_rows", lambda *ts: all(t is None or t.is_contiguous() for t in ts))
    monkeypatch.setattr(layer_ops, "_PLAIN", (torch.Tensor, nn.Parameter, FakeTensor), raising=False)
    return FakeTensorMode(allow_non_fake_inputs=True)


def _halting(mode, linear, threshold=0.9):
    with mode:
        h = torch.empty(2, 3, D, device="cuda:0")
        acc = torch.empty(2, 3, device="cuda:0")
    return layer_ops.HaltingState.start(linear(), threshold, h, h, acc, acc)


@pytest.mark.parametrize("change", ["narrow", "wide", "two outputs", "device", "bias device", "bias shape",
                                    "bias type", "no bias", "threshold"])
def test_halting_unit_must_fit(mode, change):
    def linear(change):
        with mode:
            d = {"narrow": D // 2, "wide": 2 * D}.get(change, D)
            m = nn.Linear(d, 2 if change == "two outputs" else 1, bias=change != "no bias",
                          device="cuda:1" if change == "device" else "cuda:0")
            b = {"bias device": dict(device="cuda:1"), "bias shape": dict(device="cuda:0"),
                 "bias type": dict(device="cuda:0", dtype=torch.float16)}.get(change)
            if b is not None:
                m.bias = nn.Parameter(torch.empty(2 if change == "bias shape" else 1, **b))
        return m
    assert _halting(mode, lambda: linear("")) is not None
    threshold = torch.tensor(0.9) if change == "threshold" else 0.9
    assert _halting(mode, lambda: linear(change), threshold) is None


@pytest.mark.parametrize("change", ["shorter", "longer", "device", "type", "no weight", "other shape"])
@pytest.mark.parametrize("place", ["norm1", "norm2"])
def test_norm_weight_must_fit(mode, monkeypatch, change, place):
    """norm_add with a replaced RMSNorm weight goes to the module's call (which refuses or converts)."""
    taken = []
    monkeypatch.setattr(layer_ops._lib, "load", lambda: taken.append("kernel") or _Lib())
    monkeypatch.setattr(layer_ops._lib, "stream_handle", lambda device: None)
    monkeypatch.setattr(nn.RMSNorm, "forward", lambda self, x: taken.append("module") or x)
    with mode:
        a = torch.empty(3, D, device="cuda:0")
        norm = nn.RMSNorm(D, device="cuda:0")
        layer_ops.norm_add(a, **{place: norm})
        assert taken == ["kernel"]
        if change == "no weight":
            norm = nn.RMSNorm(D, elementwise_affine=False)
        elif change == "other shape":
            norm = nn.RMSNorm((3, D), device="cuda:0")
        else:
            norm.weight = nn.Parameter(torch.empty(
                {"shorter": D // 2, "longer": 2 * D}.get(change, D),
                device="cuda:1" if change == "device" else "cuda:0",
                dtype=torch.float16 if change == "type" else torch.float32))
        layer_ops.norm_add(a, **{place: norm})
    assert taken == ["kernel", "module"]


@pytest.mark.parametrize("change", ["router", "sigma", "sigma device", "sigma type", "vproj rows"])
def test_mcmoe_coefficients_must_fit(mode, monkeypatch, change):
    """Logits, sigma or projections of other sizes than the module's go to the torch ops."""
    taken = []
    monkeypatch.setattr(layer_ops._lib, "load", lambda: taken.append("kernel") or _Lib())
    monkeypatch.setattr(layer_ops._lib, "stream_handle", lambda device: None)
    n, C, r = 5, 16, 8

    def make(rows, cols, **kw):
        return torch.empty(rows, cols, **{"device": "cuda:0", **kw})
    with mode:
        good = make(n, C), make(n, C * r), make(n, C * r)
        layer_ops.mcmoe_coef(*good, 4, C)
        assert taken == ["kernel"]
        bad = list(good)
        i, t = {"router": (0, make(n, C // 2)), "sigma": (1, make(n, C * r // 2)),
                "sigma device": (1, make(n, C * r, device="cuda:1")),
                "sigma type": (1, make(n, C * r, dtype=torch.float16)),
                "vproj rows": (2, make(n - 1, C * r))}[change]
        bad[i] = t
        try:
            layer_ops.mcmoe_coef(*bad, 4, C)
        except (RuntimeError, ValueError):   # the torch ops' refusal
            assert change != "sigma type"
        else:
            assert change == "sigma type"
    assert taken == ["kernel"]


def test_mcmoe_router_of_another_size_is_refused():
    """As ever: the coefficients have the module's components, whatever the router gives."""
    from verace_amd import ManifoldContinuousMoE
    m = ManifoldContinuousMoE(D, rank=8, num_components=16, top_k_components=4)
    m.router = nn.Linear(D, 8, bias=False)
    with torch.no_grad(), pytest.raises(RuntimeError):
        m(torch.randn(2, 3, D))


def test_plain_modules_only():
    """A module compiled in place runs its compiled call, as one with hooks or another forward does."""
    assert layer_ops.plain(nn.Linear(4, 4), nn.Linear)
    m = nn.Linear(4, 4)
    m.compile(backend="eager")
    assert not layer_ops.plain(m, nn.Linear)
    m = nn.Linear(4, 4)
    m.register_forward_pre_hook(lambda *a: None)
    assert not layer_ops.plain(m, nn.Linear)
    m = nn.Linear(4, 4)
    m.forward = lambda x: x
    assert not layer_ops.plain(m, nn.Linear)


def test_only_the_current_device(monkeypatch):
    """Launches go to the current device: tensors of another one keep the torch ops, which run there."""
    from verace_amd import hip_kernels
    current = [0]
    monkeypatch.setattr(torch._C, "_cuda_getDevice", lambda: current[0])
    with FakeTensorMode():
        a, b = torch.empty(2, device="cuda:0"), torch.empty(2, device="cuda:1")
    assert hip_kernels.on_current_device(a) and not hip_kernels.on_current_device(b)
    current[0] = 1
    assert hip_kernels.on_current_device(b) and not hip_kernels.on_current_device(a)
    assert not hip_kernels.on_current_device(torch.empty(2))


class _Lib:
    """Every entry point of the library, doing nothing."""

    def __getattr__(self, name):
        return lambda *args: 0
