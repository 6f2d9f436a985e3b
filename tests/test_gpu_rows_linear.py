"""The few-rows linear product (csrc/rows_linear.hip) against fp64.  Both operands are exact in the
products; the error is fp32 accumulation in chains of at most K / 16 products and an 8-term sum, under
(K / 16 + 16) 2^-24 of sum |x w|, and one rounding of the result.  Shapes: one and sixteen rows, one output
row, a remainder of the 16 output rows, K of one 16-byte piece, below and past the 64-column pieces and the
columns in flight; a row stride wider than K; what has to be refused."""
import ctypes

import pytest
import torch
import torch.nn as nn
import torch.nn.functional as F

pytestmark = pytest.mark.gpu
ULP = {torch.float32: 2.0 ** -24, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


def _call(x, xs, w, y, M, N, K):
    from verace_amd import _lib, hip_kernels as hk
    return _lib.load().vmi_rows_linear(hk._ptr(x), xs, hk._ptr(w), _lib.dtype_code(w.dtype), hk._ptr(y), M, N, K,
                                       _lib.stream_handle(w.device))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,K,pad", [(1, 1, 8, 0), (2, 17, 72, 8), (16, 16, 64, 0), (3, 100, 520, 0),
                                       (16, 257, 1024, 16), (5, 33, 2056, 0)])
def test_rows_linear(device, M, N, K, pad, dtype):
    print(f"[case] rows linear M{M} N{N} K{K} {dtype}", flush=True)
    g = torch.Generator().manual_seed(K + M)
    x = torch.randn(M, K + pad, generator=g).to(dtype).to(device)
    w = torch.randn(N, K, generator=g).to(dtype).to(device)
    y = torch.full((M * N + 8,), 7.0, device=device, dtype=dtype)
    assert _call(x, K + pad, w, y, M, N, K) == 0
    torch.cuda.synchronize()
    xd, wd = x[:, :K].double().cpu(), w.double().cpu()
    ref, mag = xd @ wd.T, xd.abs() @ wd.abs().T
    got = y[:M * N].view(M, N).double().cpu()
    assert bool(((got - ref).abs() <= (K / 16 + 16) * 2.0 ** -24 * mag + ULP[dtype] * ref.abs()).all())
    assert bool((y[M * N:] == 7).all())


def test_rows_linear_special_values(device):
    """A NaN or infinite element reaches its own row's results only, as in F.linear."""
    x = torch.ones(3, 1, 256, device=device)
    x[1, 0, 5] = float("nan")
    x[2, 0, 250] = float("inf")
    w = torch.ones(20, 256, device=device)
    from verace_amd.layer_ops import rows_linear
    with torch.no_grad():
        y, ref = rows_linear(x, w), F.linear(x, w)
    assert y.shape == ref.shape and torch.equal(torch.nan_to_num(y, -1.0), torch.nan_to_num(ref, -1.0))


def test_rows_linear_refusals_and_general_path(device):
    x, w = torch.ones(17, 64, device=device), torch.ones(8, 64, device=device)
    y = torch.zeros(17 * 8, device=device)
    assert _call(x, 64, w, y, 17, 8, 64) != 0 and _call(x, 64, w, y, 2, 8, 63) != 0
    assert _call(x, 62, w, y, 2, 8, 64) != 0 and _call(x.view(-1)[1:], 64, w, y, 2, 8, 64) != 0
    from verace_amd.layer_ops import rows_call, rows_linear
    lin = nn.Linear(64, 8, bias=False).to(device)
    seen = []
    for xs in (x.view(17, 1, 64), x[:2].view(2, 1, 64), x[:0].view(0, 1, 64), x.t().contiguous().t()[:2].unsqueeze(1)):
        with torch.no_grad():
            torch.testing.assert_close(rows_linear(xs, lin.weight), F.linear(xs, lin.weight))
    assert rows_linear(x[:2], lin.weight).requires_grad  # autograd keeps the library product
    hook = lin.register_forward_hook(lambda m, i, o: seen.append(1))
    with torch.no_grad():
        rows_call(lin, x[:2])
    hook.remove()
    assert seen == [1]
    with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16):
        assert rows_linear(x[:2], lin.weight).dtype == torch.bfloat16
