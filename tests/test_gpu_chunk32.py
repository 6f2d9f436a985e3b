"""GPU parity of the chunked fp32 scan (csrc/sssd_chunk32.hip): fp32 inputs, head_dim other than
128 and short 16-bit calls, against the fp64 closed form and against the token-sequential scan
that the same C entry point runs when it is given no workspace.

Bars: fp32 I/O 1e-5 relative Frobenius error per (b, h) slice (the repository's fp32 bar; measured
5e-8 .. 1.2e-6 here, the token-sequential scan 1e-7 .. 3.4e-6); 16-bit I/O: the output within one
rounding of the type (2^-8 / 2^-11), the fp32 state at 1e-5."""
import ctypes
import math

import numpy as np
import pytest
import torch
import torch.nn.functional as F

from oracle import sssd_closed

pytestmark = pytest.mark.gpu

OUT_BAR = {torch.float32: 1e-5, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


def _inputs(B, T, H, D, dtype, seed, delta_scale=0.1):
    g = torch.Generator().manual_seed(seed)
    q, k, v = (F.normalize(torch.randn(B, T, H, D, generator=g), dim=-1).to(dtype) for _ in range(3))
    delta = (delta_scale * torch.sigmoid(torch.randn(B, T, H, generator=g))).to(dtype)
    psi0 = torch.linalg.qr(torch.randn(B, H, D, D, generator=g))[0].contiguous()
    return q, k, v, delta, psi0


def _c_scan(q, k, v, delta, psi0, device, workspace=True, offset=0):
    """vmi_sssd_scan_fwd itself; offset shifts every input and the output by that many elements
    inside a larger buffer, workspace False passes none."""
    from verace_amd import _lib
    lib = _lib.load()
    B, T, H, D = q.shape

    def place(t):
        buf = torch.empty(t.numel() + offset, dtype=t.dtype, device=device)
        buf[offset:].copy_(t.reshape(-1).to(device))
        return buf[offset:]
    ins = [place(t) for t in (q, k, v, delta)]
    out = place(torch.zeros_like(q))
    init = None if psi0 is None else psi0.to(device)
    psi = torch.empty(B, H, D, D, device=device)
    ws, need = None, ctypes.c_size_t(0)
    if workspace:
        _lib.check(lib.vmi_sssd_scan_workspace_bytes(B, T, H, D, _lib.dtype_code(q.dtype),
                                                     ctypes.byref(need)), "workspace_bytes")
        ws = torch.empty(max(need.value, 16), dtype=torch.uint8, device=device)
    ptr = lambda t: None if t is None else ctypes.c_void_p(t.data_ptr())  # noqa: E731
    _lib.check(lib.vmi_sssd_scan_fwd(*map(ptr, ins), _lib.dtype_code(q.dtype),
                                     _lib.dtype_code(delta.dtype), ptr(init), ptr(out), ptr(psi),
                                     B, T, H, D, ptr(ws), need.value,
                                     _lib.stream_handle(torch.device(device))), "scan")
    torch.cuda.synchronize()
    return out.view(q.shape).float().cpu(), psi.cpu()


def _oracle(q, k, v, delta, psi0):
    a = [t.float().numpy() for t in (q, k, v, delta)]
    return sssd_closed.sssd_scan_closed_c(*a, None if psi0 is None else psi0.double().numpy())


def _slice_err(x, ref, dims):
    x = np.asarray(x, dtype=np.float64)
    num = np.sqrt(((x - ref) ** 2).sum(axis=dims))
    return float((num / np.maximum(np.sqrt((ref ** 2).sum(axis=dims)), 1e-30)).max())


# edges of a chunk (16 tokens) and of the shortest call, of the padded head sizes (32, 64, 128), of
# rows that are not whole 16-byte pieces, and sequences long enough for several segments
SHAPES = [(1, 5, 1, 1), (1, 8, 2, 128), (2, 15, 2, 15), (1, 16, 3, 16), (2, 17, 1, 17), (1, 31, 2, 32),
          (1, 33, 2, 33), (2, 48, 2, 63), (1, 129, 2, 64), (2, 20, 3, 65), (1, 50, 2, 100),
          (1, 9, 1, 1), (1, 7, 2, 16), (1, 5, 2, 33), (1, 5, 1, 65), (1, 40, 2, 127), (2, 100, 2, 128), (1, 1030, 2, 128), (2, 999, 1, 40), (3, 700, 3, 30)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,T,H,D", SHAPES)
def test_chunk32_matches_oracle(device, B, T, H, D, dtype):
    if dtype != torch.float32 and D == 128 and T >= 32:
        T = 31   # longer ones are the 16-bit chunk scan's
    print(f"[case] chunk32 B={B} T={T} H={H} D={D} {dtype}", flush=True)
    q, k, v, delta, psi0 = _inputs(B, T, H, D, dtype, 1000 * T + D)
    for init in (None, psi0):
        o64, p64 = _oracle(q, k, v, delta, init)
        o, psi = _c_scan(q, k, v, delta, init, device)
        assert _slice_err(o, o64, (1, 3)) <= OUT_BAR[dtype]
        assert _slice_err(psi, p64, (2, 3)) <= 1e-5
        os, ps = _c_scan(q, k, v, delta, init, device, workspace=False)   # token by token
        assert _slice_err(os, o64, (1, 3)) <= OUT_BAR[dtype]
        assert _slice_err(ps, p64, (2, 3)) <= 1e-5


@pytest.mark.parametrize("dtype,D", [(torch.float32, 128), (torch.float32, 20), (torch.bfloat16, 64)])
@pytest.mark.parametrize("offset", [1, 2, 4])
def test_chunk32_unaligned_rows(device, dtype, D, offset):
    """Inputs and output at any element offset of a buffer give the aligned call's bits."""
    print(f"[case] chunk32 offset={offset} D={D} {dtype}", flush=True)
    q, k, v, delta, psi0 = _inputs(2, 37, 2, D, dtype, 5)
    a = _c_scan(q, k, v, delta, psi0, device)
    b = _c_scan(q, k, v, delta, psi0, device, offset=offset)
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])


def _pairs(T, D, length, angle, skew, distinct, seed):
    """Tokens with |k| = |v| = length, the given angle between k and v and (delta / 2) |k| |v| = skew,
    taken in turn from ``distinct`` k, v pairs (few repeated pairs are what the chunk's substitution
    cancels worst on)."""
    g = torch.Generator().manual_seed(seed)
    k, w = (F.normalize(torch.randn(2, distinct, D, generator=g), dim=-1) for _ in range(2))
    w = F.normalize(w - (w * k).sum(-1, keepdim=True) * k, dim=-1)
    v = math.cos(angle) * k + math.sin(angle) * w
    turn = torch.arange(T) % distinct
    k, v = (length * t[:, turn].transpose(0, 1)[None] for t in (k, v))
    q = F.normalize(torch.randn(1, T, 2, D, generator=g), dim=-1)
    delta = torch.full((1, T, 2), 2.0 * skew / length ** 2)
    return q, k.contiguous(), v.contiguous(), delta


def test_chunk32_related_tokens(device):
    """Tokens whose k and v are nearly the same vectors all along (the Gram matrix of a chunk is
    close to rank 2), at the largest delta that the chunk form takes of unit k, v."""
    B, T, H, D = 1, 600, 2, 64
    q, k, v, delta, psi0 = _inputs(B, T, H, D, torch.float32, 8, delta_scale=0.109)
    k = F.normalize(k[:, :1] + 1e-2 * k, dim=-1)
    v = F.normalize(v[:, :1] + 1e-2 * v, dim=-1)
    o64, p64 = _oracle(q, k, v, delta, psi0)
    o, psi = _c_scan(q, k, v, delta, psi0, device)
    print(f"[case] chunk32 related tokens: o {_slice_err(o, o64, (1, 3)):.1e} psi {_slice_err(psi, p64, (2, 3)):.1e}", flush=True)
    assert _slice_err(o, o64, (1, 3)) <= 1e-5 and _slice_err(psi, p64, (2, 3)) <= 1e-5
    assert not torch.equal(psi, _c_scan(q, k, v, delta, psi0, device, workspace=False)[1])


@pytest.mark.parametrize("length", [1.0, 3.0, 10.0, 30.0])
@pytest.mark.parametrize("angle", [1.5, 0.1, 0.01, 0.003])
@pytest.mark.parametrize("skew", [0.054, 0.06, 0.5, 5.0])
def test_chunk32_never_rounds_worse_than_the_sequential_scan(device, length, angle, skew):
    """Nearly parallel k and v rotate little however long they are, but T~'s terms grow with
    (delta / 2) |k| |v|: past its bound (0.0547) a call is the token-sequential scan's bits, below it
    no more than twice as far from fp64 (1.5 measured over tokens of this kind), both sides' few last
    bits (2e-7) apart."""
    D, T = 64, 256
    if skew * math.sin(angle) > 0.25:
        skew = 0.25 / math.sin(angle)   # the rotation m stays where the 16-bit scan's rule has it
    for distinct in (2, 3):
        q, k, v, delta = _pairs(T, D, length, angle, skew, distinct, 7)
        o, psi = _c_scan(q, k, v, delta, None, device)
        os, ps = _c_scan(q, k, v, delta, None, device, workspace=False)
        if skew > 0.055:
            assert torch.equal(o, os) and torch.equal(psi, ps)
            continue
        assert not torch.equal(psi, ps)
        o64, p64 = _oracle(q, k, v, delta, None)
        for x, xs, ref, dims in ((o, os, o64, (1, 3)), (psi, ps, p64, (2, 3))):
            e, es = _slice_err(x, ref, dims), _slice_err(xs, ref, dims)
            print(f"[case] chunk32 length {length} angle {angle} skew {skew:.3f}: {e:.1e} ({es:.1e})", flush=True)
            assert e <= 2.0 * es + 2e-7


def test_scan_without_room_for_its_workspace(device, monkeypatch):
    """The fp32 scan, whose workspace is optional, runs without it where its allocation fails; the
    16-bit chunk scan, which needs its own, raises that failure."""
    from verace_amd import launch_sssd_hip_scan
    empty = torch.empty

    def no_bytes(*args, **kw):
        if kw.get("dtype") is torch.uint8:
            raise torch.OutOfMemoryError("no room")
        return empty(*args, **kw)
    q, k, v, delta, psi0 = _inputs(1, 600, 2, 64, torch.float32, 11)
    ref = _c_scan(q, k, v, delta, psi0, device, workspace=False)
    monkeypatch.setattr(torch, "empty", no_bytes)
    o, psi = launch_sssd_hip_scan(*(t.to(device) for t in (q, k, v, delta, psi0)))
    assert torch.equal(o.cpu(), ref[0]) and torch.equal(psi.cpu(), ref[1])
    q, k, v, delta, _ = _inputs(1, 600, 2, 128, torch.bfloat16, 12)
    with pytest.raises(torch.OutOfMemoryError):
        launch_sssd_hip_scan(*(t.to(device) for t in (q, k, v, delta)))


def test_chunk32_wide_and_nonfinite_sequences_take_the_sequential_scan(device):
    """A sequence with a token above the chunk form's limit, or one whose Cayley factor
    is not finite, gives the token-sequential scan's bits; the others the chunk result."""
    B, T, H, D = 1, 700, 4, 64
    q, k, v, delta, psi0 = _inputs(B, T, H, D, torch.float32, 9)
    delta[0, 500, 1] = 3.0           # (delta / 2) |k| |v| = 1.5
    k[0, 3, 2, 5] = float("nan")
    v[0, T - 1, 3, 0] = float("inf")
    o, psi = _c_scan(q, k, v, delta, psi0, device)
    os, ps = _c_scan(q, k, v, delta, psi0, device, workspace=False)
    for h in (1, 2, 3):
        assert torch.equal(o[:, :, h], os[:, :, h]) and torch.equal(psi[:, h], ps[:, h]), h
    assert not torch.equal(psi[:, 0], ps[:, 0])
    assert torch.isfinite(o).all() and torch.isfinite(psi).all()
