"""The matrix-core CHAM route reads and writes its hologram planes in 16-byte pieces where h and the
planes' addresses allow, else element by element (csrc/cham_mfma.hip load_plane): both move the same
values, so planes at an odd 4-byte offset give the same bits as aligned ones, with the floats
around the final planes untouched.  Sizes: a last column block of 8 (h = 136, 264, 600) and a whole one
(256), one chunk and several, fewer 16-feature blocks than the chunk's waves (136)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _planes(device, B, h, off, fill=None):
    buf = torch.full((B * h * h + 8,), 7.0, device=device)
    view = buf[off:off + B * h * h].view(B, h, h)
    if fill is not None:
        view.copy_(fill)
    return buf, view


def _scan(device, q, k, v, gam, h0, off):
    from verace_amd import _lib, hip_kernels as hk
    import ctypes
    B, T, h = q.shape
    lib = _lib.load()
    n = ctypes.c_size_t()
    _lib.check(lib.vmi_cham_scan_workspace_bytes(B, T, h, ctypes.byref(n)), "workspace")
    ws = torch.empty(max(n.value, 16), device=device, dtype=torch.uint8)
    out = torch.empty_like(q)
    ir, ii = _planes(device, B, h, off, h0[0])[1], _planes(device, B, h, off, h0[1])[1]
    (br, fr), (bi, fi) = _planes(device, B, h, off), _planes(device, B, h, off)
    _lib.check(lib.vmi_cham_scan_fwd(hk._ptr(q), hk._ptr(k), hk._ptr(v), hk._ptr(gam),
                                     _lib.dtype_code(q.dtype), _lib.dtype_code(gam.dtype), hk._ptr(ir),
                                     hk._ptr(ii), hk._ptr(out), hk._ptr(fr), hk._ptr(fi), B, T, h,
                                     hk._ptr(ws), n.value, _lib.stream_handle(q.device)), "scan")
    torch.cuda.synchronize()
    for b in (br, bi):
        assert (b[:off] == 7).all() and (b[off + B * h * h:] == 7).all()
    return out.clone(), fr.clone(), fi.clone()


@pytest.mark.parametrize("B,T,h", [(1, 1, 136), (2, 40, 256), (1, 17, 264), (2, 33, 600)])
def test_unaligned_hologram_planes_same_bits(device, B, T, h):
    print(f"[case] cham planes B{B} T{T} h{h}", flush=True)
    g = torch.Generator().manual_seed(h + T)
    nrm = torch.nn.functional.normalize
    q, k, v = (nrm(torch.randn(B, T, h, generator=g), dim=-1).to(torch.bfloat16).to(device) for _ in range(3))
    gam = (0.1 * torch.rand(B, T, generator=g)).to(device)
    # largest singular value near 0.3 * 2 * sqrt(2) < sqrt(3): the readout's retraction converges
    h0 = torch.randn(2, B, h, h, generator=g).mul(0.3 * h ** -0.5).to(device)
    want = _scan(device, q, k, v, gam, h0, 0)
    got = _scan(device, q, k, v, gam, h0, 1)
    for name, a, b in zip(("out", "H_real", "H_imag"), got, want):
        assert torch.equal(a, b), name
    assert all(torch.isfinite(x).all() for x in want) and (want[1] - h0[0]).abs().max() > 0
