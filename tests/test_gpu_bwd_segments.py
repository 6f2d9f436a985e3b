"""GPU parity of the chunked backward (csrc/sssd_bwd_chunk.hip) where its splits can go wrong:
ragged chunks, one and several segments (a segment holds at least four chunks of 16 tokens), the
last segment short, and the output gradient in another type than the inputs (bf16 inputs with a
bf16 gradient take the exact-parts pass, with another type the general one).

Reference: fp64 autograd through the eager restatement.  Bars, relative Frobenius per tensor: fp32
1e-5 (as tests/test_gpu_bwd.py); 16-bit inputs 1e-2: the per-chunk gradient products round both
operands to bf16 (2^-9 relative each) and the result is stored once more in 16 bits, so a few
2^-9 = 2e-3 (measured 2e-3 .. 4.4e-3)."""
import pytest
import torch

from oracle import sssd_eager

pytestmark = pytest.mark.gpu


def _inputs(B, T, H, D, dtype, go_dtype):
    g = torch.Generator().manual_seed(7 * T + D)
    q, k, v = (torch.nn.functional.normalize(torch.randn(B, T, H, D, generator=g), dim=-1).to(dtype)
               for _ in range(3))
    d = (0.1 * torch.sigmoid(torch.randn(B, T, H, generator=g))).to(dtype)
    psi0 = torch.linalg.qr(torch.randn(B, H, D, D, generator=g))[0].contiguous()
    return q, k, v, d, psi0, torch.randn(B, T, H, D, generator=g).to(go_dtype), \
        torch.randn(B, H, D, D, generator=g)


CASES = [
    # one segment: whole, ragged and single-token last chunks
    (1, 32, 1, 64), (2, 33, 1, 128), (1, 47, 2, 64), (1, 65, 1, 128),
    # several: whole segments, a short last one, a ragged last chunk
    (1, 512, 1, 64), (1, 513, 1, 128), (1, 610, 2, 64), (2, 345, 1, 128),
]


@pytest.mark.parametrize("B,T,H,D", CASES)
@pytest.mark.parametrize("dtype,go_dtype", [(torch.float32, torch.float32),
                                            (torch.bfloat16, torch.bfloat16),
                                            (torch.bfloat16, torch.float32),
                                            (torch.float16, torch.bfloat16)])
def test_backward_segments_match_oracle(device, B, T, H, D, dtype, go_dtype):
    from verace_amd import launch_sssd_hip_scan, launch_sssd_hip_scan_bwd
    print(f"[case] bwd segments B={B} T={T} H={H} D={D} {dtype} dout {go_dtype}", flush=True)
    q, k, v, d, psi0, d_out, d_psi = _inputs(B, T, H, D, dtype, go_dtype)
    a = [x.double().clone().requires_grad_(True) for x in (q, k, v, d, psi0)]
    o, s = sssd_eager.sssd_scan_eager(*a, compute_dtype=torch.float64)
    ((o * d_out.double()).sum() + (s * d_psi.double()).sum()).backward()
    dev = [x.to(device) for x in (q, k, v, d)]
    _, psi_T = launch_sssd_hip_scan(*dev, psi0.to(device))
    grads = launch_sssd_hip_scan_bwd(*dev, psi_T, d_out.to(device), d_psi.to(device))
    for name, x, r in zip(("dq", "dk", "dv", "ddelta", "dpsi0"), grads, a):
        e = float((x.double().cpu() - r.grad).norm() / r.grad.norm())
        assert e <= (1e-5 if dtype == torch.float32 else 1e-2), (name, e)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_backward_segments_without_state_gradients(device, dtype):
    """No final-state gradient and no initial-state gradient asked for: as zeros given."""
    from verace_amd import launch_sssd_hip_scan, launch_sssd_hip_scan_bwd
    q, k, v, d, psi0, d_out, _ = (x.to(device) for x in _inputs(1, 400, 2, 128, dtype, dtype))
    _, psi_T = launch_sssd_hip_scan(q, k, v, d, psi0)
    none = launch_sssd_hip_scan_bwd(q, k, v, d, psi_T, d_out, None, False)
    zero = launch_sssd_hip_scan_bwd(q, k, v, d, psi_T, d_out, torch.zeros_like(psi_T), True)
    assert none[4] is None
    for x, y in zip(none[:4], zero[:4]):
        assert torch.equal(x, y)
