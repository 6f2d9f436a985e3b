"""The retraction's two tile sizes: a launch of few 128 x 128 tiles takes 64 x 64 ones.  A matrix
retracted alone and in a batch large enough for the wide tiles: the two differ in rounding alone
(below the diagonal of a wide diagonal tile the Gram sums its terms in another order)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _ns64(r, i, steps):
    h = torch.complex(r.double(), i.double())
    eye = 3.0 * torch.eye(h.shape[-1], dtype=h.dtype)
    for _ in range(steps):
        h = 0.5 * (h @ (eye - h.mH @ h))
    return h


# alone: 64 x 64 tiles; in a batch of this size both products (at 3 x 1536 and 7 x 1024), or the
# update alone, take 128 x 128 ones; the batches of 128 and 256 lie on the line (850 tiles of 64)
@pytest.mark.parametrize("batch,n", [(213, 128), (212, 128), (54, 256), (53, 256), (15, 512),
                                     (4, 1024), (7, 1024), (3, 1536)])
@pytest.mark.parametrize("steps", [1, 3])
def test_alone_and_in_a_batch(batch, n, steps):
    import verace_amd as va
    g = torch.Generator().manual_seed(n + steps)
    q = torch.linalg.qr(torch.complex(torch.randn(n, n, generator=g, dtype=torch.double),
                                      torch.randn(n, n, generator=g, dtype=torch.double)))[0]
    noise = 0.02 / n ** 0.5
    r = (q.real + noise * torch.randn(batch, n, n, generator=g)).float()
    i = (q.imag + noise * torch.randn(batch, n, n, generator=g)).float()
    rd, id_ = r.cuda(), i.cuda()
    br, bi = va.newton_schulz_unitary_retraction(rd, id_, steps=steps)
    for b in (0, batch // 2, batch - 1):
        sr, si = va.newton_schulz_unitary_retraction(rd[b:b + 1], id_[b:b + 1], steps=steps)
        ref = _ns64(r[b], i[b], steps)
        wide = torch.complex(br[b].cpu().double(), bi[b].cpu().double())
        narrow = torch.complex(sr[0].cpu().double(), si[0].cpu().double())
        e_wide, e_narrow = (float((x - ref).norm() / ref.norm()) for x in (wide, narrow))
        # f16 pairs drop 2^-22 of a product and fp32 sums add a few 2^-24, per step
        assert e_wide < 2e-6 and e_narrow < 2e-6, (e_wide, e_narrow)
        assert e_narrow < 1.2 * e_wide, (e_wide, e_narrow)
        assert float((wide - narrow).norm() / ref.norm()) < 1e-6
