"""The 128 x 128 product tiles with operands that run along the summed dimension
('T' 'N' and 'N' 'N'), as the inverse from a factor takes them (orders whose products
have at least 512 such tiles): whole tiles, and ragged unaligned ones.

Against the inverse in float64 on the GPU; every spectrum lies in [0.5, 4.6], so the
computed inverse is within 10 n eps of it (Frobenius norm)."""
import pytest
import torch

from libddla_amd import autograd as ag

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("n", [2944, 2951])
def test_potri_large_tiles(handle, n, dtype):
    print(f"case potri tiles n={n} {dtype}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(n)
    g = torch.randn(n, n, dtype=torch.float64, device="cuda", generator=gen)
    a = torch.mm(g, g.t().contiguous()) / n
    a.diagonal().add_(0.5)
    low = torch.linalg.cholesky(a)
    ref = torch.cholesky_inverse(low)
    inv = ag.potri(low.to(dtype), handle).double()
    assert (torch.linalg.norm(inv - ref) / torch.linalg.norm(ref)).item() <= 10 * n * torch.finfo(dtype).eps
