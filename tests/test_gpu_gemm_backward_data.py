"""GPU parity of the GEMM-level data gradient on both sides of its kernel
choice (64 and 256 channels, 4e8 products), against fp64: rel 1e-5 of the sum
of |terms| plus 1e-6."""
import pytest
import torch

from approxtorch_amd.backend import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("exact", [False, True])
@pytest.mark.parametrize("N,K,L,Oc", [
    (2, 33, 17, 63), (2, 33, 17, 64), (1, 40, 21, 255), (1, 129, 7, 256), (3, 100, 37, 500),
    (4, 576, 2713, 64), (4, 576, 2712, 64), (16, 1152, 196, 128)])
def test_gemm_backward_data(N, K, L, Oc, exact):
    gen = torch.Generator(device="cuda").manual_seed(N + K + L + Oc)
    go = torch.randn(N, Oc, L, generator=gen, device="cuda")
    wq = torch.randint(0, 256, (Oc, K), generator=gen, device="cuda", dtype=torch.uint8)
    tab = torch.arange(256, device="cuda").float() - 128 if exact else \
        torch.randn(256, generator=gen, device="cuda")
    got = ops.gemm_backward_data(go, wq, tab)
    w = tab[wq.long()].double().t().contiguous()
    for n in range(N):
        want, bound = w @ go[n].double(), w.abs() @ go[n].double().abs()
        assert bool(((got[n].double() - want).abs() <= 1e-5 * bound + 1e-6).all())
