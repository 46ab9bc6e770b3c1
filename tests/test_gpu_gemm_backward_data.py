"""GPU parity of the GEMM-level data gradient on both sides of its kernel
choice (tables known to hold bf16 values or not, 64 and 256 channels, 4e8
products), against fp64: rel 1e-5 of the sum of |terms| plus 1e-6."""
import pytest
import torch

from approxtorch_amd.backend import ops
from approxtorch_amd.nn import bgemm_int8

pytestmark = pytest.mark.gpu


def operands(N, K, L, Oc, exact):
    gen = torch.Generator(device="cuda").manual_seed(N + K + L + Oc)
    go = torch.randn(N, Oc, L, generator=gen, device="cuda")
    wq = torch.randint(0, 256, (Oc, K), generator=gen, device="cuda", dtype=torch.uint8)
    tab = torch.arange(256, device="cuda").float() - 128 if exact else \
        torch.randn(256, generator=gen, device="cuda")
    return go, wq, tab


@pytest.mark.parametrize("exact", [False, True])
@pytest.mark.parametrize("N,K,L,Oc", [
    (2, 33, 17, 63), (2, 33, 17, 64), (1, 40, 21, 255), (1, 129, 7, 256), (3, 100, 37, 500),
    (4, 576, 2713, 64), (4, 576, 2712, 64), (16, 1152, 196, 128)])
def test_gemm_backward_data(N, K, L, Oc, exact):
    go, wq, tab = operands(N, K, L, Oc, exact)
    got = ops.gemm_backward_data(go, wq, tab, exact)
    w = tab[wq.long()].double().t().contiguous()
    for n in range(N):
        want, bound = w @ go[n].double(), w.abs() @ go[n].double().abs()
        assert bool(((got[n].double() - want).abs() <= 1e-5 * bound + 1e-6).all())


@pytest.mark.parametrize("exact", [False, True])
@pytest.mark.parametrize("Oc", [128, 512, 4096])
def test_one_signed_operands_leave_no_bias(Oc, exact):
    """Rounding errors of fp32 products and sums average out: the mean signed
    error stays below 2e-8 of the sum (fp32 kernels measure 1e-9 to 9e-9 here);
    dropped part products of a general table would leave -5e-8."""
    go, wq, tab = operands(2, 300, 700, Oc, exact)
    go, tab = go.abs(), tab.abs()
    got = ops.gemm_backward_data(go, wq, tab, exact)
    w = tab[wq.long()].double().t().contiguous()
    for n in range(2):
        want = w @ go[n].double()
        assert abs(float(((got[n].double() - want) / want).mean())) < 2e-8


@pytest.mark.parametrize("exact", [False, True])
@pytest.mark.parametrize("Oc", [40, 256])
def test_infinite_output_gradients(Oc, exact):
    """Through the autograd ops: an infinite go gives the infinities and NaNs
    that its products with the table have, bf16 table values among others."""
    gen = torch.Generator(device="cuda").manual_seed(Oc)
    x = torch.randint(-128, 128, (2, 30, 21), generator=gen, device="cuda").float()
    w = torch.randint(-128, 128, (Oc, 30), generator=gen, device="cuda").float()
    lut = torch.zeros(65536, device="cuda")
    go = torch.randn(2, Oc, 21, generator=gen, device="cuda")
    go[0, 3, 5], go[0, 7, 5], go[1, Oc - 1, 0] = float("inf"), float("-inf"), float("inf")
    x.requires_grad_(), w.requires_grad_()
    if exact:
        tab = torch.arange(256, device="cuda").float() - 128
        y = bgemm_int8.bgemm_int8_ste(x, w, lut)
    else:
        tab = torch.randn(256, generator=gen, device="cuda")
        tab[::2] = torch.arange(1, 129, device="cuda").float()       # bf16 values
        y = bgemm_int8.bgemm_int8_lre(x, w, lut, tab, tab)
    gx, = torch.autograd.grad(y, [x], go)
    wt = tab[(w.detach() + 128).long()].double().t().contiguous()
    want = torch.stack([(wt.unsqueeze(2) * go[n].double().unsqueeze(0)).sum(1) for n in range(2)])
    assert torch.equal(torch.isnan(gx), torch.isnan(want))
    inf = torch.isinf(want)
    assert torch.equal(gx[inf], want[inf].float()) and bool(inf.any())
    assert bool(torch.isfinite(gx[torch.isfinite(want)]).all())
