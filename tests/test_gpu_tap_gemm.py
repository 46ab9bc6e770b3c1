"""GPU parity of the backward-data tap GEMM (go split once into bf16 planes,
image gradient without columns): residue classes of strides 1 and 2, odd and
even sizes, paddings and dilations of both parities, rectangular kernels,
channel counts around a tile and a 32-channel block, bf16-exact and general
tables, with and without the go scale and the STE, contraction splits, and
batches of two passes (planes past 2 GiB, a nearly empty last round).  The
workspace query tells that a shape takes this kernel.

Bar: the fp64 gradient within rel 1e-5 of the sum of |terms| plus 1e-6, and a
2-norm error of at most 4e-7 of the result (what one fp32 sum per tap shows).
"""
import pytest
import torch
import torch.nn.functional as F

from approxtorch_amd.backend import _lib as L
from approxtorch_amd.backend import ops

pytestmark = pytest.mark.gpu


def tap_splits(g, Oc):
    """Contraction splits of the tap GEMM (1: none), or None when
    atx_conv_bwd_data takes another way: in one pass its workspace holds the
    weight planes, the go planes and whole partial images, and not columns."""
    K, P = g.C * g.KH * g.KW, g.N * g.OH * g.OW
    rest = L.query("atx_conv_bwd_data_workspace_bytes", g, Oc) - \
        6 * L.round_up(K, 128) * L.round_up(Oc, 32)
    images, odd = divmod(rest - L.round_up(P * 6 * L.round_up(Oc, 32), 256),
                         4 * g.N * g.C * g.H * g.W)
    columns = rest % (4 * K * P) == 0
    return max(images, 1) if not (odd or columns) and images in (0, *range(2, 65)) else None


def check(N, C, H, W, Oc, k, s, p, d, table, fused, seed=0):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    g = ops.conv_geom((N, C, H, W), k, s, p, d)
    go = torch.randn(N, Oc, g.OH, g.OW, generator=gen, device="cuda")
    wq = torch.randint(0, 256, (Oc, C * g.KH * g.KW), generator=gen, device="cuda",
                       dtype=torch.uint8)
    tx = torch.arange(256, device="cuda").float() - 128 if table == "exact" else \
        torch.randn(256, generator=gen, device="cuda")
    sx = torch.rand(1, generator=gen, device="cuda") + 0.1
    sw = torch.rand(Oc, generator=gen, device="cuda") + 0.5
    mask = torch.rand(N, C, H, W, generator=gen, device="cuda") < 0.8
    kw = dict(go_sx=sx, go_sw=sw, mask=mask, scale=sx) if fused else {}
    gx = ops.conv_backward_data(go, wq, tx, g, **kw)
    wt = tx[wq.long()].double().t().contiguous()
    gd = go.double() * ((sx * sw).double().view(1, -1, 1, 1) if fused else 1.0)
    num, den, worst = 0.0, 0.0, 0.0
    for n in range(N):
        fold = [F.fold((w @ v.reshape(Oc, -1)).unsqueeze(0), (H, W), (g.KH, g.KW), d, p, s)[0]
                for w, v in ((wt, gd[n]), (wt.abs(), gd[n].abs()))]
        if fused:
            fold = [torch.where(mask[n], f, 0.0) / sx.double() for f in fold]
        diff = gx[n].double() - fold[0]
        num, den = num + float((diff ** 2).sum()), den + float((fold[0] ** 2).sum())
        worst = max(worst, float((diff.abs() - 1e-5 * fold[1]).max()))
    assert worst <= 1e-6 and (num / den) ** 0.5 <= 4e-7


# (..., contraction splits): strides 1 and 2 with odd sizes, paddings 0 to 3,
# dilations of both parities, kernels of one tap or none in some class, and
# different strides per axis; every shape is large and full enough for the rule
@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("table", ["exact", "general"])
@pytest.mark.parametrize("N,C,H,W,Oc,k,s,p,d,splits", [
    (8, 65, 57, 56, 33, 3, 1, 1, 1, 1), (6, 65, 57, 56, 33, 3, 1, 1, 1, 3),
    (24, 64, 40, 40, 32, 3, 1, 0, 1, 1), (4, 64, 40, 40, 32, 3, 1, 0, 1, 2),
    (4, 66, 48, 45, 40, (3, 5), 1, 2, 1, 3), (4, 96, 64, 60, 96, 3, 1, 2, 2, 2),
    (8, 96, 64, 60, 96, 3, 1, 2, 2, 1), (12, 256, 4, 4, 256, 3, 1, 1, 1, 18),
    (16, 64, 56, 56, 8, 3, 1, 1, 1, 1),
    (6, 128, 33, 31, 64, 3, 2, 1, 1, 2), (12, 128, 33, 31, 64, 3, 2, 1, 1, 1),
    (48, 129, 28, 27, 31, 3, 2, 0, 1, 1), (192, 48, 36, 37, 65, 3, 2, 2, 2, 1),
    (64, 100, 32, 35, 96, 3, 2, 3, 2, 1), (12, 128, 33, 35, 64, 3, 2, 1, 3, 1),
    (8, 512, 7, 9, 512, 3, 2, 1, 1, 11), (12, 64, 50, 51, 64, 2, 2, 0, 1, 1),
    (16, 128, 40, 38, 64, (2, 3), 2, 0, 1, 1), (64, 64, 30, 66, 64, (1, 4), 2, 1, 1, 1),
    (12, 64, 41, 38, 64, 3, (1, 2), 1, 1, 3), (12, 64, 41, 38, 64, 3, (2, 1), (0, 2), 1, 3)])
def test_tap_gemm(N, C, H, W, Oc, k, s, p, d, splits, table, fused):
    assert tap_splits(ops.conv_geom((N, C, H, W), k, s, p, d), Oc) == splits
    check(N, C, H, W, Oc, k, s, p, d, table, fused)


@pytest.mark.parametrize("N,C,H,W,Oc", [(83, 100, 30, 30, 100), (44, 128, 39, 39, 72)])
def test_tap_gemm_last_round_split(N, C, H, W, Oc):
    """A nearly empty last round of blocks: its images are a pass of their own,
    and the workspace holds less than the whole batch's go planes."""
    g = ops.conv_geom((N, C, H, W), 3, 1, 1, 1)
    assert L.query("atx_conv_bwd_data_workspace_bytes", g, Oc) < \
        6 * L.round_up(9 * C, 128) * L.round_up(Oc, 32) + N * H * W * 6 * L.round_up(Oc, 32)
    check(N, C, H, W, Oc, 3, 1, 1, 1, "general", True)


def test_tap_gemm_two_passes():
    """11 images of 1024 x 1024: 2.2 GB of go planes, more than a pass holds;
    the workspace stays under the pass's bound."""
    g = ops.conv_geom((11, 24, 1024, 1024), 3, 1, 1, 1)
    assert L.query("atx_conv_bwd_data_workspace_bytes", g, 4) < 2 ** 31 + 2 ** 20
    check(11, 24, 1024, 1024, 4, 3, 1, 1, 1, "general", True)


@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("table", ["exact", "general"])
@pytest.mark.parametrize("N,C,H,W,Oc,p", [
    (3, 33, 9, 11, 40, 1), (2, 130, 12, 8, 96, (0, 2)), (5, 64, 1, 1, 33, 3), (2, 24, 7, 7, 520, 1),
    (16, 64, 56, 56, 64, 1)])
def test_padded_1x1(N, C, H, W, Oc, p, table, fused):
    """The image gradient of a padded 1x1 conv from go's positions inside the
    image, without columns: ragged sizes, paddings of either axis, a split
    contraction."""
    g = ops.conv_geom((N, C, H, W), 1, 1, p, 1)
    rest = L.query("atx_conv_bwd_data_workspace_bytes", g, Oc) - \
        6 * L.round_up(C, 128) * L.round_up(Oc, 32)
    assert rest % (4 * N * C * H * W) == 0
    check(N, C, H, W, Oc, 1, 1, p, 1, table, fused)


@pytest.mark.parametrize("table", ["exact", "general"])
@pytest.mark.parametrize("N,C,H,W,Oc,k,s,p,d", [
    (8, 64, 28, 28, 64, 3, 1, 1, 1), (32, 70, 33, 31, 65, 3, 1, 1, 1),
    (8, 128, 33, 31, 64, 3, 2, 1, 1), (64, 130, 34, 30, 64, 3, 2, 2, 2),
    (16, 128, 40, 38, 64, (2, 3), 2, 0, 1), (83, 100, 30, 30, 100, 3, 1, 1, 1)])
def test_non_finite_table_entries_stay_with_their_taps(N, C, H, W, Oc, k, s, p, d, table):
    """A tap adds nothing to the pixels whose output lies outside go, also when
    its factor is infinite or NaN: everything else keeps its finite value."""
    gen = torch.Generator(device="cuda").manual_seed(C)
    g = ops.conv_geom((N, C, H, W), k, s, p, d)
    go = torch.randn(N, Oc, g.OH, g.OW, generator=gen, device="cuda")
    wq = torch.randint(2, 256, (Oc, C, g.KH, g.KW), generator=gen, device="cuda",
                       dtype=torch.uint8)
    wq[1, ::2, 0, 0], wq[Oc - 1, 1::3, g.KH - 1, g.KW - 1] = 0, 1
    wq = wq.view(Oc, -1)
    tx = torch.arange(256, device="cuda").float() if table == "exact" else \
        torch.randn(256, generator=gen, device="cuda")
    tx[0], tx[1] = float("inf"), float("nan")
    assert N == 83 or tap_splits(g, Oc)
    gx = ops.conv_backward_data(go, wq, tx, g)
    wt = tx[wq.long()].double().t().contiguous()
    for n in (*range(0, N, 7), N - 1):
        v = go[n].double().reshape(Oc, -1)
        want, terms = (F.fold((a @ b).unsqueeze(0), (H, W), (g.KH, g.KW), d, p, s)[0]
                       for a, b in ((wt, v), (wt.abs(), v.abs())))
        ok = torch.isfinite(want)
        assert torch.equal(torch.isfinite(gx[n]), ok)
        assert bool(((gx[n].double() - want).abs()[ok] <= 1e-5 * terms[ok] + 1e-6).all())
        assert bool(ok.any()) and not bool(ok.all())
