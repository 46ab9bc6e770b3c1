"""GPU parity of the 3x3 depthwise backward strip kernels (square stride and
dilation 1 or 2) over ragged and tiny images, paddings around the kernel's
reach, whole and partial strips and row runs, and every image type.

Bar: the image gradient bit for bit the fp32 sum over ascending taps of
go' * tx[w] (go' = fp32(go * fp32(sx * sw))); the weight gradient within rel
1e-5 of the sum of |terms| (the bound any fp32 order of at most 2^14 terms
meets) of the fp64 sum.
"""
import numpy as np
import pytest
import torch

from approxtorch_amd.backend import _lib as L
from approxtorch_amd.backend import ops

pytestmark = pytest.mark.gpu
f32 = np.float32


def t(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("dtype", ["int8", "uint8", "float32"])
@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("N,C,H,W,s,p,d", [
    (1, 1, 3, 3, 1, 0, 1), (2, 3, 5, 4, 1, 1, 1), (3, 5, 9, 12, 1, 1, 1), (2, 2, 30, 16, 1, 2, 2),
    (2, 3, 7, 11, 1, 3, 2), (2, 4, 17, 13, 1, 0, 2), (2, 3, 8, 8, 2, 1, 1), (1, 2, 31, 18, 2, 0, 1),
    (2, 3, 9, 7, 2, 3, 1), (3, 2, 12, 15, 2, 2, 2), (1, 3, 7, 9, 2, 1, 2), (1, 2, 1, 1, 1, 1, 1),
    (5, 70, 14, 14, 1, 1, 1), (2, 2, 6, 5, 2, 0, 2)])
def test_strip_gradients(N, C, H, W, s, p, d, fused, dtype):
    rng = np.random.default_rng(H * 100 + W * 10 + s + d)
    g = ops.conv_geom((N, C, H, W), 3, s, p, d)
    OH, OW = g.OH, g.OW
    go = rng.normal(size=(N, C, OH, OW)).astype(f32)
    lo, hi = (0, 256) if dtype == "uint8" else (-128, 128)
    img = rng.integers(lo, hi, (N, C, H, W)).astype(dtype)
    wq = rng.integers(0, 256, (C, 9)).astype(np.uint8)
    tx, tw = (rng.normal(size=256).astype(f32) for _ in range(2))
    pad = int(rng.integers(0, 256))
    sx, sw = f32(0.37), rng.uniform(0.5, 2, C).astype(f32)
    mask, mask_w = rng.random((N, C, H, W)) < 0.8, rng.random((C, 9)) < 0.8
    kw = dict(go_sx=t(np.array([sx])), go_sw=t(sw)) if fused else {}
    gx = ops.dwconv_backward_data(t(go), t(wq), t(tx), g, **kw,
                                  **(dict(mask=t(mask), scale=t(np.array([sx]))) if fused else {}))
    gw = ops.dwconv_backward_weight(t(go), t(img), t(tw), g, pad, **kw,
                                    **(dict(mask_w=t(mask_w), scale_w=t(sw)) if fused else {}))
    gs = go * (sx * sw).astype(f32)[None, :, None, None] if fused else go
    want = np.zeros((N, C, H, W), f32)
    idx = np.full((N, C, H + 2 * p, W + 2 * p), pad, np.int64)
    idx[:, :, p:p + H, p:p + W] = img.astype(np.int64) + (0 if dtype == "uint8" else 128)
    sums, absum = np.zeros((C, 9)), np.zeros((C, 9))
    for i in range(3):
        for j in range(3):
            w = tx[wq[:, i * 3 + j]]
            for oh in range(OH):
                h = oh * s + i * d - p
                cols = np.arange(OW) * s + j * d - p
                ok = (cols >= 0) & (cols < W)
                if 0 <= h < H:
                    want[:, :, h, cols[ok]] += gs[:, :, oh, ok] * w[None, :, None]
                terms = gs[:, :, oh].astype(np.float64) * tw[idx[:, :, oh * s + i * d, cols + p]]
                sums[:, i * 3 + j] += terms.sum((0, 2))
                absum[:, i * 3 + j] += np.abs(terms).sum((0, 2))
    if fused:
        want = (np.where(mask, want, f32(0)) / np.maximum(sx, f32(1e-12))).astype(f32)
        sums, absum = np.where(mask_w, sums, 0) / sw[:, None], absum / sw[:, None]
    assert np.array_equal(gx.cpu().numpy(), want)
    assert np.all(np.abs(gw.cpu().numpy() - sums) <= 1e-5 * absum + 1e-6)


def test_strip_gradients_keep_non_finite_table_entries_to_their_taps():
    """An infinite weight factor reaches only the pixels of its tap: an
    out-of-image output contributes nothing, not 0 * inf."""
    g = ops.conv_geom((1, 1, 6, 6), 3, 1, 1, 1)
    tx = torch.zeros(256, device="cuda")
    tx[7] = float("inf")
    wq = torch.zeros((1, 9), dtype=torch.uint8, device="cuda")
    wq[0, 0] = 7                                      # tap (0, 0) reads outputs one down, right
    gx = ops.dwconv_backward_data(torch.ones(1, 1, 6, 6, device="cuda"), wq, tx, g)[0, 0]
    assert torch.isinf(gx[:5, :5]).all()
    assert (gx[5] == 0).all() and (gx[:, 5] == 0).all()


@pytest.mark.parametrize("H,W", [(0, 4), (4, 0), (0, 0)])
def test_weight_gradient_of_an_empty_image(H, W):
    """An image without rows or columns is all padding: no load of it, and every
    tap's gradient is the sum of go times the padding's factor."""
    g = ops.conv_geom((2, 3, H, W), 3, 1, 2, 1)
    gen = torch.Generator(device="cuda").manual_seed(1)
    go = torch.randn(2, 3, g.OH, g.OW, generator=gen, device="cuda")
    img = torch.zeros(64, dtype=torch.int8, device="cuda")      # a valid pointer to no pixels
    tw = torch.randn(256, generator=gen, device="cuda")
    ws = torch.empty(L.query("atx_dwconv_bwd_weight_workspace_bytes", g) // 4, device="cuda")
    gw = torch.empty(3, 9, device="cuda")
    L.call("atx_dwconv_bwd_weight", L.ptr(go), L.ptr(img), 0, g, 77, None, L.ptr(tw), None, None,
           None, None, L.ptr(gw), L.ptr(ws), L.stream_of(go))
    want = (go * tw[77]).double().sum((0, 2, 3)).unsqueeze(1).expand(3, 9)
    assert bool(((gw.double() - want).abs() <= 1e-5).all())


def test_weight_gradient_of_a_long_batch():
    """15360 images of 1 x 4 over 2048 channels: one 1 in each of the first 256
    images, 2^-24 (half an ulp of 1, which a chain beside it drops) elsewhere.
    Chains of at most two tasks lose at most 8 x 2^-24 of the result beside
    the 1s, and 32 partial sums as many roundings: 2e-6 bounds both; one
    chain over the batch would lose 1.4e-5."""
    N, C = 15360, 2048
    g = ops.conv_geom((N, C, 1, 4), 3, 1, 1, 1)
    go = torch.full((N, C, 1, 4), 2.0 ** -24, device="cuda")
    go[:256, :, 0, 0] = 1.0
    img = torch.zeros(N, C, 1, 4, dtype=torch.int8, device="cuda")
    gw = ops.dwconv_backward_weight(go, img, torch.ones(256, device="cuda"), g, 128)
    want = 256 + (N * 4 - 256) * 2.0 ** -24
    assert float((gw.double() / want - 1).abs().max()) <= 2e-6
