"""Which way atx_conv_bwd_data goes to an image gradient, told from its
workspace (a host query, no GPU): the tap GEMM where it measured faster, the
columns where padding would be most of its work, and no columns for a padded
1x1 conv; and how many blocks share a depthwise weight gradient."""
import pytest

from approxtorch_amd.backend import _lib as L
from approxtorch_amd.backend import ops


def route(shape, Oc, k, s, p, d=1):
    g = ops.conv_geom(shape, k, s, p, d)
    K, P = g.C * g.KH * g.KW, g.N * g.OH * g.OW
    rest = L.query("atx_conv_bwd_data_workspace_bytes", g, Oc) - \
        6 * L.round_up(K, 128) * L.round_up(Oc, 32)
    planes = L.round_up(P * 6 * L.round_up(Oc, 32), 256)
    image, columns = 4 * g.N * g.C * g.H * g.W, 4 * K * P
    slices = (0, *range(2, 65))
    fits = {"tap": (rest - planes) % image == 0 and (rest - planes) // image in slices,
            "columns": rest % columns == 0 and rest // columns - 1 in slices,
            "image": rest % image == 0 and rest // image in slices}
    assert not (fits["tap"] and fits["columns"])         # the sizes tell them apart
    # stride 1: the columns are KH KW images, so they are looked for first
    return next(name for name, ok in fits.items() if ok)


# (tap GEMM, columns and their fold in us, LRE table)
@pytest.mark.parametrize("shape,Oc,k,s,p,way", [
    ((64, 64, 56, 56), 64, 3, 1, 1, "tap"),             # 137 / 296
    ((64, 128, 28, 28), 128, 3, 1, 1, "tap"),           # 126 / 175
    ((64, 512, 7, 7), 512, 3, 1, 1, "tap"),             # 119 / 135
    ((64, 128, 56, 56), 128, 3, 2, 1, "tap"),           # 205 / 242
    ((64, 64, 56, 56), 8, 3, 1, 1, "tap"),              # 82 / 248
    ((128, 256, 28, 28), 8, 3, 1, 1, "tap"),            # 147 / 466
    ((64, 3, 64, 64), 64, 3, 1, 1, "columns"),          # 125 / 38
    ((64, 8, 56, 56), 128, 3, 1, 1, "columns"),         # 270 / 77
    ((64, 4, 64, 64), 512, 3, 1, 1, "columns"),         # 1337 / 172
    ((32, 3, 224, 224), 64, 7, 2, 3, "columns"),        # 803 / 241
    ((64, 24, 56, 56), 24, 3, 2, 1, "columns"),         # 66 / 48
    ((13, 1, 1024, 1024), 2, 3, 1, 1, "columns"),       # 3262 / 693
    ((76, 3, 24, 126), 131, 3, 1, 1, "columns"),        # 366 / 59
    ((64, 64, 56, 56), 64, 1, 1, 1, "image"),
    ((2, 24, 9, 11), 40, 1, 1, (0, 2), "image"),
    ((64, 64, 56, 56), 64, 1, 1, 0, "image")])
def test_route(shape, Oc, k, s, p, way):
    assert route(shape, Oc, k, s, p) == way


@pytest.mark.parametrize("shape,s,least", [
    ((32, 36, 85, 32), 2, 216),        # 41 us on 72 blocks, 17 on 216
    ((64, 144, 56, 56), 1, 2016),      # 14-row runs
    ((1, 8, 64, 64), 1, 8)])           # no more work to share
def test_depthwise_weight_gradient_blocks(shape, s, least):
    g = ops.conv_geom(shape, 3, s, 0 if s == 2 else 1, 1)
    assert L.query("atx_dwconv_bwd_weight_workspace_bytes", g) // 36 >= least
