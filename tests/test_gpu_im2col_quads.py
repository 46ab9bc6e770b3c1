"""The implicit-im2col operand of byte images whose rows are whole dwords
(four taps of a row quad from aligned dwords), against an unfold on the CPU
and the kernel that reads byte by byte."""
import zlib

import numpy as np
import pytest
import torch

from approxtorch_amd.backend import _lib as L
from approxtorch_amd.backend import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"

# (N, C, H, W, KH, KW, SH, SW, PH, PW, DH, DW), W % 4 == 0 and OW % 4 == 0:
# one quad per row, ragged heights and tap counts, both column strides, every
# alignment of a tap (kernel widths, dilations), padding wider than a dword,
# no padding, 1x1 with a stride, padding rows (every N*OH*OW is far from 2048).
CASES = [
    (1, 1, 4, 4, 3, 3, 1, 1, 1, 1, 1, 1), (2, 3, 5, 8, 3, 3, 1, 1, 1, 1, 1, 1),
    (3, 5, 9, 12, 5, 3, 2, 1, 2, 1, 1, 1), (2, 4, 7, 8, 3, 3, 1, 1, 2, 2, 2, 2),
    (2, 2, 6, 4, 1, 11, 1, 1, 0, 5, 1, 1), (2, 3, 6, 12, 5, 5, 1, 1, 0, 0, 1, 1),
    (2, 7, 11, 16, 3, 3, 2, 2, 1, 1, 1, 1), (1, 3, 24, 24, 7, 7, 2, 2, 3, 3, 1, 1),
    (2, 3, 16, 16, 3, 3, 2, 2, 3, 3, 3, 3), (3, 6, 5, 16, 1, 1, 2, 2, 0, 0, 1, 1),
    (2, 1, 3, 4, 3, 15, 1, 1, 1, 7, 1, 1), (4, 33, 14, 28, 3, 3, 1, 1, 1, 1, 1, 1),
]


def operand(img, g, pad, pad_dev):
    K, Rpad = g.C * g.KH * g.KW, L.round_up(g.N * g.OH * g.OW, L.ROW_TILE)
    xt = torch.full((L.operand_rows(K), Rpad), -1, dtype=torch.int16, device=DEV)
    L.call("atx_im2col_rows", L.ptr(img), 0 if img.dtype == torch.int8 else 1, g, pad,
           L.ptr(pad_dev), L.ptr(xt), Rpad, L.stream_of(img))
    return xt.cpu().numpy().astype(np.int64) & 0xFFFF


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("dtype", [torch.int8, torch.uint8])
def test_operand_of_dword_rows(case, dtype):
    N, C, H, W, KH, KW, SH, SW, PH, PW, DH, DW = case
    g = ops.conv_geom((N, C, H, W), (KH, KW), (SH, SW), (PH, PW), (DH, DW))
    assert g.W % 4 == 0 and g.OW % 4 == 0
    r = np.random.default_rng(zlib.crc32(repr(case).encode()))
    idx = r.integers(0, 256, (N, C, H, W))
    off = 128 if dtype == torch.int8 else 0
    flat = torch.zeros(idx.size + 4, dtype=dtype, device=DEV)
    pad = 77
    pad_dev = None if dtype == torch.int8 else torch.tensor([float(pad)], device=DEV)
    got = []
    for shift in (0, 1):                       # an unaligned image is read byte by byte
        img = flat[shift:shift + idx.size].view(N, C, H, W)
        img.copy_(torch.from_numpy(idx - off).to(dtype))
        got.append(operand(img, g, pad if pad_dev is None else 0, pad_dev))
    assert np.array_equal(got[0], got[1])
    cols = torch.nn.functional.unfold(
        torch.nn.functional.pad(torch.from_numpy(idx).double(), (PW, PW, PH, PH), value=pad),
        (KH, KW), (DH, DW), 0, (SH, SW)).long().numpy()          # [N, K, L]
    K, R = C * KH * KW, N * g.OH * g.OW
    cols = cols.transpose(1, 0, 2).reshape(K, R)
    slot, row = np.meshgrid(np.arange(got[0].shape[0]), np.arange(got[0].shape[1]), indexing="ij")
    k = (slot & ~3) | ((slot + (row >> 2)) & 3)
    live = (k < K) & (row < R)
    v = np.where(live, cols[np.minimum(k, K - 1), np.minimum(row, R - 1)], 0)
    assert np.array_equal(got[0], np.where(live, v * 256 + ((v >> 1) & 3) * 16, 0))
