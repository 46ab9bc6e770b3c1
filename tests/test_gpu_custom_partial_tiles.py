"""Pair-table gradients where the last 2048-row tile lacks rows for some of its
eight waves of 256 rows: the waves without rows only build tables, and the
tile's workgroups come last in the order.

Bar: rel 1e-5 of the sum of |terms| plus 1e-6 against the fp64 oracle.
"""
import zlib

import numpy as np
import pytest
import torch

from approxtorch_amd.backend import ops
from oracle import oracle as O

pytestmark = pytest.mark.gpu

# (N, K, L, O): one row in the last tile, one wave full and one row more, seven
# waves full (no row for the eighth) and one row more (every wave has rows),
# with L % 4 == 0 (resident-table grad_w) and without, one and several quads
# per workgroup, K % 4 != 0, O % 16 != 0, and 16 quads and more (split over
# workgroups)
SHAPES = [(1, 9, 1, 5), (1, 9, 255, 17), (1, 9, 257, 40), (1, 6, 1792, 24), (1, 6, 1793, 24),
          (1, 66, 2049, 20), (1, 130, 2303, 33), (3, 70, 1301, 16), (7, 64, 586, 48),
          (8, 12, 268, 130), (4, 37, 964, 16), (32, 40, 196, 24), (64, 66, 65, 40),
          # many quads: runs of them per workgroup, the last one shorter, on
          # partial tiles alone, with full ones before them, and on full ones
          (10, 609, 25, 20), (87, 405, 25, 40), (41, 333, 49, 24)]


@pytest.mark.parametrize("shape", SHAPES)
def test_custom_grads_partial_row_tiles(shape):
    N, K, L, Oc = shape
    r = np.random.default_rng(zlib.crc32(repr(shape).encode()))
    xi = r.integers(0, 256, (N, K, L), dtype=np.uint8)
    wi = r.integers(0, 256, (Oc, K), dtype=np.uint8)
    dx, dw = r.standard_normal((2, 65536)).astype(np.float32)
    go = r.standard_normal((N, Oc, L)).astype(np.float32)
    dev = [torch.from_numpy(a).cuda() for a in (xi, wi, go, dx, dw)]
    gx, gw = ops.custom_grads(ops.pack_rows_u8(dev[0]), *dev[1:], N, K, L)
    for got, want, terms in zip((gx, gw), O.gemm_grads(go, xi, wi, "custom", (dx, dw)),
                                O.gemm_grads(go, xi, wi, "custom", (dx, dw), absolute=True)):
        assert (np.abs(got.cpu().numpy() - want) <= 1e-5 * terms + 1e-6).all()
