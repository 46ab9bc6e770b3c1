"""GPU parity of the LUT GEMM's byte-plane tables and matrix-core sums at the
edges of its layout: a single tap to two quads and a partial one, rows around
a row quad, a wave (256) and a tile (2048), channels around a 16-channel chunk
and a 32-channel tile, every byte value in both planes, both classes, full and
upper-half tables, and forced split-K and stream-K schedules.

Bar: the int32 sums equal the int64 oracle's.
"""
import numpy as np
import pytest
import torch

from approxtorch_amd.backend import ops
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def lut_of(kind, rng):
    """Random entries over the whole range of a class, its extremes included."""
    lo, hi = (-32767, 32767) if kind == "i16" else (0, 65535)
    lut = rng.integers(lo, hi + 1, 65536)
    lut[rng.integers(0, 65536, 512)] = lo
    lut[rng.integers(0, 65536, 512)] = hi
    return lut


def check(kind, upper, N, K, L, Oc):
    rng = np.random.default_rng(1000 * K + 10 * L + Oc)
    lut = lut_of(kind, rng)
    xi = rng.integers(128 if upper else 0, 256, (N, K, L)).astype(np.uint8)
    wi = rng.integers(0, 256, (Oc, K)).astype(np.uint8)
    if not upper:
        xi.reshape(-1)[0] = 0                            # one index below 128: full tables
    y = ops.lut_gemm_i32(torch.from_numpy(xi).cuda(), torch.from_numpy(wi).cuda(),
                         torch.from_numpy(lut.astype(np.float32)).cuda())
    assert np.array_equal(y.cpu().numpy().astype(np.int64), O.lut_gemm_i64(xi, wi, lut))


@pytest.mark.parametrize("kind", ["i16", "u16"])
@pytest.mark.parametrize("upper", [False, True])
@pytest.mark.parametrize("N,K,L,Oc", [
    (1, 1, 1, 1), (1, 3, 3, 15), (2, 4, 126, 16), (1, 5, 255, 17), (3, 8, 256, 31),
    (1, 9, 257, 32), (1, 12, 2047, 33), (7, 13, 293, 48), (1, 64, 2052, 65), (5, 37, 1000, 7)])
def test_lut_gemm_layout_edges(kind, upper, N, K, L, Oc):
    check(kind, upper, N, K, L, Oc)


@pytest.mark.parametrize("kind", ["i16", "u16"])
@pytest.mark.parametrize("upper", [False, True])
@pytest.mark.parametrize("N,K,L,Oc,splits", [
    (1, 8, 1, 1, 2), (2, 9, 126, 16, 3), (1, 12, 2047, 33, 3), (7, 21, 293, 48, 2),
    (1, 64, 2052, 65, 4), (5, 37, 1000, 7, 4)])
def test_lut_gemm_split_edges(monkeypatch, kind, upper, N, K, L, Oc, splits):
    """The same edges in raw int32 partial sums and their reduce."""
    monkeypatch.setenv("ATX_LUT_SPLITS", str(splits))
    assert ops.L.query("atx_lut_gemm_workspace_bytes", N, K, L, Oc) == splits * N * L * Oc * 4
    check(kind, upper, N, K, L, Oc)


@pytest.mark.parametrize("kind", ["i16", "u16"])
@pytest.mark.parametrize("upper", [False, True])
@pytest.mark.parametrize("N,K,L,Oc", [
    (1, 1029, 1, 1), (1, 1030, 255, 17), (1, 523, 257, 48), (3, 701, 684, 65), (1, 2053, 64, 7)])
def test_lut_gemm_stream_k_edges(monkeypatch, kind, upper, N, K, L, Oc):
    """The same edges in the stream-K slots (more quads than workgroups)."""
    monkeypatch.setenv("ATX_LUT_SCHEDULE", "stream_k")
    assert ops.L.query("atx_lut_gemm_workspace_bytes", N, K, L, Oc) == 255 * 2048 * 32 * 4
    check(kind, upper, N, K, L, Oc)
