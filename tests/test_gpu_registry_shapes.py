"""Registry scoring at the edges of its launch shapes: chunks of 64 and 256 rows,
16- and 32-query blocks, 16-dim steps with a remainder, the two group counts of
the pick, rows that tie or hold no finite score, and the smallest workspace a
caller may bring.  Against the oracle's registry_topk: the same ranking, the
scores to one f32 rounding of the 64-bit value.
"""
import zlib

import numpy as np
import pytest

import pyoracle as O
from gpu_util import announce, device_ok
from test_gpu_registry import _check, _unit
from vdamd import lib

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not device_ok(), reason="no HIP device")]


@pytest.mark.parametrize("case", [
    (1, 63, 192, 5), (16, 65, 256, 16), (17, 64, 20, 17), (33, 257, 4, 64), (2, 16384, 192, 10),
    (16, 16385, 256, 5), (32, 16640, 20, 64), (65, 20001, 516, 16), (1, 30000, 512, 1), (3, 120000, 192, 64),
])
def test_registry_edges(case):
    B, N, D, k = case
    announce(f"registry edges B={B} N={N} D={D} k={k}")
    rng = np.random.default_rng(zlib.crc32(repr(case).encode()))
    reg = _unit(rng, N, D)
    if N >= 257:
        reg[N // 2:N // 2 + 80] = reg[7]      # a run of equal scores across chunks
        reg[N - 90:N - 4] = 0.0
    _check(_unit(rng, B, D), reg, k)


@pytest.mark.parametrize("N", [300, 20000])
def test_registry_equal_rows_and_smallest_workspace(N):
    """All rows equal: the k lowest rows; with a workspace of 256-row lists."""
    announce(f"registry equal rows N={N}")
    L = lib.lib()
    q = np.ones((20, 64), dtype=np.float32)
    reg = np.ones((N, 64), dtype=np.float32)
    k = 40
    ws = 20 * ((N + 255) // 256) * k * 12 + 256
    dq, dr, dw = lib.DeviceBuffer.from_array(q), lib.DeviceBuffer.from_array(reg), lib.DeviceBuffer(ws)
    di, ds = lib.DeviceBuffer(20 * k * 4), lib.DeviceBuffer(20 * k * 4)
    lib.check(L.vdk_registry_topk(dq.ptr, 20, dr.ptr, N, 64, k, dw.ptr, ws, di.ptr, ds.ptr, None))
    lib.check(L.vdk_synchronize())
    assert np.array_equal(di.to_array(np.int32, (20, k)), np.tile(np.arange(k, dtype=np.int32), (20, 1)))
    assert np.all(ds.to_array(np.float32, (20, k)) == 64.0)
    assert L.vdk_registry_topk(dq.ptr, 20, dr.ptr, N, 64, k, dw.ptr, ws - 1, di.ptr, ds.ptr, None) != 0


def test_registry_rows_without_a_finite_score():
    """Rows whose score is not finite are never picked; short of k, the list
    ends with INT_MAX at -inf."""
    announce("registry rows with NaN / inf")
    L = lib.lib()
    rng = np.random.default_rng(5)
    reg = _unit(rng, 100, 32)
    reg[::2, 3] = np.nan
    reg[1::4, 5] = np.inf
    q = np.abs(_unit(rng, 2, 32))
    good = [r for r in range(100) if np.isfinite(reg[r]).all()]
    k = 30
    ws = L.vdk_registry_topk_workspace_size(2, 100, k)
    dq, dr, dw = lib.DeviceBuffer.from_array(q), lib.DeviceBuffer.from_array(reg), lib.DeviceBuffer(ws)
    di, ds = lib.DeviceBuffer(2 * k * 4), lib.DeviceBuffer(2 * k * 4)
    lib.check(L.vdk_registry_topk(dq.ptr, 2, dr.ptr, 100, 32, k, dw.ptr, ws, di.ptr, ds.ptr, None))
    lib.check(L.vdk_synchronize())
    idx, score = di.to_array(np.int32, (2, k)), ds.to_array(np.float32, (2, k))
    oi, _ = O.registry_topk(q, reg[good], len(good))
    for b in range(2):
        assert idx[b, :len(good)].tolist() == [good[i] for i in oi[b]]
        assert np.all(idx[b, len(good):] == np.iinfo(np.int32).max)
        assert np.all(np.isneginf(score[b, len(good):]))
