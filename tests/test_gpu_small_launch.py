"""The GEMM kernel's tiles for small launches: same bits as the wide tiles.

A layer with few output pixels runs on the smallest tile whose workgroups fit
the chip in one round; the K order (taps, planes, 16-channel steps) is the same
in every tile, so its result equals the LDS-DMA / register-staged tiles' bit
for bit, and the default pick's.  Compared against f64 as well.
"""
import ctypes

import numpy as np
import pytest

import pyoracle as O
from gpu_util import announce
from vdamd import lib

pytestmark = pytest.mark.gpu

SMALL = list(range(92, 102))
BANDS = [57, 58, 59, 64, 65, 76, 77, 78, 79]


def run_tiles(d, dy, shape, tiles):
    outs = {}
    for t in tiles:
        d.tile = t
        if t >= 0 and not lib.lib().vdk_conv2d_tile_fits_ex(t, d):
            continue
        lib.check(lib.lib().vdk_conv2d_ex(d, None))
        lib.check(lib.lib().vdk_synchronize())
        outs[t] = dy.to_array(np.uint16, shape)
    return outs


# pixels around the 32 / 64 / 128 tile edges, outputs that no tile divides,
# one and several K chunks, 1-D strides and taps, and a 2-D stride-2 3x3
CASES = [
    # B, H, W, IC, OC, KH, KW, stride, pad, residual
    (1, 1, 1, 128, 32, 1, 1, 1, 0, False),
    (1, 1, 31, 128, 40, 1, 1, 1, 0, True),
    (1, 1, 159, 768, 768, 1, 1, 1, 0, True),
    (3, 1, 53, 256, 200, 1, 1, 1, 0, False),
    (2, 1, 129, 64, 72, 1, 1, 1, 0, True),
    (5, 1, 259, 96, 136, 1, 5, 1, 0, False),
    (1, 1, 639, 512, 512, 1, 3, 2, 0, False),
    (2, 1, 600, 512, 128, 1, 2, 2, 0, False),
    (1, 20, 75, 128, 256, 3, 3, 2, 1, False),
    (1, 21, 33, 64, 128, 3, 3, 2, 1, False),
    (1, 40, 37, 32, 32, 3, 3, 2, 1, False),
]


@pytest.mark.parametrize("case", CASES)
def test_small_tiles_bitwise(case):
    B, H, W, IC, OC, KH, KW, stride, pad, res = case
    rng = np.random.default_rng(sum(case[:9]))
    announce(f"small launch {case}")
    x = rng.standard_normal((B, H, W, IC)).astype(np.float16)
    w = (rng.standard_normal((OC, KH, KW, IC)) * np.sqrt(2.0 / (KH * KW * IC))).astype(np.float16)
    b = rng.uniform(-0.5, 0.5, OC).astype(np.float32)
    sh = stride if KH > 1 else 1
    Ho = (H + 2 * (pad if KH > 1 else 0) - KH) // sh + 1
    Wo = (W + 2 * pad - KW) // stride + 1
    keep = [lib.DeviceBuffer.from_array(v) for v in (x, w, b)]
    d = lib.ConvDesc()
    d.x, d.batch, d.H, d.W, d.IC = keep[0].ptr, B, H, W, IC
    d.w, d.OC, d.KH, d.KW = keep[1].ptr, OC, KH, KW
    d.stride_h, d.stride_w, d.pad_h, d.pad_w = sh, stride, pad if KH > 1 else 0, pad
    d.dil_h = d.dil_w = 1
    d.bias, d.act = keep[2].ptr, lib.ACT_RELU
    if res:
        r = rng.standard_normal((B, Ho, Wo, OC)).astype(np.float16)
        keep.append(lib.DeviceBuffer.from_array(r))
        d.residual = keep[3].ptr
    dy = lib.DeviceBuffer(B * Ho * Wo * OC * 2)
    d.y = dy.ptr
    ref_tile = 18 if IC % 64 == 0 else 39      # LDS-DMA tiles with 64- / 32-channel chunks
    outs = run_tiles(d, dy, (B, Ho, Wo, OC), [ref_tile, -1] + SMALL)
    assert sum(t >= 92 for t in outs) >= 2, sorted(outs)
    for t, o in outs.items():
        assert np.array_equal(o, outs[ref_tile]), f"tile {t}"
    # f16 products are exact in f32; K f32 additions (half an ulp each) and the f16 store
    xp = np.pad(x.astype(np.float64), ((0, 0), (d.pad_h, d.pad_h), (d.pad_w, d.pad_w), (0, 0)))
    want = np.zeros((B, Ho, Wo, OC))
    mag = np.zeros((B, Ho, Wo, OC))
    for kh in range(KH):
        for kw in range(KW):
            xs = xp[:, kh:kh + (Ho - 1) * sh + 1:sh, kw:kw + (Wo - 1) * stride + 1:stride]
            want += xs @ w[:, kh, kw].astype(np.float64).T
            mag += np.abs(xs) @ np.abs(w[:, kh, kw].astype(np.float64)).T
    want += b
    mag += np.abs(b)
    if res:
        want += r
        mag += np.abs(r)
    want = np.maximum(want, 0)
    got = outs[-1].view(np.float16).astype(np.float64)
    K = KH * KW * IC
    assert (np.abs(got - want) <= K * 2.0 ** -24 * mag + 2.0 ** -11 * np.abs(want) + 2.0 ** -24).all()


@pytest.mark.parametrize("split,KH,stride,IC,OC", [(1, 1, 1, 128, 64), (1, 1, 1, 64, 32), (2, 3, 2, 64, 128),
                                                   (1, 3, 2, 128, 72), (2, 1, 1, 32, 64)])
def test_small_tiles_split_bitwise(split, KH, stride, IC, OC):
    """Split-f16 inputs (two or three plane terms per tap), 1x1 and the stride-2
    3x3 downsamples, against the LDS-DMA tile with the same chunk width."""
    rng = np.random.default_rng(split + KH + IC + OC)
    B, H, W = 2, 10, 91
    announce(f"small launch split {split} K {KH} s {stride} {IC}->{OC}")
    x = rng.standard_normal((B, H, W, IC)).astype(np.float32)
    w = (rng.standard_normal((OC, KH, KH, IC)) * np.sqrt(2.0 / (KH * KH * IC))).astype(np.float32)
    if split == 2:
        w = w.astype(np.float16).astype(np.float32)

    def halves(v):
        hi = v.astype(np.float16)
        return hi, (v - hi.astype(np.float32)).astype(np.float16)

    wh, wl = halves(w)
    pack = np.concatenate([wh, wh] if split == 2 else [wh, wh, wl], axis=3)
    bias = rng.uniform(-0.5, 0.5, OC).astype(np.float32)
    keep = [lib.DeviceBuffer.from_array(np.ascontiguousarray(v)) for v in
            (np.concatenate(halves(x), axis=3), pack, bias)]
    pad = KH // 2
    Ho, Wo = (H + 2 * pad - KH) // stride + 1, (W + 2 * pad - KH) // stride + 1
    d = lib.ConvDesc()
    d.x, d.batch, d.H, d.W, d.IC, d.x_stride, d.x_lo = keep[0].ptr, B, H, W, IC, 2 * IC, IC
    d.w, d.OC, d.KH, d.KW = keep[1].ptr, OC, KH, KH
    d.stride_h = d.stride_w = stride
    d.pad_h = d.pad_w = pad
    d.dil_h = d.dil_w = 1
    d.bias, d.act, d.split = keep[2].ptr, lib.ACT_NONE, split
    dy = lib.DeviceBuffer(B * Ho * Wo * 2 * OC * 2)
    d.y, d.y_stride, d.y_lo = dy.ptr, 2 * OC, OC
    ref_tile = 18 if IC % 64 == 0 else 39
    outs = run_tiles(d, dy, (B, Ho, Wo, 2 * OC), [ref_tile, -1] + SMALL)
    assert sum(t >= 92 for t in outs) >= 2, sorted(outs)
    for t, o in outs.items():
        assert np.array_equal(o, outs[ref_tile]), f"tile {t}"
    o = outs[-1].view(np.float16).astype(np.float64)
    got = o[..., :OC] + o[..., OC:]
    want = np.stack([O.conv2d_g(x[c].transpose(2, 0, 1), np.ascontiguousarray(w.transpose(0, 3, 1, 2)), sh=stride,
                                sw=stride, ph=pad, pw=pad, bias=bias, f64=True) for c in range(B)])
    assert np.abs(got.transpose(0, 3, 1, 2) - want).max() <= 2e-6 * np.abs(want).max()


@pytest.mark.parametrize("batch,T,dil,scale", [(1, 5, 4, 8), (1, 32, 2, 8), (1, 95, 2, 8), (5, 259, 4, 8),
                                              (2, 333, 3, 4), (40, 301, 4, 8), (1, 1198, 3, 8)])
def test_res2_block_out_tiles(batch, T, dil, scale):
    """One ECAPA Res2Net block over many short tiles: every split into time
    tiles gives the bits of the block run in place, one clip at a time (few
    tiles or one), and x stays as it was."""
    rng = np.random.default_rng(batch + T + dil + scale)
    G, L = 128, lib.lib()
    S = (scale + 1) * G
    announce(f"res2 block out B={batch} T={T} dil={dil} scale={scale}")
    x = rng.standard_normal((batch, T, S), dtype=np.float32).astype(np.float16)
    keep, rw = [], lib.Res2Weights()
    for j in range(scale - 1):
        w = (rng.standard_normal((G, 3, G)) * np.sqrt(2.0 / (3 * G))).astype(np.float16)
        vec = [rng.uniform(lo, hi, G).astype(np.float32) for lo, hi in ((-0.1, 0.1), (0.5, 1.0), (-0.2, 0.2))]
        bufs = [lib.DeviceBuffer.from_array(v) for v in [w] + vec]
        keep += bufs
        rw.w[j], rw.bias[j], rw.scale[j], rw.shift[j] = (b.ptr for b in bufs)
    dx = lib.DeviceBuffer.from_array(x)
    ys = scale * G + 64
    dy = lib.DeviceBuffer.from_array(np.zeros((batch, T, ys), np.float16))
    lib.check(L.vdk_res2_block_out(dx.ptr, S, batch, T, G, scale, dil, rw, dy.ptr, ys, None))
    lib.check(L.vdk_synchronize())
    got = dy.to_array(np.uint16, (batch, T, ys))
    assert np.array_equal(dx.to_array(np.uint16, (batch, T, S)), x.view(np.uint16))
    assert not got[:, :, scale * G:].any()
    for c in sorted({0, batch // 2, batch - 1}):
        one = lib.DeviceBuffer.from_array(x[c:c + 1])
        lib.check(L.vdk_res2_block(one.ptr, S, 1, T, G, scale, dil, rw, None))
        lib.check(L.vdk_synchronize())
        assert np.array_equal(got[c, :, :scale * G], one.to_array(np.uint16, (1, T, S))[0, :, :scale * G])
    # the first group against f64 (f32 sums of 3 * 128 products, then the f16 store)
    c = batch - 1
    w, b, sc, sh = (k.to_array(t, s).astype(np.float64) for k, t, s in
                    zip(keep[:4], (np.float16,) + (np.float32,) * 3, ((G, 3, G), (G,), (G,), (G,))))
    xp = np.pad(x[c, :, 2 * G:3 * G].astype(np.float64), ((dil, dil), (0, 0)), mode="reflect")
    taps = [xp[k * dil:k * dil + T] for k in range(3)]
    want = np.maximum(sum(v @ w[:, k].T for k, v in enumerate(taps)) + b, 0) * sc + sh
    mag = (sum(np.abs(v) @ np.abs(w[:, k]).T for k, v in enumerate(taps)) + np.abs(b)) * sc + np.abs(sh)
    err = np.abs(got[c, :, :G].view(np.float16).astype(np.float64) - want)
    assert (err <= 3 * G * 2.0 ** -24 * mag + 2.0 ** -11 * np.abs(want) + 2.0 ** -24).all()


def pool_used():
    """Bytes in use of the device's stream-ordered memory pool."""
    hip, pool, used = lib.lib(), ctypes.c_void_p(), ctypes.c_uint64()
    assert hip.hipDeviceGetDefaultMemPool(ctypes.byref(pool), 0) == 0
    assert hip.hipMemPoolGetAttribute(pool, 7, ctypes.byref(used)) == 0   # hipMemPoolAttrUsedMemCurrent
    return used.value


def test_res2_block_in_place_gives_its_side_buffer_back():
    """In place over several time tiles the results go through a side buffer
    of the stream's pool: given back after the call, also when it fails on the
    way (here on an error that an earlier HIP call left behind)."""
    G, scale, T, dil, L = 128, 8, 400, 2, lib.lib()
    announce("res2 block in place: the side buffer")
    w, b = lib.DeviceBuffer.from_array(np.zeros((G, 3, G), np.float16)), lib.DeviceBuffer.from_array(np.zeros(G, np.float32))
    rw = lib.Res2Weights()
    for j in range(scale - 1):
        rw.w[j], rw.bias[j] = w.ptr, b.ptr
    S = (scale + 1) * G
    buf = lib.DeviceBuffer.from_array(np.zeros((4, T, S), np.float16))
    lib.check(L.vdk_synchronize())
    used = pool_used()
    lib.check(L.vdk_res2_block(buf.ptr, S, 4, T, G, scale, dil, rw, None))
    lib.check(L.vdk_synchronize())
    assert pool_used() == used
    assert L.hipSetDevice(1 << 20) != 0
    rc = L.vdk_res2_block(buf.ptr, S, 4, T, G, scale, dil, rw, None)
    L.hipGetLastError()
    lib.check(L.vdk_synchronize())
    assert rc != 0
    assert pool_used() == used
    lib.check(L.vdk_res2_block(buf.ptr, S, 4, T, G, scale, dil, rw, None))
    lib.check(L.vdk_synchronize())


@pytest.mark.parametrize("B,H,W,IC,OC,res,relu", [
    (1, 20, 75, 128, 128, True, True),      # one segment, the 5-row band's own width
    (2, 7, 76, 128, 128, False, True),      # just past it: two segments of 38
    (1, 6, 151, 64, 128, True, False),      # three segments, the last one narrower
    (3, 5, 13, 256, 256, True, True),       # narrow map, ragged bands
    (1, 1, 1, 16, 128, False, False),       # one pixel, one chunk
    (1, 10, 39, 256, 384, True, True),      # three output groups, two segments of 20
])
def test_band_tiles_bitwise(B, H, W, IC, OC, res, relu):
    """The stride-1 3x3 band kernels at any width: the 32 x 32 tiles and every
    band height and segment width give the same bits (so the batch may choose),
    with and without the chunk-major weights, and agree with f64."""
    rng = np.random.default_rng(B + H + W + IC + OC)
    announce(f"bands B={B} H={H} W={W} {IC}->{OC} res={res}")
    x = rng.standard_normal((B, H, W, IC)).astype(np.float16)
    w = (rng.standard_normal((OC, 3, 3, IC)) * np.sqrt(2.0 / (9 * IC))).astype(np.float16)
    b = rng.uniform(-0.5, 0.5, OC).astype(np.float32)
    r = rng.standard_normal((B, H, W, OC)).astype(np.float16)
    wc = np.ascontiguousarray(w.reshape(OC, 9, IC // 16, 16).transpose(2, 1, 0, 3))
    keep = [lib.DeviceBuffer.from_array(v) for v in (x, w, b, r, wc)]
    d = lib.ConvDesc()
    d.x, d.batch, d.H, d.W, d.IC = keep[0].ptr, B, H, W, IC
    d.w, d.OC, d.KH, d.KW = keep[1].ptr, OC, 3, 3
    d.stride_h = d.stride_w = d.pad_h = d.pad_w = d.dil_h = d.dil_w = 1
    d.bias, d.act = keep[2].ptr, lib.ACT_RELU if relu else lib.ACT_NONE
    if res:
        d.residual = keep[3].ptr
    dy = lib.DeviceBuffer(B * H * W * OC * 2)
    d.y = dy.ptr
    outs = run_tiles(d, dy, (B, H, W, OC), [-1] + BANDS)
    assert len(outs) == 10, sorted(outs)
    d.w_chunked = keep[4].ptr
    chunked = run_tiles(d, dy, (B, H, W, OC), [-1] + BANDS)
    for o in (outs, chunked):
        for t in o:
            assert np.array_equal(o[t], outs[64]), f"tile {t}"
    xp = np.pad(x.astype(np.float64), ((0, 0), (1, 1), (1, 1), (0, 0)))
    want, mag = b + np.zeros((B, H, W, OC)), np.abs(b) + np.zeros((B, H, W, OC))
    for kh in range(3):
        for kw in range(3):
            xs = xp[:, kh:kh + H, kw:kw + W]
            want += xs @ w[:, kh, kw].astype(np.float64).T
            mag += np.abs(xs) @ np.abs(w[:, kh, kw].astype(np.float64)).T
    if res:
        want += r
        mag += np.abs(r)
    if relu:
        want = np.maximum(want, 0)
    got = outs[-1].view(np.float16).astype(np.float64)
    assert (np.abs(got - want) <= 9 * IC * 2.0 ** -24 * mag + 2.0 ** -11 * np.abs(want) + 2.0 ** -24).all()


@pytest.mark.parametrize("T,H,G,K", [(149, 768, 16, 128), (31, 128, 2, 128), (33, 96, 2, 33), (1, 128, 2, 7)])
def test_pos_conv_small_launch_bitwise(T, H, G, K):
    """wav2vec2's positional conv: one clip (32-frame workgroups) gives the
    bits it has in a batch that fills the chip (192-frame workgroups)."""
    rng = np.random.default_rng(T + H + K)
    announce(f"pos_conv small T={T} H={H} G={G} K={K}")
    B, icg, L = 1 + 256 // (G * ((T + 31) // 32)), H // G, lib.lib()
    x = rng.standard_normal((B, T, H)).astype(np.float16)
    w = np.zeros((G, 64, K, icg), np.float16)
    w[:, :icg] = rng.standard_normal((G, icg, K, icg)) * np.sqrt(1.0 / (icg * K))
    keep = [lib.DeviceBuffer.from_array(v) for v in (x, w, (0.1 * rng.standard_normal(H)).astype(np.float32))]
    dy, d1 = lib.DeviceBuffer(B * T * H * 4), lib.DeviceBuffer(T * H * 4)
    lib.check(L.vdk_pos_conv(keep[0].ptr, B, T, H, G, keep[1].ptr, keep[2].ptr, K, K // 2, dy.ptr, None))
    for c in (0, B - 1):
        lib.check(L.vdk_pos_conv(keep[0].ptr + c * T * H * 2, 1, T, H, G, keep[1].ptr, keep[2].ptr, K, K // 2, d1.ptr,
                                 None))
        lib.check(L.vdk_synchronize())
        assert np.array_equal(d1.to_array(np.uint32, (T, H)), dy.to_array(np.uint32, (B, T, H))[c])


@pytest.mark.parametrize("n,B,T,C", [(13, 1, 159, 768), (1, 3, 1, 32), (25, 2, 1000, 100), (32, 1, 7, 1024)])
def test_time_mean_states_equals_one_by_one(n, B, T, C):
    """The pooled states in one launch: the bits of one accumulating launch per
    state, zero weights skipped, a gap between the states."""
    rng = np.random.default_rng(n + T + C)
    announce(f"time_mean_states n={n} B={B} T={T} C={C}")
    L, gap = lib.lib(), (B * T * C + 71) // 8 * 8
    x = rng.standard_normal((n, gap)).astype(np.float16)
    w = rng.uniform(-1, 1, n).astype(np.float32)
    w[n // 2 + 1:n // 2 + 2] = 0.0
    dx, do, dr = lib.DeviceBuffer.from_array(x), lib.DeviceBuffer(B * C * 4), lib.DeviceBuffer(B * C * 4)
    lib.check(L.vdk_time_mean_states(dx.ptr, gap, n, B, T, C, w.ctypes.data_as(ctypes.POINTER(ctypes.c_float)), do.ptr,
                                     None))
    first = True
    for i in range(n):
        if w[i] != 0:
            lib.check(L.vdk_time_mean_acc(dx.ptr + i * gap * 2, 0, B, T, C, ctypes.c_float(w[i]), 0 if first else 1,
                                          dr.ptr, None))
            first = False
    lib.check(L.vdk_synchronize())
    assert np.array_equal(do.to_array(np.uint32, (B, C)), dr.to_array(np.uint32, (B, C)))


@pytest.mark.parametrize("B,H,W,IC,OC,split,groups", [(2, 10, 91, 128, 128, 2, False), (1, 10, 33, 128, 128, 1, False),
                                                      (1, 20, 50, 64, 64, 2, False), (1, 1, 1, 64, 32, 2, False),
                                                      (1, 13, 37, 32, 32, 2, True), (1, 7, 45, 32, 64, 1, False)])
def test_slim_split_bitwise(B, H, W, IC, OC, split, groups):
    """Split-f16 stride-1 3x3 convs on 32 x 32 tiles: the halo kernel's bits (or
    the register-weight kernel's, where the channel groups need it), the
    default's, and f64 to split-f16's accuracy."""
    rng = np.random.default_rng(B + H + W + IC + OC)
    announce(f"slim split B={B} H={H} W={W} {IC}->{OC} split={split} groups={groups}")
    x = rng.standard_normal((B, H, W, IC)).astype(np.float32)
    w = (rng.standard_normal((OC, 3, 3, IC)) * np.sqrt(2.0 / (9 * IC))).astype(np.float32)
    if split == 2:
        w = w.astype(np.float16).astype(np.float32)

    def halves(v):
        hi = v.astype(np.float16)
        return hi, (v - hi.astype(np.float32)).astype(np.float16)

    wh, wl = halves(w)
    bias = rng.uniform(-0.5, 0.5, OC).astype(np.float32)
    keep = [lib.DeviceBuffer.from_array(np.ascontiguousarray(v)) for v in
            (np.concatenate(halves(x), axis=3), np.concatenate([wh, wh] if split == 2 else [wh, wh, wl], axis=3), bias)]
    d = lib.ConvDesc()
    d.x, d.batch, d.H, d.W, d.IC, d.x_stride, d.x_lo = keep[0].ptr, B, H, W, IC, 2 * IC, IC
    d.w, d.OC, d.KH, d.KW = keep[1].ptr, OC, 3, 3
    d.stride_h = d.stride_w = d.pad_h = d.pad_w = d.dil_h = d.dil_w = 1
    d.bias, d.act, d.clamp_hi, d.split = keep[2].ptr, lib.ACT_RELU, 20.0, split
    if groups:   # one 32-channel group, its lo half inside the group stride
        d.x_group, d.x_group_stride, d.y_group, d.y_group_stride = 32, 64, 32, 64
    dy = lib.DeviceBuffer(B * H * W * 2 * OC * 2)
    d.y, d.y_stride, d.y_lo = dy.ptr, 2 * OC, OC
    outs = run_tiles(d, dy, (B, H, W, 2 * OC), [-1, 26, 28, 30, 72, 74, 75, 102])
    assert 102 in outs and len(outs) >= 3, sorted(outs)
    for t, o in outs.items():
        assert np.array_equal(o, outs[102]), f"tile {t}"
    o = outs[102].view(np.float16).astype(np.float64)
    got = o[..., :OC] + o[..., OC:]
    want = np.stack([O.conv2d_g(x[c].transpose(2, 0, 1), np.ascontiguousarray(w.transpose(0, 3, 1, 2)), ph=1, pw=1,
                                bias=bias, f64=True) for c in range(B)])
    want = np.clip(want, 0, 20)
    assert np.abs(got.transpose(0, 3, 1, 2) - want).max() <= 2e-6 * max(np.abs(want).max(), 1.0)


def test_band_output_past_two_gigabytes():
    """16 -> 128 channels over 5600 clips of 20 x 75 (output and residual of 2.15
    GB): the first and last clips have the bits they have in a batch of three."""
    B, H, W, IC, OC, n = 5600, 20, 75, 16, 128, 3
    rng = np.random.default_rng(5600)
    announce(f"band output of {B * H * W * OC * 2 / 2**30:.2f} GiB")
    x, r = (rng.standard_normal((n, H, W, c)).astype(np.float16) for c in (IC, OC))
    w = (rng.standard_normal((OC, 3, 3, IC)) * np.sqrt(2.0 / (9 * IC))).astype(np.float16)
    b = rng.uniform(-0.5, 0.5, OC).astype(np.float32)
    L, dw, db = lib.lib(), lib.DeviceBuffer.from_array(w), lib.DeviceBuffer.from_array(b)

    def run(batch):
        clip = H * W * 2
        dx, dr, dy = (lib.DeviceBuffer(batch * clip * c) for c in (IC, OC, OC))
        dx.copy_from(np.resize(x, (batch, H, W, IC)))
        for c0 in range(0, batch, 300):   # (300 % n == 0)
            part = np.resize(r, (min(300, batch - c0), H, W, OC))
            lib.check(L.vdk_memcpy_h2d(dr.ptr + c0 * clip * OC, part.ctypes.data, part.nbytes))
        d = lib.ConvDesc()
        d.x, d.batch, d.H, d.W, d.IC = dx.ptr, batch, H, W, IC
        d.w, d.OC, d.KH, d.KW = dw.ptr, OC, 3, 3
        d.stride_h = d.stride_w = d.pad_h = d.pad_w = d.dil_h = d.dil_w = 1
        d.bias, d.residual, d.act, d.y, d.tile = db.ptr, dr.ptr, lib.ACT_RELU, dy.ptr, -1
        lib.check(L.vdk_conv2d_ex(d, None))
        lib.check(L.vdk_synchronize())
        out = {}
        for c in range(n), range(batch - n, batch):
            for i in c:
                o = np.empty((H, W, OC), np.uint16)
                lib.check(L.vdk_memcpy_d2h(o.ctypes.data, dy.ptr + i * clip * OC, o.nbytes))
                out[i] = o
        return out

    want, got = run(n), run(B)
    for i, o in got.items():
        assert np.array_equal(o, want[i % n]), f"clip {i}"
