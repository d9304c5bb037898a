"""The conv dispatch on the host (vdk_conv2d_pick, vdk_conv2d_tile_fits_ex): which
tile takes which call, over shapes, layouts and batches, with no GPU."""
import itertools

import pytest

from vdamd import lib

BATCHES = (1, 2, 5, 16, 24, 64, 256, 1500, 12000)


def desc(B, H, W, IC, OC, K=3, stride=1, pad=1, out_w=0, split=0, group=0, res=False, act=lib.ACT_RELU):
    d = lib.ConvDesc()
    d.batch, d.H, d.W, d.IC, d.OC, d.KH, d.KW = B, H, W, IC, OC, K, K
    d.stride_h = d.stride_w = stride
    d.pad_h = d.pad_w = pad
    d.dil_h = d.dil_w = 1
    d.out_w, d.act = out_w, act
    d.residual = 16 if res else None   # only its presence matters
    d.split = split
    if split:
        d.x_stride, d.x_lo, d.y_stride, d.y_lo, d.res_lo = 2 * IC, IC, 2 * OC, OC, OC
        d.res_stride = 2 * OC if res else 0
    if group:
        d.x_group = d.y_group = d.x_lo = d.y_lo = group
        d.x_group_stride = d.y_group_stride = 2 * group
    return d


def fits(t, d):
    return bool(lib.lib().vdk_conv2d_tile_fits_ex(t, d))


def too_large(d):
    return d.batch * d.H * d.W * (d.x_stride or d.IC) >= 1 << 30 or d.batch * d.H * d.W * (d.y_stride or d.OC) >= 1 << 31


# the register-weight, split-f16 register-weight, band and 32 x 32 3x3 kernels:
# they store every row as wide as they read it
WHOLE_ROWS = list(range(53, 60)) + list(range(64, 80)) + [102]


@pytest.mark.parametrize("split,group", [(0, 0), (1, 0), (2, 0), (2, 32)])
def test_cropped_3x3_never_on_whole_row_kernels(split, group):
    """out_w < W: no kernel that stores whole rows takes the call (it would
    write past y), explicitly or by default, and some kernel does."""
    L, n = lib.lib(), 0
    for IC, OC, H, W, res, act in itertools.product((32, 64, 128, 256), (32, 64, 128, 256), (1, 10, 20, 40),
                                                    (20, 38, 75, 77, 126, 300), (False, True),
                                                    (lib.ACT_RELU, lib.ACT_NONE)):
        if group and res:
            continue
        whole = desc(1, H, W, IC, OC, split=split, group=group, res=res, act=act)
        n += sum(fits(t, whole) for t in WHOLE_ROWS if t < L.vdk_conv2d_tile_count())
        for out_w in (1, W - 7, W - 1):
            d = desc(1, H, W, IC, OC, out_w=out_w, split=split, group=group, res=res, act=act)
            for t in range(L.vdk_conv2d_tile_count()):
                assert not (t in WHOLE_ROWS and fits(t, d)), (t, IC, OC, H, W, out_w)
            for B in BATCHES:
                d.batch = B
                if not too_large(d):
                    t = L.vdk_conv2d_pick(d)
                    assert t >= 0 and t not in WHOLE_ROWS, (t, B, IC, OC, H, W, out_w)
    assert n > 100   # they do take the uncropped calls


# tiles by the order their sums run in: the halo kernel's split-f16 order (plane
# terms, 32-channel chunks, taps) and the band kernels' (16-channel chunks, taps,
# bias first); the rest run taps first, but for the 16-row MFMA tiles
def sum_order(t, d):
    if t in (70, 71, 73):
        return f"16-row MFMA, tile {t}"
    if t in (72, 74, 75, 102) or (26 <= t <= 32 and (d.split or d.IC > 32)):
        return "halo"
    if t in (57, 58, 59, 64, 65) or 76 <= t <= 79:
        return "band"
    return "taps"


@pytest.mark.parametrize("split,group", [(1, 0), (1, 16), (1, 32), (2, 0), (2, 16), (2, 32)])
def test_split_3x3_order_does_not_depend_on_the_batch(split, group):
    """Every batch of a split-f16 3x3 shape runs its sums in the same order, so a
    clip's bits do not depend on the batch it is in."""
    L = lib.lib()
    for IC, OC, H, W, act in itertools.product((16, 32, 64, 128), (16, 32, 64, 128), (1, 10, 20, 40),
                                               (13, 49, 91, 150, 998, 1998), (lib.ACT_RELU, lib.ACT_SILU)):
        if IC == 16 and (split != 2 or OC != 16) or (group == 32 and (IC % 32 or OC % 32)):
            continue
        seen = {}
        for B in BATCHES:
            d = desc(B, H, W, IC, OC, split=split, group=group, act=act)
            if not too_large(d):
                t = L.vdk_conv2d_pick(d)
                seen.setdefault(sum_order(t, d) if t >= 0 else "refused", []).append((B, t))
        assert len(seen) == 1, (IC, OC, H, W, act, seen)


def test_plain_3x3_order_does_not_depend_on_the_batch():
    """The same for f16 3x3 layers, up to the largest launch (outputs of 2^31
    elements)."""
    L, large = lib.lib(), 0
    for IC, OC, H, W, res in itertools.product((16, 32, 64, 128, 256), (32, 64, 128, 256, 384), (5, 10, 20, 80),
                                               (13, 38, 75, 77, 126, 300), (False, True)):
        seen = {}
        for B in BATCHES + (4000, 6000, 9000):
            d = desc(B, H, W, IC, OC, res=res)
            if not too_large(d):
                t = L.vdk_conv2d_pick(d)
                seen.setdefault(sum_order(t, d) if t >= 0 else "refused", []).append((B, t))
                large += OC % 128 == 0 and B * H * W * OC >= 1 << 30
        assert len(seen) == 1, (IC, OC, H, W, res, seen)
    assert large > 50


@pytest.mark.parametrize("IC,OC,seg_len,taken", [
    (128, 128, 100, True), (64, 128, 64, True), (1024, 512, 100, True), (96, 128, 100, True),
    (64, 128, 40, False),    # segments shorter than the wide tile's 64 pixels
    (32, 32, 100, False), (64, 8, 100, False), (96, 40, 100, False),   # 128-pixel tiles for narrow outputs
])
def test_segment_sums_taken_or_refused_at_every_batch(IC, OC, seg_len, taken):
    """seg_sum calls: whether a shape is taken does not depend on the batch (the
    small-launch tiles would take shorter segments)."""
    for B, T in itertools.product((1, 2, 8, 32), (1, 49, 249, 499)):
        d = desc(B, 1, T, IC, OC, K=1, pad=0)
        d.in_scale = d.in_shift = d.seg_sum = 16
        d.seg_len = seg_len
        assert (lib.lib().vdk_conv2d_pick(d) >= 0) == taken, (B, T)
