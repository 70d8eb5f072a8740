"""fp32 conv2d on the kernel whose blocks walk the flattened batch (1x1, 3x3 and 7x7) against the CPU checker, at the sizes where
its tiles end: channels that do not fill a chunk, output channels that do not fill a wavefront, a pixel more and a pixel less than
a tile, several images in one tile, rows of any width, strides and paddings, channels shared between blocks; and every compiled
variant of it against sums in 64 bits.

Bar: 1e-5 relative plus K * eps * max|x||w| for the order of summation (fp32 sums of K products); against 64 bits what the chains of
additions give.
"""
import numpy as np
import pytest

import support
import tannic_amd as ta
from tannic_amd import ops
from test_conv_plan import conv_plan

pytestmark = pytest.mark.gpu

# x shape, w shape, stride, padding
CASES = {
    "k1_channels_end_in_a_chunk": ((2, 20, 6, 10), (50, 20, 1, 1), (1, 1), (0, 0)),
    "k1_four_channels": ((3, 4, 8, 8), (33, 4, 1, 1), (1, 1), (0, 0)),
    "k1_odd_images": ((5, 36, 7, 7), (70, 36, 1, 1), (1, 1), (0, 0)),
    "k1_one_pixel_an_image": ((70, 16, 1, 1), (20, 16, 1, 1), (1, 1), (0, 0)),
    "k1_stride_2_odd_rows": ((3, 24, 15, 13), (40, 24, 1, 1), (2, 2), (0, 0)),
    "k1_rect_stride": ((2, 16, 9, 12), (17, 16, 1, 1), (3, 1), (0, 0)),
    "k1_pixel_past_a_tile": ((1, 32, 13, 5), (129, 32, 1, 1), (1, 1), (0, 0)),
    "k1_many_channels_few_pixels": ((1, 1024, 5, 5), (40, 1024, 1, 1), (1, 1), (0, 0)),
    "k1_wide_many_tiles": ((6, 64, 40, 40), (130, 64, 1, 1), (1, 1), (0, 0)),
    "k3_seven_wide": ((5, 16, 7, 7), (40, 16, 3, 3), (1, 1), (1, 1)),
    "k3_one_channel_group": ((2, 4, 9, 11), (33, 4, 3, 3), (1, 1), (1, 1)),
    "k3_fourteen_wide_stride_2": ((3, 8, 14, 14), (20, 8, 3, 3), (2, 2), (1, 1)),
    "k3_stride_2_odd": ((2, 12, 15, 29), (34, 12, 3, 3), (2, 2), (1, 1)),
    "k3_no_padding": ((2, 8, 12, 10), (16, 8, 3, 3), (1, 1), (0, 0)),
    "k3_wide_padding": ((2, 8, 6, 5), (16, 8, 3, 3), (1, 1), (2, 3)),
    "k3_padding_of_four": ((8, 16, 14, 14), (64, 16, 3, 3), (1, 1), (4, 4)),
    "k3_padding_of_five": ((16, 16, 7, 7), (32, 16, 3, 3), (1, 1), (5, 1)),
    "k3_padding_of_nine": ((3, 8, 5, 9), (33, 8, 3, 3), (1, 1), (9, 9)),
    "k3_rect_stride": ((2, 8, 13, 17), (16, 8, 3, 3), (2, 1), (1, 0)),
    "k3_stride_3": ((2, 8, 20, 20), (16, 8, 3, 3), (3, 3), (1, 1)),
    "k3_small_maps_many_images": ((40, 8, 3, 4), (16, 8, 3, 3), (1, 1), (1, 1)),
    "k3_shared_channels": ((1, 256, 8, 8), (48, 256, 3, 3), (1, 1), (1, 1)),
    "k3_wide_rows": ((1, 8, 5, 150), (64, 8, 3, 3), (1, 1), (1, 1)),
    "k3_many_tiles": ((4, 16, 56, 56), (64, 16, 3, 3), (1, 1), (1, 1)),
    "k7_stem": ((2, 3, 40, 40), (64, 3, 7, 7), (2, 2), (3, 3)),
    "k7_odd_rows": ((3, 3, 23, 29), (70, 3, 7, 7), (2, 2), (3, 3)),
    "k7_padding_of_eight": ((8, 3, 9, 9), (16, 3, 7, 7), (1, 1), (8, 8)),
    "k7_padding_of_nine": ((5, 2, 12, 10), (20, 2, 7, 7), (1, 1), (9, 9)),
    "k7_two_channels_stride_1": ((2, 2, 17, 19), (20, 2, 7, 7), (1, 1), (3, 3)),
    "k7_one_channel_no_padding": ((2, 1, 16, 40), (8, 1, 7, 7), (1, 1), (0, 0)),
}

# (planes too wide for the kernel's stages, and few results, run elsewhere)
ELSEWHERE = ("k3_fourteen_wide_stride_2", "k3_stride_3", "k3_shared_channels")

# Every compiled variant: side, U, PT, NL, WO, WIDE -> x shape, w shape, stride.  Output channels and pixels that end inside a tile, channels
# inside a group (1x1), tiles over several images, and enough groups for every part of the pipeline.
VARIANTS = {
    (1, 4, 2, 4, 2, 0): ((29, 56, 5, 10), (675, 56, 1, 1), 1),
    (1, 4, 2, 4, 2, 1): ((3, 56, 36, 30), (309, 56, 1, 1), 1),
    (1, 4, 2, 8, 1, 0): ((2, 68, 3, 3), (3, 68, 1, 1), 2),
    (1, 4, 2, 8, 1, 1): ((2, 52, 4, 3), (3, 52, 1, 1), 1),
    (1, 4, 4, 8, 2, 0): ((3, 52, 74, 77), (33, 52, 1, 1), 1),
    (1, 4, 4, 8, 2, 1): ((3, 52, 73, 76), (37, 52, 1, 1), 1),
    (1, 4, 6, 12, 2, 0): ((9, 52, 63, 61), (34, 52, 1, 1), 1),
    (1, 4, 6, 12, 2, 1): ((13, 52, 49, 52), (37, 52, 1, 1), 1),
    (1, 4, 7, 8, 4, 0): ((14, 52, 42, 45), (65, 52, 1, 1), 1),
    (1, 4, 7, 8, 4, 1): ((11, 52, 46, 50), (69, 52, 1, 1), 1),
    (1, 4, 7, 16, 2, 0): ((13, 52, 62, 63), (34, 52, 1, 1), 1),
    (1, 4, 7, 16, 2, 1): ((11, 56, 67, 68), (33, 56, 1, 1), 1),
    (1, 4, 13, 16, 4, 0): ((31, 132, 41, 39), (68, 132, 1, 1), 1),
    (1, 4, 13, 16, 4, 1): ((36, 132, 36, 35), (66, 132, 1, 1), 1),
    (1, 4, 13, 28, 2, 0): ((16, 132, 65, 69), (35, 132, 1, 1), 1),
    (1, 4, 13, 28, 2, 1): ((19, 136, 58, 60), (34, 136, 1, 1), 1),
    (1, 8, 2, 4, 4, 0): ((2, 116, 4, 3), (72, 116, 1, 1), 2),
    (1, 8, 2, 4, 4, 1): ((25, 116, 4, 3), (694, 116, 1, 1), 1),
    (1, 8, 4, 8, 4, 0): ((24, 116, 43, 44), (65, 116, 1, 1), 2),
    (1, 8, 4, 8, 4, 1): ((9, 120, 38, 34), (69, 120, 1, 1), 1),
    (1, 8, 6, 12, 4, 0): ((23, 116, 66, 60), (69, 116, 1, 1), 2),
    (1, 8, 6, 12, 4, 1): ((38, 120, 28, 22), (65, 120, 1, 1), 1),
    (1, 8, 8, 16, 4, 0): ((31, 104, 33, 30), (66, 104, 1, 1), 1),
    (1, 8, 8, 16, 4, 1): ((24, 100, 34, 38), (66, 100, 1, 1), 1),
    (3, 3, 2, 8, 1, 0): ((2, 16, 4, 3), (3, 16, 3, 3), 1),
    (3, 3, 2, 8, 2, 0): ((2, 16, 4, 3), (36, 16, 3, 3), 2),
    (3, 3, 2, 8, 4, 0): ((2, 24, 48, 53), (67, 24, 3, 3), 2),
    (3, 3, 4, 8, 2, 0): ((14, 16, 36, 33), (33, 16, 3, 3), 1),
    (3, 3, 4, 8, 4, 0): ((22, 16, 38, 39), (67, 16, 3, 3), 2),
    (3, 3, 4, 12, 2, 0): ((2, 20, 50, 51), (52, 20, 3, 3), 2),
    (3, 3, 5, 8, 2, 0): ((7, 16, 52, 46), (65, 16, 3, 3), 1),
    (3, 3, 5, 8, 4, 0): ((3, 16, 75, 76), (65, 16, 3, 3), 1),
    (3, 3, 7, 6, 4, 0): ((5, 16, 45, 42), (348, 16, 3, 3), 1),
    (3, 3, 7, 8, 2, 0): ((28, 16, 41, 41), (34, 16, 3, 3), 1),
    (3, 3, 7, 12, 4, 0): ((5, 16, 60, 60), (90, 16, 3, 3), 2),
    (3, 3, 7, 16, 2, 0): ((6, 16, 74, 74), (41, 16, 3, 3), 1),
    (3, 3, 10, 10, 2, 0): ((38, 16, 31, 30), (68, 16, 3, 3), 1),
    (3, 3, 10, 12, 4, 0): ((4, 16, 91, 95), (67, 16, 3, 3), 1),
    (3, 3, 13, 10, 4, 0): ((3, 20, 86, 88), (147, 20, 3, 3), 1),
    (3, 3, 13, 12, 2, 0): ((25, 16, 44, 40), (66, 16, 3, 3), 1),
    (7, 1, 2, 1, 1, 0): ((2, 1, 4, 3), (3, 1, 7, 7), 2),
    (7, 1, 2, 1, 2, 0): ((2, 1, 52, 52), (169, 1, 7, 7), 1),
    (7, 1, 4, 1, 2, 0): ((27, 1, 23, 27), (33, 1, 7, 7), 1),
    (7, 1, 7, 1, 2, 0): ((5, 1, 80, 85), (33, 1, 7, 7), 1),
}


def convolve64(x, w, stride, pad):
    """In float64, a product for every tap."""
    side = w.shape[2]
    padded = np.pad(x, ((0, 0), (0, 0), (pad, pad), (pad, pad))).astype(np.float64)
    ho, wo = ((n + 2 * pad - side) // stride + 1 for n in x.shape[2:])
    want = np.zeros((w.shape[0], x.shape[0], ho, wo))
    for i in range(side):
        for j in range(side):
            want += np.tensordot(w[:, :, i, j].astype(np.float64), padded[:, :, i:i + (ho - 1) * stride + 1:stride, j:j + (wo - 1) * stride + 1:stride], (1, 1))
    return want.transpose(1, 0, 2, 3)


def check_norm(got, want, additions, what):
    """n additions of values that grow with their root, each off by an error uniform within half a unit of the last place, 2^-24 / sqrt(3)
    of the partial sum at most: 2^-24 / sqrt(6) * sqrt(n) of the result's norm."""
    error = np.linalg.norm(got - want) / np.linalg.norm(want)
    assert error <= 2.0 ** -24 / 6 ** 0.5 * additions ** 0.5, (error, additions, what)


@pytest.mark.parametrize("biased", [False, True])
@pytest.mark.parametrize("name", list(CASES))
def test_conv2d_f32(name, biased, device):
    xs, ws, stride, padding = CASES[name]
    assert (conv_plan("float32", xs, ws, stride, padding)[0] == "f32") == (name not in ELSEWHERE)
    x, w = support.uniform(5, 1, xs, -1, 1), support.uniform(5, 2, ws, -1, 1)
    b = support.uniform(5, 3, (ws[0],), -1, 1)
    (hx, dx), (hw, dw), (hb, db) = (support.both(v, ta.float32, device) for v in (x, w, b))
    want = ops.convolve2d(hx, hw, hb if biased else None, stride, padding).numpy()
    got = ops.convolve2d(dx, dw, db if biased else None, stride, padding).numpy()
    terms = ws[1] * ws[2] * ws[3]
    support.assert_close(got, want, 1e-5, terms * np.finfo(np.float32).eps, name)


def test_values_beside_the_image_do_not_leak(device):
    """Infinities next to a view's rows and in the images around it stay out of the results: padding counts as zero, not as zero
    times what lies there."""
    x = np.full((3, 8, 10, 12), np.inf, np.float32)
    x[1, :, 2:8, 3:10] = support.uniform(7, 1, (8, 6, 7), -1, 1)
    w = support.uniform(7, 2, (16, 8, 3, 3), -1, 1)
    hx, dx = support.both(x, ta.float32, device)
    hw, dw = support.both(w, ta.float32, device)
    want = ops.convolve2d(hx[1:2, :, 2:8, 3:10], hw, None, 1, 1).numpy()
    got = ops.convolve2d(dx[1:2, :, 2:8, 3:10], dw, None, 1, 1).numpy()
    support.assert_close(got, want, 1e-5, 72 * np.finfo(np.float32).eps, "view")


# Problems that products with a finely shared K ran before this kernel took them, and some that those keep.  x shape, w shape, stride.
SUMS = {
    "k3_seven_wide": ((9, 512, 7, 7), (512, 512, 3, 3), 1),
    "k3_shared_by_many_blocks": ((3, 512, 7, 7), (512, 512, 3, 3), 1),
    "k3_one_block_each": ((4, 128, 37, 37), (128, 128, 3, 3), 1),
    "k3_stride": ((17, 256, 20, 20), (256, 256, 3, 3), 2),
    "k3_short": ((2, 64, 59, 59), (64, 64, 3, 3), 1),
    "k3_wide_tile_of_few_channels": ((17, 972, 34, 34), (36, 972, 3, 3), 1),
    "k3_few_results": ((2, 304, 35, 37), (3, 304, 3, 3), 1),
    "k1_odd_image": ((3, 512, 37, 37), (128, 512, 1, 1), 1),
    "k1_long": ((21, 1024, 8, 8), (512, 1024, 1, 1), 1),
    "k1_seven_wide": ((17, 512, 6, 6), (2048, 512, 1, 1), 1),
    "k1_stride": ((18, 512, 10, 10), (1024, 512, 1, 1), 2),
    "k1_stride_short": ((2, 128, 56, 56), (64, 128, 1, 1), 2),
    "k1_small_product": ((2, 512, 20, 20), (256, 512, 1, 1), 1),
}


@pytest.mark.parametrize("name", list(SUMS))
def test_sums_are_short_chains(name, device):
    """The error against 64 bits is what chains of 36 or 64 products, and the sums over groups and blocks, give."""
    xs, ws, stride = SUMS[name]
    pad, side = ws[2] // 2, ws[2]
    rng = np.random.default_rng(11)
    x, w = rng.standard_normal(xs, dtype=np.float32), rng.standard_normal(ws, dtype=np.float32)
    got = ops.convolve2d(ta.tensor(x, ta.float32, device), ta.tensor(w, ta.float32, device), None, stride, pad).numpy()
    kernel, plan = conv_plan("float32", xs, ws, (stride, stride), (pad, pad))
    k = ws[1] * side * side
    if kernel == "f32":
        additions = (36 if side == 3 else 64) + plan["chunks_per_split"] + plan["splits"]
    else:       # a wavefront's quarter of K, or a thread's 256th
        additions = k // 256 + 16 if side == 3 else k // 4 + 4
    check_norm(got, convolve64(x, w, stride, pad), additions, (kernel, plan))


@pytest.mark.parametrize("variant", list(VARIANTS), ids=lambda v: "-".join(map(str, v)))
def test_variant(variant, device):
    xs, ws, stride = VARIANTS[variant]
    pad, side = ws[2] // 2, ws[2]
    kernel, plan = conv_plan("float32", xs, ws, (stride, stride), (pad, pad))
    assert kernel == "f32" and tuple(plan[n] for n in ("side", "u", "pt", "nl", "wo", "wide")) == variant
    rng = np.random.default_rng(12)
    x, w, b = (rng.standard_normal(s, dtype=np.float32) for s in (xs, ws, ws[:1]))
    got = ops.convolve2d(*(ta.tensor(v, ta.float32, device) for v in (x, w, b)), stride, pad).numpy()
    # (the widest tiles and a 7x7 kernel add all products one after the other)
    additions = ws[1] * side * side + 1 if plan["pt"] >= 10 or side == 7 else (36 if side == 3 else 64) + plan["chunks_per_split"] + plan["splits"]
    check_norm(got, convolve64(x, w, stride, pad) + b[:, None, None], additions, plan)
