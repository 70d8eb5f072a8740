"""fp32 conv2d on the 16-bit matrix pipe (values as three bfloat16 values): which problems it takes and where its tiles' windows lie, asked
of the library without a GPU, and every compiled variant against sums in 64 bits."""
import ctypes as C
import os
import random
import re

import numpy as np
import pytest

import tannic_amd as ta
from tannic_amd import abi, ops
from test_conv_plan import descriptor, out_shape
from test_gpu_conv_f32 import convolve64

SOURCE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tannic_amd", "csrc", "conv2d_split.hip")
NAMES = ("side", "pt", "wo", "nl", "tile", "co_tiles", "splits", "chunks", "chunks_per_split", "plane", "hp", "wp")


def split_plan(x, w, stride, padding):
    out = (C.c_uint32 * 20)()
    args = [C.byref(descriptor("float32", s)) for s in (x, w, out_shape(x, w, stride, padding))]
    assert ta.library().conv2d_plan(*args, abi.SIZE2(*padding), abi.SIZE2(*stride), out) == abi.SUCCESS
    return dict(zip(NAMES, out[1:])) if out[0] == 3 else None


# side, PT, WO, NL -> x, w, stride: channels that end inside a chunk, output channels and pixels that end inside a tile
VARIANTS = {
    (1, 4, 2, 2): ((29, 340, 56, 59), (36, 340, 1, 1), 1),
    (1, 4, 4, 1): ((29, 376, 31, 34), (85, 376, 1, 1), 1),
    (1, 7, 4, 2): ((22, 276, 28, 29), (242, 276, 1, 1), 1),
    (3, 2, 2, 2): ((36, 220, 7, 8), (327, 220, 3, 3), 1),
    (3, 2, 2, 3): ((8, 532, 11, 12), (279, 532, 3, 3), 1),
    (3, 4, 2, 4): ((10, 500, 14, 17), (138, 500, 3, 3), 1),
    (3, 4, 2, 5): ((10, 284, 28, 31), (50, 284, 3, 3), 1),
    (3, 4, 4, 2): ((16, 360, 7, 10), (498, 360, 3, 3), 1),
    (3, 4, 4, 3): ((36, 148, 14, 14), (140, 148, 3, 3), 1),
    (3, 4, 4, 4): ((8, 144, 28, 31), (161, 144, 3, 3), 1),
    (3, 7, 4, 4): ((37, 316, 7, 10), (213, 316, 3, 3), 1),
    (3, 7, 4, 5): ((3, 328, 39, 39), (106, 328, 3, 3), 1),
}
# strides, padding beyond the kernel, long and short K, few channels out
OTHERS = {
    "k1_stride": ((16, 300, 57, 65), (330, 300, 1, 1), (2, 2), (0, 0)),
    "k1_rect_stride": ((30, 200, 61, 68), (260, 200, 1, 1), (3, 1), (0, 0)),
    "k1_long": ((32, 2048, 7, 7), (512, 2048, 1, 1), (1, 1), (0, 0)),
    "k1_odd_image": ((32, 260, 17, 17), (512, 260, 1, 1), (1, 1), (0, 0)),
    "k3_no_padding": ((32, 128, 20, 19), (128, 128, 3, 3), (1, 1), (0, 0)),
    "k3_wide_padding": ((32, 128, 11, 10), (128, 128, 3, 3), (1, 1), (5, 4)),
    "k3_rect_stride": ((27, 260, 22, 8), (199, 260, 3, 3), (1, 2), (1, 1)),
    "k3_few_channels": ((21, 68, 27, 24), (456, 68, 3, 3), (1, 1), (1, 1)),
}


def test_variants_are_all_reached():
    compiled = {tuple(map(int, v)) for v in re.findall(r"\bF\((\d), (\d), (\d), (\d)\)", open(SOURCE).read())}
    assert len(compiled) >= 12 and compiled == set(VARIANTS)


@pytest.mark.parametrize("variant", list(VARIANTS), ids=lambda v: "-".join(map(str, v)))
def test_variant_is_the_plan_of_its_shape(variant):
    x, w, stride = VARIANTS[variant]
    q = split_plan(x, w, (stride, stride), (w[2] // 2,) * 2)
    assert q is not None and tuple(q[n] for n in NAMES[:4]) == variant


def test_windows_lie_in_their_planes():
    """Every tap of every pixel of random problems: the place in the tile's plane holds the signal's value there, or a zero of the padding."""
    rng, taken = random.Random(3), 0
    for _ in range(3000):
        channels, padding = rng.randrange(32, 200), (rng.randrange(0, 6), rng.randrange(0, 6))
        x = (rng.randrange(1, 24), channels, rng.randrange(3, 40), rng.randrange(3, 40))
        stride = (rng.randrange(1, 4), rng.randrange(1, 4)) if rng.random() < 0.4 else (1, 1)
        w = (rng.randrange(32, 400), channels, 3, 3)
        q = split_plan(x, w, stride, padding)
        if q is None:
            continue
        taken += 1
        ho, wo = out_shape(x, w, stride, padding)[2:]
        pixel = np.arange(x[0] * ho * wo, dtype=np.int64)
        first = pixel // q["tile"] * q["tile"]
        n, oh, ow = pixel // (ho * wo), pixel // wo % ho, pixel % wo
        n0, oh0 = first // (ho * wo), first // wo % ho
        e = (((n - n0) * q["hp"] + (oh - oh0) * stride[0]) * q["wp"] + ow * stride[1])[:, None, None] + np.arange(3)[:, None] * q["wp"] + np.arange(3)
        assert e.min() >= 0 and e.max() < q["plane"] <= 64 * q["nl"], (x, w, stride, padding, q)
        line = oh0[:, None, None] * stride[0] + e // q["wp"]
        image, ih, iw = n0[:, None, None] + line // q["hp"], line % q["hp"] - padding[0], e % q["wp"] - padding[1]
        inside = (image < x[0]) & (ih >= 0) & (ih < x[2]) & (iw >= 0) & (iw < x[3])
        want_h, want_w = (oh * stride[0] - padding[0])[:, None, None] + np.arange(3)[:, None], (ow * stride[1] - padding[1])[:, None, None] + np.arange(3)
        want = (want_h >= 0) & (want_h < x[2]) & (want_w >= 0) & (want_w < x[3])
        assert np.array_equal(inside, want), (x, w, stride, padding, q)
        assert ((image == n[:, None, None]) & (ih == want_h) & (iw == want_w))[want].all(), (x, w, stride, padding, q)
    assert taken >= 60, taken


# channels in that are rounded up to whole chunks, and the output channels from which their three parts take more bytes than 32 bits count
@pytest.mark.parametrize("x,beyond,neighbour", [((1, 68, 30, 30), 828497, True), ((1, 44, 18, 18), 1242753, True), ((22, 1774052, 7, 7), 33, False)], ids=["68", "44", "long"])
def test_parts_of_the_weights_are_counted_in_32_bits(x, beyond, neighbour):
    """(Below, the problem runs here; the longest K does not for another reason, and all go on to the kernel of the fp32 pipe.)"""
    def parts(o):
        return ((o + 15) // 16 * ((x[1] + 31) // 32) * 9 + 2) * 3 * 1024
    assert parts(beyond - 1) < 2 ** 32 <= parts(beyond)
    assert (split_plan(x, (beyond - 1, x[1], 3, 3), (1, 1), (1, 1)) is not None) == neighbour
    w = (beyond, x[1], 3, 3)
    assert split_plan(x, w, (1, 1), (1, 1)) is None
    out = (C.c_uint32 * 20)()
    args = [C.byref(descriptor("float32", s)) for s in (x, w, out_shape(x, w, (1, 1), (1, 1)))]
    assert ta.library().conv2d_plan(*args, abi.SIZE2(1, 1), abi.SIZE2(1, 1), out) == abi.SUCCESS and out[0] == 1


def run(xs, ws, stride, padding, device, change=lambda x, w: None):
    rng = np.random.default_rng(21)
    x, w, b = (rng.standard_normal(s, dtype=np.float32) for s in (xs, ws, ws[:1]))
    change(x, w)
    q = split_plan(xs, ws, stride, padding)
    assert q is not None
    return x, w, b, q, ops.convolve2d(*(ta.tensor(v, ta.float32, device) for v in (x, w, b)), stride, padding).numpy()


def reference(x, w, b, stride, padding):
    import torch
    y = torch.nn.functional.conv2d(*(torch.from_numpy(v.astype(np.float64)) for v in (x, w, b)), stride, padding)
    return y.numpy()


def check(got, want, q, what):
    """Roundings that matter, each uniform within half a unit of the last place of a partial sum that grows with its root: one behind
    every 32 products, two MFMAs' worth inside (chains of nine, or of sixteen and the last), the sums over chains and blocks, the three sets."""
    chain = 9 if q["side"] == 3 else 16
    additions = 4 * chain + q["chunks_per_split"] + q["splits"] + 3
    error = np.linalg.norm(got - want) / np.linalg.norm(want)
    assert error <= 2.0 ** -24 / 6 ** 0.5 * additions ** 0.5, (error, additions, what)


@pytest.mark.gpu
@pytest.mark.parametrize("variant", list(VARIANTS), ids=lambda v: "-".join(map(str, v)))
def test_variant(variant, device):
    xs, ws, stride = VARIANTS[variant]
    padding = (ws[2] // 2,) * 2
    x, w, b, q, got = run(xs, ws, (stride, stride), padding, device)
    check(got, convolve64(x, w, stride, padding[0]) + b[:, None, None], q, variant)


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(OTHERS))
def test_other_shapes(name, device):
    xs, ws, stride, padding = OTHERS[name]
    x, w, b, q, got = run(xs, ws, stride, padding, device)
    check(got, reference(x, w, b, stride, padding), q, name)


def infinities_in_x(x, w):
    x[0, 3, 5, 5], x[2, 7, 0, 1], x[3, 40, 9, 9], x[3, 41, 9, 9] = np.inf, np.nan, np.inf, -np.inf


def infinities_in_w(x, w):
    w[5, 7], w[70, 33, 0, 0] = np.inf, np.nan


def largest(x, w):
    x[1, 9, 4, 4], x[2, 50, 6, 6] = 3.4028235e38, -3.4e38
    w *= 1e-3


def smallest(x, w):
    x *= 1e-36


def smallest_weights(x, w):
    w *= 1e-36


def beside_others(x, w):
    x[::2] *= 1e-34     # tiny images between others


def large_results(x, w):
    x[1] *= 1e15
    w *= 1e12


def almost_infinite(x, w):
    x[0, 0, 5, 5] = w[:, 0] = 1.999 * 2.0 ** 63     # (their product is finite, that of the nearest bfloat16 values is not)


SPECIAL = [infinities_in_x, infinities_in_w, largest, smallest, smallest_weights, beside_others, large_results, almost_infinite]


@pytest.mark.gpu
@pytest.mark.parametrize("side", [1, 3])
@pytest.mark.parametrize("change", SPECIAL, ids=lambda f: f.__name__)
def test_values_without_three_parts(change, side, device):
    """Infinities and NaNs where fp32 has them and nowhere else; values at the ends of the range as exact as others."""
    xs, ws = ((16, 256, 24, 24), (512, 256, 1, 1)) if side == 1 else ((16, 128, 20, 20), (256, 128, 3, 3))
    x, w, b, q, got = run(xs, ws, (1, 1), (0, 0), device, change)
    b *= 0          # (compared without a bias: it would hide the smallest results)
    got = ops.convolve2d(*(ta.tensor(v, ta.float32, device) for v in (x, w, b)), (1, 1), (0, 0)).numpy()
    want = reference(x, w, b, (1, 1), (0, 0))
    with np.errstate(over="ignore"):
        rounded = want.astype(np.float32)
    assert np.array_equal(np.isnan(got), np.isnan(rounded)) and np.array_equal(np.isinf(got), np.isinf(rounded))
    assert np.array_equal(got[np.isinf(got)], rounded[np.isinf(rounded)])
    # image by image, as the magnitudes differ
    for i in range(xs[0]):
        finite = np.isfinite(rounded[i])
        error = np.linalg.norm(got[i][finite] - want[i][finite]) / np.linalg.norm(want[i][finite])
        assert error < 5e-7, (i, error)


@pytest.mark.gpu
@pytest.mark.parametrize("side", [1, 3])
@pytest.mark.parametrize("magnitude", [1e-33, 1e-36, 1e-38, 1e-40])
def test_small_values_beside_ordinary_ones(magnitude, side, device):
    """Output channels of small weights, and pixels of small values, in the same tiles as others: as exact as those, down to where fp32 ends
    (a partial sum, the sum of all and the bias's are rounded to whole 2^-149 there)."""
    xs, ws = ((16, 256, 24, 24), (512, 256, 1, 1)) if side == 1 else ((16, 128, 20, 20), (256, 128, 3, 3))
    rng = np.random.default_rng(22)
    q = split_plan(xs, ws, (1, 1), (0, 0))

    def error(got, want):
        return np.linalg.norm(got - want) - (q["splits"] + 2) * 2.0 ** -150 * want.size ** 0.5, np.linalg.norm(want)

    def both(x, w):
        return ops.convolve2d(ta.tensor(x, ta.float32, device), ta.tensor(w, ta.float32, device)).numpy(), reference(x, w, np.zeros(ws[0], np.float32), (1, 1), (0, 0))
    x, w = (rng.standard_normal(s, dtype=np.float32) for s in (xs, ws))
    small = w.copy()
    small[::7] *= np.float32(magnitude)
    got, want = both(x, small)
    for channel in range(ws[0]):
        off, norm = error(got[:, channel], want[:, channel])
        assert off < 5e-7 * norm, ("channel", channel, off / norm)
    x[:, :, 4:11, 4:11] *= np.float32(magnitude)
    got, want = both(x, w)
    for i in range(xs[0]):
        off, norm = error(got[i, :, 4:12 - side, 4:12 - side], want[i, :, 4:12 - side, 4:12 - side])
        assert off < 5e-7 * norm, ("pixels of image", i, off / norm)
