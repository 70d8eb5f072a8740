"""16-bit 3x3 conv2d over the flattened batch: which problems it takes and where its tiles' windows lie, asked of the library without a GPU,
and every compiled variant against sums in 64 bits."""
import ctypes as C
import os
import random
import re

import numpy as np
import pytest

import tannic_amd as ta
from tannic_amd import abi, ops
from test_conv_plan import descriptor, out_shape

SOURCE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tannic_amd", "csrc", "conv2d_batch3.hip")
NAMES = ("side", "pt", "wo", "nl", "tile", "co_tiles", "splits", "chunks", "chunks_per_split", "plane", "hp", "wp")


def batch3_plan(x, w, stride, padding, dtype="float16"):
    out = (C.c_uint32 * 20)()
    args = [C.byref(descriptor(dtype, s)) for s in (x, w, out_shape(x, w, stride, padding))]
    assert ta.library().conv2d_plan(*args, abi.SIZE2(*padding), abi.SIZE2(*stride), out) == abi.SUCCESS
    return dict(zip(NAMES, out[1:])) if out[0] == 4 else None


# PT, WO, NL -> x, w: output channels and pixels that end inside a tile, channels that end inside a chunk, channels shared between blocks
VARIANTS = {
    (2, 2, 2): ((37, 443, 6, 6), (113, 443, 3, 3)),
    (2, 2, 3): ((4, 512, 17, 15), (128, 512, 3, 3)),
    (4, 2, 4): ((16, 96, 27, 27), (64, 96, 3, 3)),
    (4, 2, 5): ((23, 330, 4, 35), (64, 330, 3, 3)),
    (4, 2, 6): ((26, 192, 4, 53), (64, 192, 3, 3)),
    (4, 4, 2): ((18, 75, 59, 4), (256, 75, 3, 3)),
    (4, 4, 3): ((25, 96, 19, 19), (82, 96, 3, 3)),
    (4, 4, 4): ((31, 128, 8, 33), (64, 128, 3, 3)),
    (4, 4, 5): ((37, 96, 6, 49), (64, 96, 3, 3)),
    (4, 4, 7): ((3, 103, 14, 57), (113, 103, 3, 3)),
    (7, 4, 3): ((16, 73, 27, 11), (512, 73, 3, 3)),
    (7, 4, 4): ((18, 85, 54, 25), (71, 85, 3, 3)),
    (7, 4, 5): ((10, 67, 47, 36), (111, 67, 3, 3)),
}
# x, w, stride, padding: strides, padding beyond the kernel and none, one block for all channels of an odd image
OTHERS = {
    "stride": ((18, 256, 30, 29), (256, 256, 3, 3), (2, 2), (1, 1)),
    "rect_stride": ((30, 130, 24, 11), (200, 130, 3, 3), (2, 1), (1, 1)),
    "no_padding": ((12, 160, 21, 20), (130, 160, 3, 3), (1, 1), (0, 0)),
    "wide_padding": ((16, 128, 11, 10), (128, 128, 3, 3), (1, 1), (5, 4)),
    "long": ((6, 1024, 14, 15), (256, 1024, 3, 3), (1, 1), (1, 1)),
}


def test_variants_are_all_reached():
    compiled = {tuple(map(int, v)) for v in re.findall(r"\bF\((\d), (\d), (\d)\)", open(SOURCE).read())}
    assert len(compiled) == 13 and compiled == set(VARIANTS)


@pytest.mark.parametrize("variant", list(VARIANTS), ids=lambda v: "-".join(map(str, v)))
def test_variant_is_the_plan_of_its_shape(variant):
    q = batch3_plan(*VARIANTS[variant], (1, 1), (1, 1))
    assert q is not None and tuple(q[n] for n in NAMES[1:4]) == variant


# what other kernels do in less time, and beside each a problem that stays
RULES = {
    "few_pixels": (((1, 320, 20, 24), (512, 320, 3, 3), 1), ((4, 136, 13, 10), (448, 136, 3, 3), 1)),
    "few_pixels_ragged": (((2, 272, 14, 15), (384, 272, 3, 3), 1), ((1, 278, 22, 24), (512, 278, 3, 3), 1)),
    "few_pixels_more": (((4, 200, 12, 9), (560, 200, 3, 3), 1), ((2, 448, 19, 16), (192, 448, 3, 3), 1)),
    "one_round_there": (((19, 192, 22, 20), (512, 192, 3, 3), 1), ((25, 256, 20, 20), (278, 256, 3, 3), 1)),
    "one_round_there_two_blocks_a_unit": (((15, 128, 22, 20), (768, 128, 3, 3), 1), ((12, 128, 24, 25), (816, 128, 3, 3), 1)),
    "two_rounds_there": (((7, 576, 28, 28), (816, 576, 3, 3), 1), ((20, 192, 24, 22), (691, 192, 3, 3), 1)),
    "stride": (((42, 480, 45, 46), (16, 480, 3, 3), 2), ((42, 480, 45, 47), (16, 480, 3, 3), 2)),
    "stride_whole_rows": (((16, 160, 45, 48), (32, 160, 3, 3), 2), ((30, 416, 30, 32), (128, 416, 3, 3), 2)),
    "stride_three_chunks": (((49, 96, 32, 30), (28, 96, 3, 3), 2), ((49, 96, 32, 31), (28, 96, 3, 3), 2)),
    "stride_four_chunks": (((27, 128, 23, 20), (512, 128, 3, 3), 2), ((52, 128, 20, 22), (725, 128, 3, 3), 2)),
    "stride_few_chunks_whole_rows": (((16, 128, 35, 32), (188, 128, 3, 3), 2), ((21, 192, 29, 32), (128, 192, 3, 3), 2)),
    "stride_two_rounds": (((19, 320, 24, 27), (693, 320, 3, 3), 2), ((19, 384, 26, 26), (560, 384, 3, 3), 2)),
    "stride_two_rounds_more_pixels": (((19, 408, 27, 25), (576, 408, 3, 3), 2), ((34, 352, 21, 22), (768, 352, 3, 3), 2)),
}


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("name", list(RULES))
def test_rules(name, dtype):
    (x, w, stride), (x2, w2, stride2) = RULES[name]
    assert batch3_plan(x, w, (stride, stride), (1, 1), dtype) is None
    assert batch3_plan(x2, w2, (stride2, stride2), (1, 1), dtype) is not None


def test_ordered_weights_are_counted_in_32_bits():
    """One output channel takes the room of sixteen: a signal of one value seen as any number of channels and images."""
    def taken(channels):
        x, w, y = (descriptor("float16", s) for s in ((200000, channels, 11, 11), (1, channels, 3, 3), (200000, 1, 11, 11)))
        for d in range(3):
            x.strides.sizes[d] = 0
        out = (C.c_uint32 * 20)()
        assert ta.library().conv2d_plan(*(C.byref(t) for t in (x, w, y)), abi.SIZE2(1, 1), abi.SIZE2(1, 1), out) == abi.SUCCESS
        return out[0] == 4
    fits = ((2 ** 32 - 1) // (9 * 1024) - 1) * 32
    assert taken(fits) and not taken(fits + 1)


def test_windows_lie_in_their_planes():
    """Every tap of every pixel of random problems: the place in the tile's plane holds the signal's value there, or a zero of the padding."""
    rng, taken = random.Random(5), 0
    for _ in range(6000):
        channels, padding = rng.randrange(64, 300), (rng.randrange(0, 6), rng.randrange(0, 6)) if rng.random() < 0.5 else (1, 1)
        x = (rng.randrange(1, 24), channels, rng.randrange(3, 30), rng.randrange(3, 30))
        stride = (rng.randrange(1, 4), rng.randrange(1, 4)) if rng.random() < 0.4 else (1, 1)
        w = (rng.randrange(64, 500), channels, 3, 3)
        q = batch3_plan(x, w, stride, padding, rng.choice(["float16", "bfloat16"]))
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


DTYPES = {"float16": (ta.float16, 2.0 ** -11), "bfloat16": (ta.bfloat16, 2.0 ** -8)}


def check(xs, ws, stride, padding, dtype, device):
    """One rounding of the result, and K * eps of fp32 times the sum of the products' magnitudes."""
    import torch
    kind, eps = DTYPES[dtype]
    assert batch3_plan(xs, ws, stride, padding, dtype) is not None
    rng = np.random.default_rng(31)
    x, w, b = (ta.tensor(rng.standard_normal(s, dtype=np.float32), kind, device) for s in (xs, ws, ws[:1]))
    got = ops.convolve2d(x, w, b, stride, padding).numpy().astype(np.float64)
    x, w, b = (torch.from_numpy(t.numpy().astype(np.float64)) for t in (x, w, b))
    want = torch.nn.functional.conv2d(x, w, b, stride, padding).numpy()
    size = torch.nn.functional.conv2d(x.abs(), w.abs(), b.abs(), stride, padding).numpy()
    off = np.abs(got - want) / (eps * np.abs(want) + ws[1] * 9 * 2.0 ** -24 * size)
    assert off.max() <= 1.0, (float(off.max()), xs, ws)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("variant", list(VARIANTS), ids=lambda v: "-".join(map(str, v)))
def test_variant(variant, dtype, device):
    check(*VARIANTS[variant], (1, 1), (1, 1), dtype, device)


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(OTHERS))
def test_other_shapes(name, device):
    check(*OTHERS[name], "float16" if len(name) % 2 else "bfloat16", device)


@pytest.mark.gpu
@pytest.mark.parametrize("skip", [0, 1])
def test_part_of_a_tensor(skip, device):
    """Channels and rows out of a larger tensor, from any element on; what lies beside is infinite."""
    import torch
    n, c, h, w, o = 12, 100, 20, 21, 130
    rng = np.random.default_rng(9)
    whole = np.full((n + 1, c + 3, h + 2, w), np.inf, np.float32)
    whole[:n, skip:c + skip, skip:h + skip, :] = rng.standard_normal((n, c, h, w))
    x = ta.tensor(whole, ta.float16, device)[0:n, skip:c + skip, skip:h + skip, :]
    k = ta.tensor(rng.standard_normal((o, c, 3, 3), dtype=np.float32), ta.float16, device)
    got = ops.convolve2d(x, k, None, 1, 1).numpy().astype(np.float64)
    inside = torch.from_numpy(whole[:n, skip:c + skip, skip:h + skip].astype(np.float16).astype(np.float64))
    kernel = torch.from_numpy(k.numpy().astype(np.float64))
    want = torch.nn.functional.conv2d(inside, kernel, None, 1, 1).numpy()
    size = torch.nn.functional.conv2d(inside.abs(), kernel.abs(), None, 1, 1).numpy()
    off = np.abs(got - want) / (2.0 ** -11 * np.abs(want) + c * 9 * 2.0 ** -24 * size)
    assert off.max() <= 1.0, float(off.max())


@pytest.mark.gpu
def test_infinities_stay_where_they_are(device):
    """An infinity or a NaN of the signal is in the results whose windows hold it, and in no other image's or tile's."""
    xs, ws = (25, 96, 19, 19), (82, 96, 3, 3)
    rng = np.random.default_rng(10)
    x, w = rng.standard_normal(xs, dtype=np.float32), rng.standard_normal(ws, dtype=np.float32)
    x[0, 3, 18, 18], x[3, 95, 0, 0], x[24, 0, 18, 5] = np.inf, np.nan, -np.inf
    got = ops.convolve2d(ta.tensor(x, ta.float16, device), ta.tensor(w, ta.float16, device), None, 1, 1).numpy()
    touched = np.zeros((xs[0],) + xs[2:], bool)
    touched[0, 17:, 17:] = touched[3, :2, :2] = touched[24, 17:, 4:7] = True
    assert np.array_equal(np.isfinite(got), np.broadcast_to(~touched[:, None], got.shape))
