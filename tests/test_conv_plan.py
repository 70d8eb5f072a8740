"""Which kernel a convolution runs and where its tiles' windows lie, asked of the library without a GPU (``tannic_hip_conv2d_plan``).

The fp32 kernel keeps a channel's plane as the rows its tile touches, with the padding between two images shared by both; a
pixel's window is read at one offset from the plane's start.  Here that arithmetic is followed for every pixel of a problem: each
value of a window has to lie in the plane and to be the signal's value there, or a zero of the padding."""
import ctypes as C
import random

import numpy as np
import pytest

import tannic_amd as ta
from tannic_amd import abi
from tannic_amd.tensor import contiguous_strides

_CODES = {"float16": abi.FLOAT16, "bfloat16": abi.BFLOAT16, "float32": abi.FLOAT32}


def descriptor(dtype, shape):
    """A contiguous tensor of that shape at an address that is never read."""
    t = abi.tensor_t()
    t.address, t.rank, t.dtype = 0x10000, len(shape), _CODES[dtype]
    t.shape.sizes[:len(shape)] = shape
    t.strides.sizes[:len(shape)] = contiguous_strides(shape)
    t.size = int(np.prod(shape))
    return t


def out_shape(x, w, stride, padding):
    return (x[0], w[0]) + tuple((x[2 + d] + 2 * padding[d] - w[2 + d]) // stride[d] + 1 for d in range(2))


def conv_plan(dtype, x, w, stride, padding):
    out = (C.c_uint32 * 20)()
    args = [C.byref(descriptor(dtype, s)) for s in (x, w, out_shape(x, w, stride, padding))]
    assert ta.library().conv2d_plan(*args, abi.SIZE2(*padding), abi.SIZE2(*stride), out) == abi.SUCCESS
    if out[0] == 1:
        names = ("side", "u", "pt", "nl", "resident", "wo", "wide", "tile", "co_tiles", "splits", "chunks", "chunks_per_split", "pitch", "plane", "hp", "wp")
        return "f32", dict(zip(names, out[1:]))
    if out[0] == 2:
        return "few", dict(zip(("side", "mo", "np", "waves", "blocks"), out[1:]))
    return None, {}


def check_windows(x, w, stride, padding):
    """True where the fp32 kernel takes the problem (after every window was found to be right)."""
    kernel, q = conv_plan("float32", x, w, stride, padding)
    if kernel != "f32":
        return False
    (n_images, _, height, width), side = x, w[2]
    ho, wo = out_shape(x, w, stride, padding)[2:]
    pixel = np.arange(n_images * ho * wo, dtype=np.int64)
    first = pixel // q["tile"] * q["tile"]
    n, oh, ow = pixel // (ho * wo), pixel // wo % ho, pixel % wo
    n0, oh0 = first // (ho * wo), first // wo % ho
    start = ((n - n0) * q["hp"] + (oh - oh0) * stride[0]) * q["wp"] + ow * stride[1]
    tap = np.arange(side)
    e = start[:, None, None] + tap[:, None] * q["wp"] + tap
    what = (x, w, stride, padding, q)
    assert e.min() >= 0 and e.max() < q["plane"], (what, int(e.min()), int(e.max()))
    assert q["plane"] <= (q["pitch"] if q["resident"] else 64 * q["nl"]), what
    # what the load of element e brings ...
    line = oh0[:, None, None] * stride[0] + e // q["wp"]
    image, ih, iw = n0[:, None, None] + line // q["hp"], line % q["hp"] - padding[0], e % q["wp"] - padding[1]
    inside = (image < n_images) & (ih >= 0) & (ih < height) & (iw >= 0) & (iw < width)
    # ... and what the window needs
    want_h, want_w = (oh * stride[0] - padding[0])[:, None, None] + tap[:, None], (ow * stride[1] - padding[1])[:, None, None] + tap
    want = (want_h >= 0) & (want_h < height) & (want_w >= 0) & (want_w < width)
    assert np.array_equal(inside, want), what
    same = (image == n[:, None, None]) & (ih == want_h) & (iw == want_w)
    assert same[want].all(), what
    return True


# padding beyond the kernel's height over several images: the next image's first window begins above this one's last
WIDE_PADDING = [((8, 16, 14, 14), (64, 16, 3, 3), 4), ((4, 8, 8, 8), (40, 8, 3, 3), 4), ((16, 16, 7, 7), (32, 16, 3, 3), 5), ((3, 8, 5, 9), (33, 8, 3, 3), 9),
                ((8, 3, 9, 9), (16, 3, 7, 7), 8), ((5, 2, 12, 10), (20, 2, 7, 7), 9)]


@pytest.mark.parametrize("x,w,padding", WIDE_PADDING, ids=lambda v: str(v).replace(" ", ""))
def test_windows_under_wide_padding(x, w, padding):
    check_windows(x, w, (1, 1), (padding, padding))


@pytest.mark.parametrize("side,problems", [(3, 400), (7, 200)])
def test_windows_lie_in_their_planes(side, problems):
    rng, taken = random.Random(side), 0
    for _ in range(problems):
        channels = rng.choice((1, 2, 3, 4)) if side == 7 else 4 * rng.randrange(1, 20)
        images, padding = rng.randrange(1, 20), (rng.randrange(0, 3 * side), rng.randrange(0, 3 * side))
        height, width = rng.randrange(max(1, side - 2 * padding[0]), 40), rng.randrange(max(1, side - 2 * padding[1]), 40)
        stride = (rng.randrange(1, 5), rng.randrange(1, 5)) if rng.random() < 0.5 else (1, 1)
        taken += check_windows((images, channels, height, width), (rng.randrange(1, 200), channels, side, side), stride, padding)
    assert taken >= problems // 4, taken


# fp32 problems that the kernels before do in less time: x, w, stride, padding
FASTER_ELSEWHERE = {
    "wide_rows_under_a_stem": ((8, 3, 294, 294), (64, 3, 7, 7), 2, 3),
    "few_channels_wide_rows": ((9, 2, 348, 347), (2, 2, 7, 7), 2, 0),
    "writing_bound": ((29, 20, 122, 122), (991, 20, 1, 1), 1, 0),
    "small_tiles_short_k": ((22, 8, 72, 72), (442, 8, 3, 3), 2, 1),
    "small_tiles_spare_channels": ((6, 324, 74, 76), (192, 324, 3, 3), 2, 1),
    "small_product": ((2, 512, 20, 20), (256, 512, 1, 1), 1, 0),
    "small_product_of_samples": ((2, 128, 56, 56), (64, 128, 1, 1), 2, 0),
}


@pytest.mark.parametrize("name", list(FASTER_ELSEWHERE))
def test_fp32_problems_left_to_other_kernels(name):
    x, w, stride, padding = FASTER_ELSEWHERE[name]
    kernel, plan = conv_plan("float32", x, w, (stride, stride), (padding, padding))
    assert kernel != "f32", plan


@pytest.mark.parametrize("x,w", [((4, 60, 123, 124), (187, 60, 1, 1)), ((18, 64, 64, 64), (256, 64, 1, 1))], ids=str)
def test_short_k_takes_no_tile_that_fills_a_compute_unit(x, w):
    kernel, plan = conv_plan("float32", x, w, (1, 1), (0, 0))
    assert kernel == "f32" and plan["pt"] < 10, plan


# 16-bit problems around the lines up to which the kernel over few output pixels is taken: x, w, stride, padding, taken
FEW_PIXELS = {
    "one_output_channel_large_maps": ((12, 512, 65, 112), (1, 512, 3, 3), 1, 1, False),
    "one_output_channel_large_image": ((1, 32, 912, 912), (1, 32, 3, 3), 1, 1, False),
    "one_output_channel_few_pixels": ((1, 512, 14, 14), (1, 512, 3, 3), 1, 1, True),
    "ragged_1x1_of_few_channels": ((32, 64, 37, 37), (64, 64, 1, 1), 1, 0, False),
    "ragged_1x1_below_the_line": ((16, 64, 37, 37), (64, 64, 1, 1), 1, 0, True),
    "ragged_1x1_of_many_channels": ((7, 1024, 14, 14), (256, 1024, 1, 1), 1, 0, False),
    "ragged_1x1_of_many_channels_below": ((4, 1024, 14, 10), (512, 1024, 1, 1), 1, 0, True),
    "stride_of_many_channels": ((27, 1024, 5, 7), (100, 1024, 3, 3), 2, 1, False),
}


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("name", list(FEW_PIXELS))
def test_few_pixels(name, dtype):
    x, w, stride, padding, taken = FEW_PIXELS[name]
    kernel, plan = conv_plan(dtype, x, w, (stride, stride), (padding, padding))
    assert (kernel == "few") == taken, plan


@pytest.mark.parametrize("outputs", [1, 15, 16])
@pytest.mark.parametrize("stride", [1, 2])
def test_sixteen_output_channels_are_one_tile(outputs, stride):
    for side in (1, 3):
        kernel, plan = conv_plan("float16", (1, 64, 90 * stride, 91 * stride), (outputs, 64, side, side), (stride, stride), (side // 2, side // 2))
        assert kernel == "few" and plan["mo"] == 1, plan
