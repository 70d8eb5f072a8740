"""16-bit 1x1 convolutions whose tiles run over the images of a batch and read them where they lie, against sums in 64 bits: images that
are not whole pieces of eight pixels, tiles over several images, every tile height, one step of channels and many.

Bar: one rounding of the result, and K * eps of fp32 times the sum of the products' magnitudes.
"""
import numpy as np
import pytest

import tannic_amd as ta
from tannic_amd import ops

pytestmark = pytest.mark.gpu

DTYPES = {"float16": (ta.float16, 2.0 ** -11), "bfloat16": (ta.bfloat16, 2.0 ** -8)}

# images, channels, height, width, channels out
SHAPES = {
    "many_images_eight_pixels": (2900, 64, 2, 4, 70),
    "many_images_ten_pixels": (1200, 128, 2, 5, 130),
    "many_images_twelve_pixels": (1200, 128, 3, 4, 66),
    "many_images_fourteen_pixels": (999, 64, 2, 7, 200),
    "many_images_forty_two_pixels": (230, 320, 6, 7, 100),
    "many_images_two_wide": (160, 512, 26, 2, 70),
    "many_images_fourteen_wide": (60, 256, 14, 14, 200),
    "many_images_whole_pieces": (35, 192, 16, 16, 129),
    "many_tiles": (24, 128, 28, 28, 300),
    "long_k": (28, 1024, 14, 14, 500),
    "many_images_few_channels_out": (150, 256, 18, 18, 24),
    "one_larger_image": (1, 512, 60, 62, 260),
}
# the same where so few pixels have a kernel of their own (conv2d_few.hip)
FEW_PIXELS = {
    "eight_pixels": (40, 64, 2, 4, 70),
    "ten_pixels": (90, 64, 2, 5, 130),
    "twelve_pixels": (33, 128, 3, 4, 66),
    "forty_two_pixels": (17, 320, 6, 7, 100),
    "fourteen_wide": (9, 256, 14, 14, 200),
    "whole_pieces": (5, 192, 16, 16, 129),
    "few_channels_out": (11, 256, 18, 18, 24),
    "one_image": (1, 512, 30, 31, 260),
}


def values(t):
    return t.numpy().astype(np.float64)


def check(x, w, b, got, eps):
    x, w, b = values(x), values(w), values(b)
    n, c, h, wd = x.shape
    flat, kernel = x.reshape(n, c, h * wd), w[:, :, 0, 0]
    want = kernel @ flat + b[:, None]
    bound = eps * np.abs(want) + c * 2.0 ** -24 * (np.abs(kernel) @ np.abs(flat) + np.abs(b)[:, None])
    off = np.abs(got.reshape(want.shape) - want)
    assert (off <= bound).all(), float((off / bound).max())


@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("name", [*SHAPES, *FEW_PIXELS])
def test_columns_in_groups(name, dtype, device):
    n, c, h, wd, o = {**SHAPES, **FEW_PIXELS}[name]
    kind, eps = DTYPES[dtype]
    rng = np.random.default_rng(7)
    x, w, b = (ta.tensor(rng.standard_normal(s, dtype=np.float32), kind, device) for s in ((n, c, h, wd), (o, c, 1, 1), (o,)))
    check(x, w, b, values(ops.convolve2d(x, w, b)), eps)


PART = (128, 6, 7, 96)      # channels, height, width, channels out: out of three channels and two images more


@pytest.mark.parametrize("skip", [0, 1, 2, 3])
@pytest.mark.parametrize("n", [6, 300])
def test_part_of_a_tensor(n, skip, device):
    """Channels and images out of a larger tensor, from any element on (an odd one goes to the kernels before); what lies beside is infinite."""
    c, h, wd, o = PART
    rng = np.random.default_rng(8)
    whole = np.full((n + 2, c + 3, h, wd), np.inf, np.float32)
    whole[1:n + 1, 2:c + 2] = rng.standard_normal((n, c, h, wd), dtype=np.float32)
    flat = ta.tensor(np.concatenate([np.full(skip, np.inf, np.float32), whole.ravel()]), ta.float16, device)
    strides = ((c + 3) * h * wd, h * wd, wd, 1)
    x = flat._view((n, c, h, wd), strides, 2 * (skip + strides[0] + 2 * strides[1]))
    w, b = (ta.tensor(rng.standard_normal(s, dtype=np.float32), ta.float16, device) for s in ((o, c, 1, 1), (o,)))
    check(ta.tensor(whole[1:n + 1, 2:c + 2], ta.float16, device), w, b, values(ops.convolve2d(x, w, b)), 2.0 ** -11)
