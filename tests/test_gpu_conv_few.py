"""16-bit conv2d over few output pixels (``conv2d_few.hip``: 1x1 and 3x3, channels a multiple of 32) against the CPU checker, at the
sizes where its tiles and its split of the channels end, and with views whose neighbours must not leak in; every compiled variant of
it against sums in 64 bits.

Bar: both sides sum in fp32 and round once: one unit of the result's last place, plus K * eps * max|x||w| for the order of the sums.
"""
import numpy as np
import pytest

import support
import tannic_amd as ta
from tannic_amd import ops
from test_conv_plan import conv_plan
from test_gpu_conv_f32 import convolve64

pytestmark = pytest.mark.gpu

# x shape, w shape, stride, padding.  A block is 1 or 2 tiles of 16 output channels by 1 or 2 of 16 pixels (which, depends on how
# many tiles there are), its 2, 4, 8 or 16 wavefronts take 32 channels at a time.
CASES = {
    "k1_one_result": ((1, 32, 1, 1), (1, 32, 1, 1), (1, 1), (0, 0)),
    "k1_three_groups_of_channels": ((1, 96, 3, 5), (17, 96, 1, 1), (1, 1), (0, 0)),
    "k1_four_wavefronts": ((2, 160, 4, 4), (16, 160, 1, 1), (1, 1), (0, 0)),
    "k1_eight_wavefronts_and_one_group": ((3, 288, 3, 3), (33, 288, 1, 1), (1, 1), (0, 0)),
    "k1_sixteen_wavefronts_and_one_group": ((1, 544, 7, 7), (40, 544, 1, 1), (1, 1), (0, 0)),
    "k1_two_pixel_tiles": ((1, 64, 57, 17), (83, 64, 1, 1), (1, 1), (0, 0)),
    "k1_two_pixel_tiles_sixteen_wavefronts": ((1, 512, 13, 13), (489, 512, 1, 1), (1, 1), (0, 0)),
    "k1_four_tiles": ((3, 256, 13, 7), (655, 256, 1, 1), (1, 1), (0, 0)),
    "k1_stride_two_channel_tiles": ((1, 512, 27, 25), (489, 512, 1, 1), (2, 2), (0, 0)),
    "k1_stride_four_tiles": ((1, 64, 57, 63), (199, 64, 1, 1), (2, 2), (0, 0)),
    "k1_rect_stride_padding": ((2, 32, 9, 12), (20, 32, 1, 1), (3, 1), (1, 2)),
    "k3_one_result": ((1, 32, 3, 3), (1, 32, 3, 3), (1, 1), (0, 0)),
    "k3_pixel_past_a_tile": ((1, 32, 1, 17), (16, 32, 3, 3), (1, 1), (1, 1)),
    "k3_seven_wide_images": ((3, 96, 7, 7), (50, 96, 3, 3), (1, 1), (1, 1)),
    "k3_two_channel_tiles": ((1, 64, 21, 19), (201, 64, 3, 3), (1, 1), (1, 1)),
    "k3_four_tiles": ((1, 64, 41, 29), (185, 64, 3, 3), (1, 1), (1, 1)),
    "k3_sixteen_wavefronts": ((1, 544, 7, 7), (70, 544, 3, 3), (1, 1), (1, 1)),
    "k3_sixteen_wavefronts_two_channel_tiles": ((5, 512, 5, 7), (497, 512, 3, 3), (1, 1), (1, 1)),
    "k3_stride_2": ((2, 128, 15, 29), (34, 128, 3, 3), (2, 2), (1, 1)),
    "k3_wide_padding": ((2, 32, 6, 5), (16, 32, 3, 3), (1, 1), (2, 3)),
    "k3_rect_stride": ((2, 32, 13, 17), (18, 32, 3, 3), (2, 3), (1, 0)),
}

# Every compiled variant: side, tiles of channels and of pixels per block, wavefronts -> x shape, w shape, stride.  Output channels and pixels
# that end inside a tile, tiles over several images, channels that are no whole turns of the wavefronts.
VARIANTS = {
    (1, 1, 1, 2): ((2, 32, 3, 3), (1, 32, 1, 1), 2),
    (1, 1, 1, 4): ((2, 160, 3, 3), (1, 160, 1, 1), 2),
    (1, 1, 1, 8): ((2, 352, 3, 3), (1, 352, 1, 1), 2),
    (1, 1, 1, 16): ((2, 544, 6, 4), (1, 544, 1, 1), 2),
    (1, 1, 2, 2): ((3, 32, 39, 41), (1, 32, 1, 1), 1),
    (1, 1, 2, 4): ((3, 160, 42, 40), (1, 160, 1, 1), 1),
    (1, 1, 2, 8): ((3, 288, 39, 43), (1, 288, 1, 1), 1),
    (1, 1, 2, 16): ((15, 576, 16, 21), (1, 576, 1, 1), 1),
    (1, 2, 1, 2): ((5, 32, 42, 47), (17, 32, 1, 1), 2),
    (1, 2, 1, 4): ((3, 160, 60, 57), (19, 160, 1, 1), 2),
    (1, 2, 1, 8): ((28, 320, 19, 17), (18, 320, 1, 1), 2),
    (1, 2, 1, 16): ((7, 544, 39, 35), (18, 544, 1, 1), 2),
    (1, 2, 2, 2): ((25, 32, 30, 30), (18, 32, 1, 1), 2),
    (1, 2, 2, 4): ((2, 160, 108, 103), (17, 160, 1, 1), 2),
    (1, 2, 2, 8): ((13, 288, 18, 24), (17, 288, 1, 1), 1),
    (3, 1, 1, 2): ((2, 32, 3, 3), (1, 32, 3, 3), 2),
    (3, 1, 1, 4): ((2, 160, 3, 4), (1, 160, 3, 3), 2),
    (3, 1, 1, 8): ((2, 288, 4, 4), (1, 288, 3, 3), 2),
    (3, 1, 1, 16): ((2, 544, 4, 3), (1, 544, 3, 3), 2),
    (3, 2, 1, 2): ((7, 32, 36, 38), (17, 32, 3, 3), 2),
    (3, 2, 1, 4): ((4, 160, 23, 29), (17, 160, 3, 3), 1),
    (3, 2, 1, 8): ((4, 288, 25, 25), (17, 288, 3, 3), 1),
    (3, 2, 1, 16): ((6, 608, 20, 21), (17, 608, 3, 3), 1),
    (3, 2, 2, 2): ((2, 32, 52, 54), (17, 32, 3, 3), 1),
    (3, 2, 2, 4): ((13, 160, 18, 24), (17, 160, 3, 3), 1),
    (3, 2, 2, 8): ((5, 288, 33, 34), (20, 288, 3, 3), 1),
}


@pytest.mark.parametrize("dtype", [ta.float16, ta.bfloat16], ids=str)
@pytest.mark.parametrize("variant", list(VARIANTS), ids=lambda v: "-".join(map(str, v)))
def test_variant(variant, dtype, device):
    xs, ws, stride = VARIANTS[variant]
    pad = ws[2] // 2
    kernel, plan = conv_plan(dtype.name, xs, ws, (stride, stride), (pad, pad))
    assert kernel == "few" and tuple(plan[n] for n in ("side", "mo", "np", "waves")) == variant
    x, w, b = (support.values_for(dtype, 6, i, shape, -1, 1) for i, shape in enumerate((xs, ws, ws[:1])))
    got = ops.convolve2d(*(ta.tensor(v, dtype, device) for v in (x, w, b)), stride, pad).numpy()
    rounded = [ta.tensor(v, dtype).numpy().astype(np.float32) for v in (x, w, b)]
    want = convolve64(rounded[0], rounded[1], stride, pad) + rounded[2][:, None, None]
    support.assert_close(got, want, 2.0 ** -10 if dtype is ta.float16 else 2.0 ** -7, (ws[1] * ws[2] * ws[3] + 1) * 2.0 ** -23, str(variant))


@pytest.mark.parametrize("dtype", [ta.float16, ta.bfloat16], ids=str)
@pytest.mark.parametrize("name", list(CASES))
def test_conv2d_few(name, dtype, device):
    xs, ws, stride, padding = CASES[name]
    x, w, b = (support.values_for(dtype, 5, i, shape, -1, 1) for i, shape in enumerate((xs, ws, (ws[0],))))
    (hx, dx), (hw, dw), (hb, db) = (support.both(v, dtype, device) for v in (x, w, b))
    assert conv_plan(dtype.name, xs, ws, stride, padding)[0] == "few"
    place = 2.0 ** -10 if dtype is ta.float16 else 2.0 ** -7
    terms = ws[1] * ws[2] * ws[3] + 1
    for hbias, dbias in ((None, None), (hb, db)):
        want = ops.convolve2d(hx, hw, hbias, stride, padding).numpy()
        got = ops.convolve2d(dx, dw, dbias, stride, padding).numpy()
        support.assert_close(got, want, place, terms * 2.0 ** -23, name)


@pytest.mark.parametrize("kernel", [1, 3])
def test_views_and_what_lies_beside_them(kernel, device):
    """A signal whose images, rows and columns are slices of a larger tensor full of infinities; weights that start inside a larger tensor."""
    x = np.full((3, 64, 10, 13), np.inf, np.float16)
    x[1, :, 2:8, 3:10] = support.uniform(7, 1, (64, 6, 7), -1, 1)
    w = support.uniform(7, 2, (17, 64, kernel, kernel), -1, 1).astype(np.float16)
    hx, dx = support.both(x, ta.float16, device)
    hw, dw = support.both(w, ta.float16, device)
    at = kernel // 2
    for part in (slice(0, 17), slice(1, 16)):
        want = ops.convolve2d(hx[1:2, :, 2:8, 3:10], hw[part], None, 1, at).numpy()
        got = ops.convolve2d(dx[1:2, :, 2:8, 3:10], dw[part], None, 1, at).numpy()
        support.assert_close(got, want, 2.0 ** -10, 64 * kernel * kernel * 2.0 ** -23, "view")
    # columns swapped with rows: no run of the signal is contiguous
    want = ops.convolve2d(hx[1:2, :, 2:8, 3:10].transpose(-1, -2), hw, None, 1, at).numpy()
    got = ops.convolve2d(dx[1:2, :, 2:8, 3:10].transpose(-1, -2), dw, None, 1, at).numpy()
    support.assert_close(got, want, 2.0 ** -10, 64 * kernel * kernel * 2.0 ** -23, "transposed view")
