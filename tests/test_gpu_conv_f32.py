"""fp32 conv2d on the kernel whose blocks walk the flattened batch (1x1, 3x3 and 7x7) against the CPU checker, at the sizes where
its tiles end: channels that do not fill a chunk, output channels that do not fill a wavefront, a pixel more and a pixel less than
a tile, several images in one tile, rows of any width, strides and paddings, channels shared between blocks.

Bar: 1e-5 relative plus K * eps * max|x||w| for the order of summation (fp32 sums of K products).
"""
import numpy as np
import pytest

import support
import tannic_amd as ta
from tannic_amd import ops

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


@pytest.mark.parametrize("biased", [False, True])
@pytest.mark.parametrize("name", list(CASES))
def test_conv2d_f32(name, biased, device):
    xs, ws, stride, padding = CASES[name]
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
