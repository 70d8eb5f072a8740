"""Which 16-bit 1x1 convolutions run as one product whose tiles go over the images of a batch, and on which tiles, asked of the library without
a GPU."""
import ctypes as C

import pytest

import tannic_amd as ta
from tannic_amd import abi
import test_gpu_conv_columns
from test_conv_plan import descriptor, out_shape


def columns_plan(x, w, dtype="float16", strides=None, start=0):
    """Rows of a tile and stages of its operands, None where another kernel takes the problem."""
    out = (C.c_uint32 * 20)()
    signal, weights, result = (descriptor(dtype, s) for s in (x, w, out_shape(x, w, (1, 1), (0, 0))))
    if strides:
        signal.strides.sizes[:4] = strides
    signal.address += 2 * start
    assert ta.library().conv2d_plan(*(C.byref(t) for t in (signal, weights, result)), abi.SIZE2(0, 0), abi.SIZE2(1, 1), out) == abi.SUCCESS
    return tuple(out[2:4]) if out[0] == 5 else None


# images, channels, height, width, channels out -> the tiles here, or None: tiles of 256 x 256 image by image, or K shared between blocks
PROBLEMS = {
    # both sides of what the tiles of 256 x 256 take: rounds of 256 against pairs of 512, images that are no whole tiles, a short K
    "large": ((8, 1024, 64, 64, 1024), None),
    "large_long_k": ((32, 2048, 28, 28, 1024), None),
    "large_few_rows": ((8, 2048, 64, 64, 320), None),
    "large_short_k": ((8, 512, 64, 64, 2048), None),
    "large_short_k_padded_rows": ((8, 512, 64, 64, 320), (128, 2)),
    "large_second_round_empty": ((16, 1024, 48, 48, 320), (128, 2)),
    "large_ragged_images": ((32, 1024, 28, 28, 1024), (128, 2)),
    "large_few_channels_out": ((32, 1024, 32, 32, 192), (128, 2)),
    "large_odd_images": ((32, 2048, 14, 14, 2048), (128, 2)),
    "large_hardly_padded": ((33, 256, 64, 68, 1018), None),
    "large_hardly_padded_images": ((60, 320, 76, 72, 992), None),
    "large_padded": ((37, 320, 72, 72, 1856), (128, 2)),
    "large_hardly_padded_shortest_k": ((33, 128, 64, 68, 1018), (128, 2)),
    "large_hardly_padded_one_round": ((7, 256, 64, 68, 1018), (128, 2)),
    # few tiles under a long K
    "long_k": ((1, 8192, 32, 32, 64), None),
    "long_k_sixteen_tiles": ((4, 2048, 16, 16, 128), None),
    "long_k_fifty_tiles": ((4, 3072, 28, 28, 128), None),
    "long_k_more_tiles": ((16, 3072, 16, 16, 256), (64, 3)),
    "shorter_k_fifty_tiles": ((4, 1536, 28, 28, 128), (64, 3)),
    "long_k_a_tile_a_unit": ((16, 8192, 16, 16, 512), (64, 3)),
    "long_k_odd_images": ((16, 8192, 14, 14, 128), None),
    "long_k_odd_images_more_tiles": ((16, 3072, 14, 14, 128), (64, 3)),
    "ordinary": ((32, 512, 28, 28, 256), (128, 2)),
    "ordinary_four_stages": ((32, 1024, 14, 14, 512), (128, 4)),
    "ordinary_small": ((32, 1024, 14, 14, 256), (64, 3)),
}


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("name", list(PROBLEMS))
def test_problems(name, dtype):
    (n, c, h, w, o), want = PROBLEMS[name]
    assert columns_plan((n, c, h, w), (o, c, 1, 1), dtype) == want


@pytest.mark.parametrize("x,w", [((8, 1024, 64, 64), (1024, 1024, 1, 1)), ((1, 8192, 32, 32), (64, 8192, 1, 1))], ids=["large", "long_k"])
def test_signals_that_the_other_tiles_load_slowly_stay(x, w):
    """Rows at addresses that no 16 bytes divide."""
    n, c, h, wd = x
    plane = h * wd
    assert columns_plan(x, w) is None
    assert columns_plan(x, w, start=2) is not None
    assert columns_plan(x, w, strides=(c * (plane + 2), plane + 2, wd, 1)) is not None
    assert columns_plan(x, w, strides=(c * plane + 2, plane, wd, 1)) is not None


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
def test_the_shapes_on_the_gpu_are_these_tiles(dtype):
    seen = set()
    for name, (n, c, h, w, o) in test_gpu_conv_columns.SHAPES.items():
        tiles = columns_plan((n, c, h, w), (o, c, 1, 1), dtype)
        assert tiles, name
        seen.add(tiles)
    assert seen == {(64, 3), (128, 2), (128, 4)}
    for name, (n, c, h, w, o) in test_gpu_conv_columns.FEW_PIXELS.items():
        assert columns_plan((n, c, h, w), (o, c, 1, 1), dtype) is None, name


@pytest.mark.parametrize("skip", [0, 1, 2, 3])
def test_parts_of_a_tensor_on_the_gpu(skip):
    """From an even element on a piece's address is a multiple of four bytes."""
    c, h, w, o = test_gpu_conv_columns.PART
    strides = ((c + 3) * h * w, h * w, w, 1)
    assert bool(columns_plan((300, c, h, w), (o, c, 1, 1), strides=strides, start=skip + strides[0] + 2 * strides[1])) == (skip % 2 == 0)
