"""16-bit 3x3 conv2d over few output pixels whose signal and weights are staged in LDS (``conv2d_few3.hip``): every compiled variant of it against
sums in 64 bits, at output channels and pixels that end inside a tile, and beside values that must not leak in.

Bar: sums in fp32, rounded once: one unit of the result's last place, plus K * eps * max|x||w| for the order of the sums.
"""
import ctypes as C

import numpy as np
import pytest

import support
import tannic_amd as ta
from tannic_amd import abi, ops
from test_conv_plan import descriptor, out_shape
from test_gpu_conv_f32 import convolve64

# output channels, tiles of 16 pixels and wavefronts of a block, pieces of the signal a lane has on their way at once -> x shape, w shape, stride
VARIANTS = {
    (8, 1, 2, 1): ((1, 64, 2, 4), (33, 64, 3, 3), 2),
    (8, 1, 2, 2): ((1, 64, 6, 24), (36, 64, 3, 3), 2),
    (8, 1, 4, 1): ((1, 128, 2, 4), (34, 128, 3, 3), 2),
    (8, 1, 4, 2): ((1, 160, 7, 22), (39, 160, 3, 3), 2),
    (8, 1, 8, 1): ((1, 288, 2, 4), (32, 288, 3, 3), 2),
    (8, 1, 8, 2): ((1, 288, 8, 22), (39, 288, 3, 3), 2),
    (8, 1, 16, 1): ((1, 576, 3, 4), (33, 576, 3, 3), 2),
    (16, 1, 2, 1): ((10, 64, 3, 4), (203, 64, 3, 3), 2),
    (16, 1, 2, 2): ((2, 64, 5, 45), (203, 64, 3, 3), 2),
    (16, 1, 4, 1): ((13, 128, 3, 5), (156, 128, 3, 3), 2),
    (16, 1, 4, 2): ((8, 128, 5, 26), (83, 128, 3, 3), 2),
    (16, 1, 8, 1): ((6, 256, 2, 5), (353, 256, 3, 3), 2),
    (16, 1, 8, 2): ((15, 256, 5, 26), (42, 256, 3, 3), 2),
    (16, 2, 2, 1): ((13, 64, 5, 11), (525, 64, 3, 3), 2),
    (16, 2, 2, 2): ((7, 64, 7, 102), (34, 64, 3, 3), 2),
    (16, 2, 4, 1): ((14, 128, 5, 11), (158, 128, 3, 3), 2),
    (16, 2, 4, 2): ((10, 128, 19, 26), (34, 128, 3, 3), 2),
    (16, 2, 8, 1): ((5, 256, 9, 7), (411, 256, 3, 3), 2),
    (16, 2, 8, 2): ((3, 256, 18, 29), (33, 256, 3, 3), 1),
    (16, 4, 2, 1): ((19, 64, 16, 21), (70, 64, 3, 3), 1),
    (16, 4, 2, 2): ((2, 64, 19, 72), (34, 64, 3, 3), 1),
    (16, 4, 4, 1): ((20, 128, 13, 9), (222, 128, 3, 3), 2),
    (16, 4, 4, 2): ((19, 128, 7, 22), (101, 128, 3, 3), 2),
    (16, 4, 8, 1): ((8, 256, 9, 13), (265, 256, 3, 3), 2),
    (16, 4, 8, 2): ((7, 256, 13, 10), (305, 256, 3, 3), 2),
    (32, 2, 2, 1): ((18, 64, 19, 24), (50, 64, 3, 3), 1),
    (32, 2, 2, 2): ((6, 64, 17, 65), (73, 64, 3, 3), 2),
    (32, 2, 4, 1): ((16, 256, 5, 5), (289, 256, 3, 3), 2),
    (32, 2, 4, 2): ((18, 128, 19, 28), (33, 128, 3, 3), 2),
    (32, 2, 8, 1): ((8, 256, 3, 4), (519, 256, 3, 3), 2),
}
# paddings and strides whose tiles see rows and columns beside the image only: x, w, stride, padding
EDGES = {
    "no_padding": ((2, 64, 9, 11), (40, 64, 3, 3), (1, 1), (0, 0)),
    "rows_of_zeros": ((1, 96, 3, 9), (33, 96, 3, 3), (1, 1), (4, 5)),
    "strides_beyond_the_kernel": ((3, 64, 13, 17), (32, 64, 3, 3), (4, 5), (1, 2)),
    "one_row": ((2, 64, 1, 23), (35, 64, 3, 3), (1, 1), (1, 1)),
    "seven_units_of_channels": ((1, 224, 7, 7), (64, 224, 3, 3), (1, 1), (1, 1)),
}


def few3_plan(dtype, x, w, stride, padding):
    out = (C.c_uint32 * 20)()
    args = [C.byref(descriptor(dtype, s)) for s in (x, w, out_shape(x, w, stride, padding))]
    assert ta.library().conv2d_plan(*args, abi.SIZE2(*padding), abi.SIZE2(*stride), out) == abi.SUCCESS
    return (out[6], out[3], out[4], out[7]) if out[0] in (2, 6) and out[7] else None


def check(dtype, xs, ws, stride, pad, device, name):
    x, w, b = (support.values_for(dtype, 6, i, shape, -1, 1) for i, shape in enumerate((xs, ws, ws[:1])))
    got = ops.convolve2d(*(ta.tensor(v, dtype, device) for v in (x, w, b)), stride, pad).numpy()
    rounded = [ta.tensor(v, dtype).numpy().astype(np.float32) for v in (x, w, b)]
    padded = np.pad(rounded[0], ((0, 0), (0, 0), (pad[0], pad[0]), (pad[1], pad[1])))
    want = (convolve64(padded, rounded[1], 1, 0) + rounded[2][:, None, None])[:, :, ::stride[0], ::stride[1]]
    support.assert_close(got, want, 2.0 ** -10 if dtype is ta.float16 else 2.0 ** -7, (9 * ws[1] + 1) * 2.0 ** -23, name)


@pytest.mark.parametrize("variant", list(VARIANTS), ids=lambda v: "-".join(map(str, v)))
def test_plan(variant):
    xs, ws, stride = VARIANTS[variant]
    assert few3_plan("float16", xs, ws, (stride, stride), (1, 1)) == few3_plan("bfloat16", xs, ws, (stride, stride), (1, 1)) == variant


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [ta.float16, ta.bfloat16], ids=str)
@pytest.mark.parametrize("variant", list(VARIANTS), ids=lambda v: "-".join(map(str, v)))
def test_variant(variant, dtype, device):
    xs, ws, stride = VARIANTS[variant]
    check(dtype, xs, ws, (stride, stride), (1, 1), device, str(variant))


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(EDGES))
def test_edges(name, device):
    xs, ws, stride, pad = EDGES[name]
    assert few3_plan("float16", xs, ws, stride, pad)
    check(ta.float16, xs, ws, stride, pad, device, name)


@pytest.mark.gpu
def test_what_lies_beside_a_view(device):
    """Images and channels that are slices of a tensor full of infinities, at an odd address; weights that are rows of a larger tensor."""
    x = np.full((3, 67, 7, 9), np.inf, np.float16)
    x[1, 1:65] = support.uniform(7, 1, (64, 7, 9), -1, 1)
    w = support.uniform(7, 2, (52, 64, 3, 3), -1, 1).astype(np.float16)
    (hx, dx), (hw, dw) = support.both(x, ta.float16, device), support.both(w, ta.float16, device)
    want = ops.convolve2d(hx[1:2, 1:65], hw[3:50], None, 1, 1).numpy()
    got = ops.convolve2d(dx[1:2, 1:65], dw[3:50], None, 1, 1).numpy()
    support.assert_close(got, want, 2.0 ** -10, 64 * 9 * 2.0 ** -23, "view")


def weights_at(start, pitch, rows=47, address=0x10000):
    """Descriptors of a problem that is the kernel's (13 x 17 pixels under 64 channels), its weights ``start`` elements behind a multiple of 16 bytes, ``pitch`` from row to row."""
    x, w, y = (descriptor("float16", s) for s in ((2, 64, 13, 17), (rows, 64, 3, 3), (2, rows, 13, 17)))
    w.address = address + 2 * start
    w.strides.sizes[0] = pitch
    return x, w, y


def runs_on_few3(x, w, y):
    out = (C.c_uint32 * 20)()
    assert ta.library().conv2d_plan(x, w, y, abi.SIZE2(1, 1), abi.SIZE2(1, 1), out) == abi.SUCCESS
    return out[0] in (2, 6) and out[7] > 0


# elements from a multiple of 16 bytes to the weights, from row to row -> loaded into LDS as they lie (at multiples of four bytes)
STARTS = {(0, 576): True, (2, 612): True, (4, 578): True, (6, 584): True, (1, 612): False, (2, 613): False}


@pytest.mark.parametrize("start,pitch", list(STARTS))
def test_plan_of_weights_as_they_lie(start, pitch):
    assert runs_on_few3(*map(C.byref, weights_at(start, pitch))) == STARTS[start, pitch]


@pytest.mark.gpu
@pytest.mark.parametrize("start,pitch", list(STARTS))
def test_weights_as_they_lie(start, pitch, device):
    """Rows of weights between infinities, and a result within a larger tensor whose other elements stay what they were."""
    w = np.full(start + 47 * pitch + 8, np.inf, np.float16)
    rows = np.lib.stride_tricks.as_strided(w[start:], (47, 576), (2 * pitch, 2))
    rows[...] = support.uniform(8, 1, (47, 576), -1, 1)
    x = support.uniform(8, 2, (2, 64, 13, 17), -1, 1).astype(np.float16)
    dx, dw = ta.tensor(x, ta.float16, device), ta.tensor(w, ta.float16, device)._view((47, 64, 3, 3), (pitch, 9, 3, 1), 2 * start)
    room = ta.tensor(np.full((3, 50, 14, 19), 7.0, np.float16), ta.float16, device)
    y = room[1:, 2:49, 1:, 1:18]
    assert runs_on_few3(dx.reference(), dw.reference(), y.reference()) == STARTS[start, pitch]
    ops._call("conv2d", device, (dx, dw), y, (abi.SIZE2(1, 1), abi.SIZE2(1, 1)))
    got = room.numpy()
    padded = np.pad(x.astype(np.float32), ((0, 0), (0, 0), (1, 1), (1, 1)))
    want = convolve64(padded, rows.reshape(47, 64, 3, 3).astype(np.float32), 1, 0)
    support.assert_close(got[1:, 2:49, 1:, 1:18], want, 2.0 ** -10, 64 * 9 * 2.0 ** -23, f"{start} {pitch}")
    beside = np.ones(got.shape, bool)
    beside[1:, 2:49, 1:, 1:18] = False
    assert (got[beside] == 7.0).all()


@pytest.mark.gpu
def test_the_view_above_is_the_kernels(device):
    x, w = ta.tensor(np.zeros((3, 67, 7, 9)), ta.float16, device)[1:2, 1:65], ta.tensor(np.zeros((52, 64, 3, 3)), ta.float16, device)[3:50]
    assert runs_on_few3(x.reference(), w.reference(), ta.Tensor(ta.float16, (1, 47, 7, 9)).initialize(device).reference())
