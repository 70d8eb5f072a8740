"""16-bit 1x1 conv2d over few output pixels whose signal comes back from LDS transposed (``conv2d_few1.hip``): every compiled variant of it against
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

# tiles of 16 output channels and of 16 pixels of a block, its wavefronts, the turns whose loads are on their way at once -> x shape, w shape
VARIANTS = {
    (1, 1, 2, 1): ((1, 64, 3, 6), (34, 64, 1, 1)),
    (1, 1, 4, 1): ((1, 96, 3, 6), (33, 96, 1, 1)),
    (1, 1, 8, 1): ((1, 160, 3, 6), (34, 160, 1, 1)),
    (1, 1, 16, 1): ((1, 320, 3, 8), (34, 320, 1, 1)),
    (1, 1, 16, 2): ((1, 672, 3, 6), (33, 672, 1, 1)),
    (1, 2, 2, 1): ((8, 64, 35, 35), (33, 64, 1, 1)),
    (1, 2, 4, 1): ((18, 128, 13, 18), (33, 128, 1, 1)),
    (1, 2, 8, 1): ((7, 256, 12, 17), (33, 256, 1, 1)),
    (1, 2, 16, 1): ((18, 288, 3, 12), (73, 288, 1, 1)),
    (1, 2, 16, 2): ((19, 544, 6, 11), (33, 544, 1, 1)),
    (2, 2, 2, 1): ((2, 32, 21, 22), (2842, 32, 1, 1)),
    (2, 2, 4, 1): ((14, 96, 36, 43), (33, 96, 1, 1)),
    (2, 2, 8, 1): ((10, 224, 4, 10), (620, 224, 1, 1)),
    (2, 2, 16, 1): ((19, 416, 12, 11), (37, 416, 1, 1)),
    (2, 2, 16, 2): ((3, 544, 26, 35), (33, 544, 1, 1)),
}


def few1_plan(dtype, x, w):
    out = (C.c_uint32 * 20)()
    args = [C.byref(descriptor(dtype, s)) for s in (x, w, out_shape(x, w, (1, 1), (0, 0)))]
    assert ta.library().conv2d_plan(*args, abi.SIZE2(0, 0), abi.SIZE2(1, 1), out) == abi.SUCCESS
    return tuple(out[i] for i in (2, 3, 4, 7)) if out[0] in (2, 6) and out[7] else None


def check(x, w, b, dtype, device, view, name):
    got = ops.convolve2d(*(view(ta.tensor(v, dtype, device), i) for i, v in enumerate((x, w, b)))).numpy()
    rounded = [view(ta.tensor(v, dtype), i).numpy().astype(np.float64) for i, v in enumerate((x, w, b))]
    want = np.einsum("oc,nchw->nohw", rounded[1][:, :, 0, 0], rounded[0]) + rounded[2][:, None, None]
    support.assert_close(got, want, 2.0 ** -10 if dtype is ta.float16 else 2.0 ** -7, (rounded[1].shape[1] + 1) * 2.0 ** -23, name)


@pytest.mark.parametrize("variant", list(VARIANTS), ids=lambda v: "-".join(map(str, v)))
def test_plan(variant):
    assert few1_plan("float16", *VARIANTS[variant]) == few1_plan("bfloat16", *VARIANTS[variant]) == variant


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [ta.float16, ta.bfloat16], ids=str)
@pytest.mark.parametrize("variant", list(VARIANTS), ids=lambda v: "-".join(map(str, v)))
def test_variant(variant, dtype, device):
    xs, ws = VARIANTS[variant]
    check(*(support.values_for(dtype, 6, i, s, -1, 1) for i, s in enumerate((xs, ws, ws[:1]))), dtype, device, lambda t, i: t, str(variant))


@pytest.mark.gpu
def test_what_lies_beside_a_view(device):
    """Images and channels that are slices of a tensor full of infinities, at an odd address; weights that are columns of a larger tensor."""
    x = np.full((3, 67, 7, 9), np.inf, np.float16)
    x[1:, 1:65] = support.uniform(7, 1, (2, 64, 7, 9), -1, 1)
    w = np.full((52, 71, 1, 1), np.inf, np.float16)
    w[:, 3:67] = support.uniform(7, 2, (52, 64, 1, 1), -1, 1)
    b = support.uniform(7, 3, (52,), -1, 1).astype(np.float16)
    check(x, w, b, ta.float16, device, lambda t, i: t[((slice(1, None), slice(1, 65)), (slice(2, 49), slice(3, 67)), (slice(2, 49),))[i]], "view")


@pytest.mark.gpu
def test_the_view_above_is_the_kernels(device):
    x, w = ta.tensor(np.zeros((3, 67, 7, 9)), ta.float16, device)[1:, 1:65], ta.tensor(np.zeros((52, 71, 1, 1)), ta.float16, device)[2:49, 3:67]
    out = (C.c_uint32 * 20)()
    y = ta.Tensor(ta.float16, (2, 47, 7, 9)).initialize(device)
    assert ta.library().conv2d_plan(x.reference(), w.reference(), y.reference(), abi.SIZE2(0, 0), abi.SIZE2(1, 1), out) == abi.SUCCESS
    assert out[0] in (2, 6) and out[7]
