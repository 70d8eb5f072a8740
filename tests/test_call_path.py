"""The operator interface keeps rules by shape between calls: what a call is refused for does not depend on the calls before it."""
import types

import numpy as np
import pytest

import tannic_amd as ta
from tannic_amd import ops


def host(shape, dtype=ta.float32):
    return ta.tensor(np.ones(shape), dtype)


@pytest.mark.parametrize("where", ["stride", "padding"])
@pytest.mark.parametrize("value", [(1.0, 1.0), (1, 1.0), (np.float64(1), 1)], ids=["floats", "one_float", "numpy_float"])
def test_strides_that_only_equal_whole_numbers_are_refused(where, value, oracle):
    """Also after a convolution of the same shapes under the whole numbers."""
    x, w = host((1, 2, 7, 6)), host((3, 2, 3, 3))
    for whole in (1, (1, 1), (np.int64(1), 1)):
        got = ops.convolve2d(x, w, **{"stride": 1, "padding": 1, where: whole})
        assert got.shape == (1, 3, 7, 6)
        with pytest.raises(TypeError):
            ops.convolve2d(x, w, **{"stride": 1, "padding": 1, where: value})


def test_shapes_are_whole_numbers_whatever_came_before(oracle):
    x, w = host((1, 2, 8, 6)), host((3, 2, 3, 3))
    ops.convolve2d(x, w, stride=(np.int64(1), np.int64(1)))
    assert all(type(s) is int for s in ops.convolve2d(x, w).shape)


def on_another_device(tensor):
    """The same tensor as if it lay on a device (never called with: there is none here)."""
    elsewhere = ta.Tensor(tensor.dtype, tensor.shape)
    device = ta.Device.__new__(ta.Device)
    device.id, device.key = 7, (device.kind, 7)
    elsewhere.buffer = types.SimpleNamespace(environment=device)
    return elsewhere


def test_different_devices_are_reported_before_types_and_strides(oracle):
    a = host((4, 4), ta.complex64)
    with pytest.raises(ops.TannicError, match="Environment"):
        ops.matmul(a, on_another_device(a))
    x, w = host((1, 2, 9, 6)), host((3, 2, 3, 3))
    with pytest.raises(ops.TannicError, match="Environment"):
        ops.convolve2d(x, on_another_device(w), stride=(1.0, 1.0))
    with pytest.raises(ops.TannicError, match="Environment"):
        ops.convolve2d(x, w, on_another_device(host((3,))), stride=(1.0, 1.0))


def test_a_tensor_initialised_again_is_where_it_lies_now(oracle):
    t = host((3, 5))
    before, held = t.packed(), t.buffer
    t.initialize(np.full((3, 5), 2.0))
    assert t.packed()[8:] == before[8:] and t.packed()[:8] == t.buffer.address.to_bytes(8, "little") != held.address.to_bytes(8, "little")
    assert t.descriptor().address == t.address
    assert (ops.add(t, t).numpy() == 4.0).all()


def test_results_do_not_depend_on_what_is_kept(oracle):
    """More shapes than the tables hold, the first of them again afterwards."""
    first = ops.matmul(host((2, 3)), host((3, 4)))
    for n in range(1, 4200):
        for table in (ops._PRODUCTS, ops._CONVOLUTIONS):
            table[n] = None
        ta.Tensor.fresh(ta.int8, (1, n), ta.Host())
    ops.convolve2d(host((1, 2, 7, 6)), host((3, 2, 3, 3)))
    again = ops.matmul(host((2, 3)), host((3, 5)))
    assert len(ops._PRODUCTS) == 1 and len(ops._CONVOLUTIONS) == 1
    assert again.shape == (2, 5) and (again.numpy() == 3.0).all() and (ops.matmul(host((2, 3)), host((3, 4))).numpy() == first.numpy()).all()
