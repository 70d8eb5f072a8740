"""The operator interface keeps rules by shape between calls: what a call is refused for does not depend on the calls before it."""
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
