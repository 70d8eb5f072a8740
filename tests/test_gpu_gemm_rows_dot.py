"""One row (two of fp32) times a matrix whose rows are contiguous along K (``gemm_rows_dot.hip``), and the few rows whose matrix is loaded past the caches
(``gemm_skinny.hip``), against sums in 64 bits: rows that end inside a turn of loads, columns that end inside a block.

Bar: sums in fp32, rounded once: one unit of the result's last place, plus K * eps * max|x||w| for the order of the sums.
"""
import numpy as np
import pytest

import support
import tannic_amd as ta
from tannic_amd import ops

pytestmark = pytest.mark.gpu

# rows, columns, K: the shortest and the longest K, turns that end after four loads and inside one, x as long as LDS takes
SHAPES = {
    "float16": [(1, 1, 2048), (1, 7, 2056), (1, 300, 4096), (1, 5, 6152), (1, 2049, 8192), (1, 33, 32768)],
    "bfloat16": [(1, 2, 2048), (1, 301, 4000), (1, 257, 6144), (1, 9, 20000)],
    "float32": [(1, 3, 1024), (2, 129, 1028), (1, 65, 2048), (2, 2050, 4096), (2, 31, 8192), (1, 5, 16384)],
}


def product(dtype, m, n, k, device, name):
    x, w = support.values_for(dtype, 3, 1, (m, k), -1, 1), support.values_for(dtype, 3, 2, (n, k), -1, 1)
    got = ops.matmul(ta.tensor(x, dtype, device), ta.tensor(w, dtype, device).transpose()).numpy()
    want = ta.tensor(x, dtype).numpy().astype(np.float64) @ ta.tensor(w, dtype).numpy().astype(np.float64).T
    place = {"float16": 2.0 ** -10, "bfloat16": 2.0 ** -7, "float32": 2.0 ** -23}[dtype.name]
    support.assert_close(got, want, place, k * 2.0 ** -23, name)


@pytest.mark.parametrize("name,shape", [(name, s) for name in SHAPES for s in SHAPES[name]], ids=lambda v: v if isinstance(v, str) else "x".join(map(str, v)))
def test_rows(name, shape, device):
    product(getattr(ta, name), *shape, device, f"{name} {shape}")


@pytest.mark.parametrize("rows", [1, 2, 17])
def test_matrix_past_the_caches(rows, device):
    """40 MB and more of W; 5121 columns end inside every kernel's block."""
    product(ta.float16, rows, 5121, 4096, device, f"{rows} rows")


def test_rows_of_a_larger_matrix(device):
    """x and W are rows and columns of larger tensors full of infinities."""
    x, w = np.full((3, 2072), np.inf, np.float16), np.full((40, 2072), np.inf, np.float16)
    x[1, 8:2064], w[3:37, 8:2064] = support.uniform(7, 1, (2056,), -1, 1), support.uniform(7, 2, (34, 2056), -1, 1)
    got = ops.matmul(ta.tensor(x, ta.float16, device)[1:2, 8:2064], ta.tensor(w, ta.float16, device)[3:37, 8:2064].transpose()).numpy()
    want = x[1:2, 8:2064].astype(np.float64) @ w[3:37, 8:2064].astype(np.float64).T
    support.assert_close(got, want, 2.0 ** -10, 2056 * 2.0 ** -23, "view")
