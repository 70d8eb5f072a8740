"""What attention does while decoding, at the sizes where its kernels end: a few rows of probabilities times cached values with few results
(``gemm_rows_few_kernel``), and the softmax of rows held in registers (``softmax_held_kernel``).

Bars: the product sums in fp32 and rounds once; the softmax rounds once, its exponentials and sum good to some units of fp32's last place
(16-bit types: of the hardware's exponential)."""
import numpy as np
import pytest

import tannic_amd as ta
from tannic_amd import ops

pytestmark = pytest.mark.gpu

EPS = {ta.float16: 2.0 ** -11, ta.bfloat16: 2.0 ** -8, ta.float32: 2.0 ** -24}

# batches, M, N, K: one wavefront's rows and a row more, a pass of 4096 and a row more, columns that end in a block, aligned and odd
PRODUCTS = [(8, 4, 128, 2049), (8, 4, 128, 2048), (3, 1, 8, 512), (2, 2, 24, 513), (5, 3, 40, 1000), (1, 4, 128, 4096), (1, 4, 16, 4097), (2, 4, 72, 9301), (16, 4, 128, 769)]
# and one beside them: rows of an odd number of 16-byte pieces whose last pass would be short
BESIDE = [(2, 4, 72, 9001)]


@pytest.mark.parametrize("dtype", [ta.float16, ta.bfloat16], ids=str)
@pytest.mark.parametrize("batch,m,n,k", PRODUCTS + BESIDE)
def test_few_results_of_row_major_matrices(batch, m, n, k, dtype, device):
    """The matrices are the first rows of larger ones (a cache with room), x is a slice of rows of another length; what lies beside is infinite."""
    rng = np.random.default_rng(5)
    x, w = np.full((batch, m, k + 3), np.inf, np.float32), np.full((batch, k + 7, n), np.inf, np.float32)
    x[:, :, 1:k + 1], w[:, :k] = rng.uniform(0, 1, (batch, m, k)), rng.standard_normal((batch, k, n))
    x, w = ta.tensor(x, dtype, device)[:, :, 1:k + 1], ta.tensor(w, dtype, device)[:, 0:k, :]
    got = ops.matmul(x, w).numpy().astype(np.float64)
    a, b = x.numpy().astype(np.float64), w.numpy().astype(np.float64)
    want = a @ b
    bound = EPS[dtype] * np.abs(want) + k * 2.0 ** -24 * (np.abs(a) @ np.abs(b))
    assert (np.abs(got - want) <= bound).all()


@pytest.mark.parametrize("dtype", [ta.float16, ta.bfloat16, ta.float32], ids=str)
@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("rows,length", [(3, 1), (5, 255), (32, 1023), (7, 1025), (32, 2049), (2, 4095), (3, 4097)])
def test_softmax_of_odd_rows(rows, length, masked, dtype, device):
    rng = np.random.default_rng(6)
    x = ta.tensor(rng.standard_normal((rows, length)) * 3, dtype, device)
    mask = np.where(rng.random((rows, length)) < 0.3, -np.inf, 0.0)
    mask[:, 0] = 0.0
    v = x.numpy().astype(np.float64) * 0.5 + (mask if masked else 0.0)
    got = ops.softmax(x, ta.tensor(mask, dtype, device) if masked else None, 0.5).numpy().astype(np.float64)
    e = np.exp(v - v.max(-1, keepdims=True))
    want = e / e.sum(-1, keepdims=True)
    # (the sum of `length` values in fp32, the exponential of a difference that is off by half a unit of its last place)
    bound = want * (EPS[dtype] + 2.0 ** -24 * (length ** 0.5 + 40)) + (2.0 ** -25 if dtype is ta.float16 else 0.0)
    assert (np.abs(got - want) <= bound).all(), float((np.abs(got - want) / np.maximum(bound, 1e-300)).max())
