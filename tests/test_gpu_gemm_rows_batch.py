"""16-bit products of at most four rows with narrow row-major matrices (``gemm_rows_batch.hip``) against the CPU checker, where its
tiles, its lanes' rows and its wavefronts end, and with views whose neighbours must not leak in.

Bar: both sides sum in fp32 and round once: one unit of the result's last place, plus K * eps * max|a||b| for the order of the sums.
"""
import numpy as np
import pytest

import support
import tannic_amd as ta
from tannic_amd import ops

pytestmark = pytest.mark.gpu

# batches, M, N, K.  Blocks are 16 columns wide, or 32 with 8192 columns in all; sixteen wavefronts take 256 or 64 rows of W in turn.
CASES = [((26,), 3, 128, 1001), ((2, 16), 4, 72, 1025), ((64,), 4, 128, 1027), ((128,), 2, 64, 1023), ((9,), 4, 256, 4099), ((86,), 4, 24, 2049)]


def check(got, want, dtype, k, what):
    support.assert_close(got.numpy(), want, 2.0 ** -10 if dtype is ta.float16 else 2.0 ** -7, k * 2.0 ** -23, what)


@pytest.mark.parametrize("dtype", [ta.float16, ta.bfloat16], ids=str)
@pytest.mark.parametrize("batch,m,n,k", CASES, ids=lambda v: str(v).replace(" ", ""))
def test_few_rows_times_narrow_matrices(batch, m, n, k, dtype, device):
    (hx, dx), (hw, dw) = (support.both(support.values_for(dtype, 3, i, batch + s, -1, 1), dtype, device) for i, s in enumerate(((m, k), (k, n))))
    want = ops.matmul(hx, hw).numpy()
    check(ops.matmul(dx, dw), want, dtype, k, str((batch, m, n, k)))


@pytest.mark.parametrize("first", [0, 1])
def test_views_and_what_lies_beside_them(first, device):
    """Slices of tensors full of infinities that start at any element, W broadcast over a batch dimension."""
    x, w = np.full((2, 50, 6, 1010), np.inf, np.float16), np.full((1, 50, 1010, 30), np.inf, np.float16)
    x[:, :, 1:5, first:first + 1003] = support.uniform(9, 1, (2, 50, 4, 1003), -1, 1)
    w[:, :, 3:1006, first:first + 24] = support.uniform(9, 2, (1, 50, 1003, 24), -1, 1)
    (hx, dx), (hw, dw) = support.both(x, ta.float16, device), support.both(w, ta.float16, device)
    want, got = (ops.matmul(a[:, :, 1:5, first:first + 1003], b[:, :, 3:1006, first:first + 24]) for a, b in ((hx, hw), (dx, dw)))
    check(got, want.numpy(), ta.float16, 1003, "views")
