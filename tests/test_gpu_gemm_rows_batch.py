"""16-bit products of two to four rows with narrow row-major matrices (``gemm_rows_batch.hip``) against the CPU checker, where its
tiles, its lanes' rows and its wavefronts end, and with views whose neighbours must not leak in.

Bar: both sides sum in fp32 and round once: one unit of the result's last place, plus K * eps * max|a||b| for the order of the sums.
"""
import numpy as np
import pytest

import support
import tannic_amd as ta
from tannic_amd import ops

pytestmark = pytest.mark.gpu

# batches, M, N, K, lanes.  Blocks are 32 columns wide, or 16 under few columns or a long K; sixteen wavefronts take 64 or 256 rows of W in turn.
CASES = [((26,), 3, 128, 1001, 4), ((2, 16), 4, 72, 1025, 4), ((64,), 4, 128, 1027, 4), ((128,), 2, 64, 1023, 4), ((9,), 4, 256, 4099, 2),
         ((86,), 4, 24, 2049, 4), ((300,), 4, 8, 1003, 2), ((130,), 4, 16, 1025, 2), ((300,), 4, 32, 1001, 4), ((512,), 2, 32, 1023, 4),
         ((25,), 4, 160, 3001, 2), ((131,), 3, 40, 1009, 2)]


def lanes_of(x, w):
    y = ta.Tensor(x.dtype, x.shape[:-1] + w.shape[-1:]).initialize(x.environment)
    return ta.library().gemm_rows_batch_lanes(x.reference(), w.reference(), y.reference())


def check(got, want, dtype, k, what):
    support.assert_close(got.numpy(), want, 2.0 ** -10 if dtype is ta.float16 else 2.0 ** -7, k * 2.0 ** -23, what)


@pytest.mark.parametrize("dtype", [ta.float16, ta.bfloat16], ids=str)
@pytest.mark.parametrize("batch,m,n,k,lanes", CASES, ids=lambda v: str(v).replace(" ", ""))
def test_few_rows_times_narrow_matrices(batch, m, n, k, lanes, dtype, device):
    (hx, dx), (hw, dw) = (support.both(support.values_for(dtype, 3, i, batch + s, -1, 1), dtype, device) for i, s in enumerate(((m, k), (k, n))))
    assert lanes_of(dx, dw) == lanes
    # (the checker counts products in eight bits, as src/cpu/matmul.cpp:121 does: 256 at a time)
    want = ops.matmul(hx, hw).numpy() if len(batch) > 1 else np.concatenate([ops.matmul(hx[i:i + 256], hw[i:i + 256]).numpy() for i in range(0, batch[0], 256)])
    check(ops.matmul(dx, dw), want, dtype, k, str((batch, m, n, k)))


@pytest.mark.parametrize("pitch,first", [(1027, 0), (1040, 3)], ids=["odd_pitch", "odd_start"])
@pytest.mark.parametrize("side", ["x", "w"])
def test_whole_k_in_misaligned_rows(side, pitch, first, device):
    """K a multiple of eight; the rows of one operand start anywhere."""
    x, w = support.uniform(4, 1, (40, 4, pitch if side == "x" else 1024), -1, 1), support.uniform(4, 2, (40, 1024, pitch % 100 + 64 if side == "w" else 64), -1, 1)
    (hx, dx), (hw, dw) = (support.both(v.astype(np.float16), ta.float16, device) for v in (x, w))
    views = [(a[:, :, first:first + 1024] if side == "x" else a, b[:, :, first:first + 64] if side == "w" else b) for a, b in ((hx, hw), (dx, dw))]
    assert lanes_of(*views[1]) == 4
    check(ops.matmul(*views[1]), ops.matmul(*views[0]).numpy(), ta.float16, 1024, side)


@pytest.mark.parametrize("first", [0, 1])
def test_views_and_what_lies_beside_them(first, device):
    """Slices of tensors full of infinities that start at any element, W broadcast over a batch dimension."""
    x, w = np.full((2, 50, 6, 1010), np.inf, np.float16), np.full((1, 50, 1010, 30), np.inf, np.float16)
    x[:, :, 1:5, first:first + 1003] = support.uniform(9, 1, (2, 50, 4, 1003), -1, 1)
    w[:, :, 3:1006, first:first + 24] = support.uniform(9, 2, (1, 50, 1003, 24), -1, 1)
    (hx, dx), (hw, dw) = support.both(x, ta.float16, device), support.both(w, ta.float16, device)
    want, got = (ops.matmul(a[:, :, 1:5, first:first + 1003], b[:, :, 3:1006, first:first + 24]) for a, b in ((hx, hw), (dx, dw)))
    check(got, want.numpy(), ta.float16, 1003, "views")
