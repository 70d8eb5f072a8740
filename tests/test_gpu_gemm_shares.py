"""Products of a few hundred rows under a long K, at the sizes where their tiles end: tiles of 128 x 96, and tiles of 256 x 128 whose K is
shared between blocks.

Bar: a matrix instruction adds 32 products to an fp32 sum, so a product is followed by at most K / 32 + 32 additions, and the sum is rounded
once."""
import numpy as np
import pytest

import tannic_amd as ta
from tannic_amd import ops

pytestmark = pytest.mark.gpu

EPS = {ta.float16: 2.0 ** -11, ta.bfloat16: 2.0 ** -8}

# M, N, K: rows that end in a tile's first half, its last row or with it, columns that end in a tile of 96 or in a piece of eight, K of whole
# steps that the stages do not divide
NARROW = [(129, 6144, 2112), (385, 5128, 1536), (201, 8789, 1536), (326, 5454, 1600), (65, 22000, 2048), (768, 3000, 1536), (512, 6144, 2048)]
# and shares of K of different lengths
SHARED = [(256, 4096, 20544), (250, 4092, 20544), (512, 4092, 10304), (511, 4084, 14400), (1020, 2044, 10368)]
# and what goes to the 64-row tiles beside them
BESIDE = [(300, 6150, 1600), (300, 6150, 2112)]


@pytest.mark.parametrize("dtype", [ta.float16, ta.bfloat16], ids=str)
@pytest.mark.parametrize("m,n,k", NARROW + SHARED + BESIDE)
def test_tiles_of_long_products(m, n, k, dtype, device):
    """Both matrices are parts of larger ones; what lies beside them is infinite."""
    rng = np.random.default_rng(7)
    x, w = np.full((m, k + 8), np.inf, np.float32), np.full((n, k + 16), np.inf, np.float32)
    x[:, :k], w[:, :k] = rng.standard_normal((m, k), np.float32), rng.standard_normal((n, k), np.float32) * 0.02
    x, w = ta.tensor(x, dtype, device)[:, 0:k], ta.tensor(w, dtype, device)[:, 0:k]
    got = ops.matmul(x, w.transpose()).numpy().astype(np.float64)
    a, b = x.numpy().astype(np.float64), w.numpy().astype(np.float64)
    want = a @ b.T
    bound = EPS[dtype] * np.abs(want) + (k / 32 + 32) * 2.0 ** -24 * (np.abs(a) @ np.abs(b).T)
    assert (np.abs(got - want) <= bound).all()
