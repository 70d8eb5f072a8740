"""Which 16-bit products of a few rows with narrow row-major matrices run on the kernel for them, asked of the library without a GPU
(``tannic_hip_gemm_rows_batch_lanes``), and which tiles those of a few hundred rows (``tannic_hip_gemm_plan``): the products of the GPU
tests are the kernels' that these name."""
import ctypes as C

import pytest

import tannic_amd as ta
import test_gpu_decode_ops
import test_gpu_gemm_rows_dot
import test_gpu_gemm_shares
from tannic_amd import abi
from test_conv_plan import descriptor


def lanes(batches, m, n, k, x_pitch=None, w_pitch=None, x_start=0):
    x, w, y = (descriptor("bfloat16", s) for s in ((batches, m, k), (batches, k, n), (batches, m, n)))
    for t, rows, pitch in ((x, m, x_pitch), (w, k, w_pitch)):
        if pitch:
            t.strides.sizes[0], t.strides.sizes[1] = rows * pitch, pitch
    x.address += 2 * x_start
    return ta.library().gemm_rows_batch_lanes(x, w, y)


# batches, M, N, K -> lanes
PRODUCTS = {
    "one_block_a_unit": ((64, 4, 128, 2049), 4),
    "a_product_less": ((63, 4, 128, 2049), 4),
    "two_blocks_a_unit": ((128, 4, 128, 2049), 4),
    "more_than_two": ((129, 4, 128, 2049), 0),
    "ragged_columns_one_block": ((85, 4, 72, 1001), 4),
    "ragged_columns_more": ((113, 4, 72, 1001), 0),
    "ragged_columns_of_104": ((78, 4, 104, 2049), 0),
    "half_a_tile": ((204, 4, 40, 1001), 2),
    "half_a_tile_one_block": ((128, 4, 40, 1001), 4),
    "eight_columns": ((1024, 4, 8, 1001), 2),
    "long_k_few_blocks": ((32, 4, 128, 4001), 2),
    "long_k_more_blocks": ((33, 4, 128, 4001), 4),
    "few_results": ((16, 4, 128, 2049), 0),
    "one_row": ((80, 1, 128, 2049), 0),
    "aligned": ((64, 4, 128, 2048), 0),
}


@pytest.mark.parametrize("name", list(PRODUCTS))
def test_products(name):
    problem, want = PRODUCTS[name]
    assert lanes(*problem) == want


def test_alignment_is_of_rows_and_addresses():
    """K a multiple of eight is no alignment: a pitch or a start that no 16 bytes divide sends the tiles to their slower loaders."""
    assert lanes(64, 4, 128, 2048, x_pitch=2056) == 0
    assert lanes(64, 4, 128, 2048, x_pitch=2049) == 4
    assert lanes(64, 4, 128, 2048, x_start=1) == 4
    assert lanes(64, 4, 128, 2048, w_pitch=129) == 4
    assert lanes(128, 4, 128, 2048, w_pitch=129) == 0


def product_plan(batches, m, n, k, dtype="bfloat16"):
    out = (C.c_uint32 * 4)()
    assert ta.library().gemm_plan(*(C.byref(descriptor(dtype, s)) for s in ((batches, m, k), (batches, k, n), (batches, m, n))), out) == abi.SUCCESS
    return tuple(out)


# batches, M, N, K of a few rows times row-major matrices with few results -> whether the kernel for them takes it
FEW_RESULTS = {
    "decoding": ((8, 4, 128, 2049), True),
    "shortest": ((1, 1, 8, 512), True),
    "shorter": ((1, 1, 8, 511), False),
    "most_results": ((16, 4, 128, 4096), True),
    "more_results": ((17, 4, 128, 4096), False),
    "five_rows": ((8, 5, 128, 4096), False),
    "columns_of_no_pieces": ((8, 4, 124, 4096), False),
    # rows of an odd number of pieces under a long K
    "odd_pieces": ((1, 4, 200, 6136), True),
    "odd_pieces_long_k": ((1, 4, 200, 6144), False),
    "odd_pieces_long_k_four_products": ((4, 4, 200, 16384), False),
    "odd_pieces_long_k_more_blocks": ((8, 4, 200, 16384), True),
    "fewer_odd_pieces": ((1, 4, 72, 12280), True),
    "fewer_odd_pieces_long_k": ((1, 4, 72, 12288), False),
    "even_pieces_long_k": ((1, 4, 192, 65536), True),
    "few_odd_pieces": ((1, 4, 40, 32760), True),
    "few_odd_pieces_long_k": ((1, 4, 40, 32768), False),
    "one_piece": ((1, 4, 8, 200000), True),
    # and a short last pass of 4096 rows
    "odd_pieces_one_pass": ((2, 2, 72, 4096), True),
    "odd_pieces_short_pass": ((2, 2, 72, 4097), False),
    "odd_pieces_shorter_pass": ((2, 2, 72, 5119), False),
    "odd_pieces_longer_pass": ((2, 2, 72, 5120), True),
    "odd_pieces_short_third_pass": ((2, 1, 88, 8250), False),
    "odd_pieces_short_pass_more_blocks": ((15, 1, 72, 4200), True),
    "odd_pieces_short_pass_fewer_blocks": ((14, 1, 72, 4200), False),
    "even_pieces_short_pass": ((2, 2, 80, 4200), True),
}


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("name", list(FEW_RESULTS))
def test_few_results_of_row_major_matrices(name, dtype):
    problem, taken = FEW_RESULTS[name]
    assert (product_plan(*problem, dtype)[0] == 2) == taken


def plan_of(x, w, y):
    out = (C.c_uint32 * 4)()
    assert ta.library().gemm_plan(C.byref(x), C.byref(w), C.byref(y), out) == abi.SUCCESS
    return tuple(out)


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("batch,m,n,k", test_gpu_decode_ops.PRODUCTS + test_gpu_decode_ops.BESIDE)
def test_few_results_on_the_gpu_are_that_kernel(batch, m, n, k, dtype):
    x, w, y = (descriptor(dtype, s) for s in ((batch, m, k), (batch, k, n), (batch, m, n)))
    x.address += 2
    x.strides.sizes[:2] = m * (k + 3), k + 3
    w.strides.sizes[0] = (k + 7) * n
    assert (plan_of(x, w, y)[0] == 2) == ((batch, m, n, k) in test_gpu_decode_ops.PRODUCTS)


# rows and columns of a tile, and whether its K is shared
TILES = {**{p: (128, 96, False) for p in test_gpu_gemm_shares.NARROW}, **{p: (256, 128, True) for p in test_gpu_gemm_shares.SHARED},
         **{p: (64, 128, False) for p in test_gpu_gemm_shares.BESIDE}}


# rows of the result that are no whole pieces, and a K beyond the tiles' longest, go to other tiles
NARROW_RULES = {(512, 3232, 2816): True, (437, 3944, 3200): False, (451, 2968, 2048): True, (451, 2964, 2048): False, (670, 3660, 2688): True,
                (320, 4084, 2944): False, (180, 8436, 7424): True, (512, 4352, 14336): True, (512, 4352, 14400): False}


@pytest.mark.parametrize("m,n,k", list(NARROW_RULES))
def test_narrow_tiles(m, n, k):
    x, w, y = (descriptor("bfloat16", s) for s in ((m, k), (k, n), (m, n)))
    w.strides.sizes[:2] = 1, k
    assert (plan_of(x, w, y)[2] == 96) == NARROW_RULES[m, n, k]


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("m,n,k", list(TILES))
def test_tiles_of_long_products_on_the_gpu(m, n, k, dtype):
    x, w, y = (descriptor(dtype, s) for s in ((m, k), (k, n), (m, n)))
    x.strides.sizes[0] = k + 8
    w.strides.sizes[:2] = 1, k + 16
    kernel, rows, columns, shares = plan_of(x, w, y)
    assert (kernel, rows, columns, shares > 1) == (3, *TILES[m, n, k])


# rows, columns, K (and products that share one matrix) -> the matrix is loaded past the caches.  16 bits from 40 MB on, fp32 one row (two) from 40 MB, more from
# 256 MB; a matrix that several products share counts once.
PAST_CACHES = {
    "bfloat16": [((1, 5120, 4096), 4, True), ((1, 5112, 4096), 4, False), ((2, 5120, 4096), 5, True), ((2, 5112, 4096), 5, False), ((4, 14336, 4096), 5, True),
                 ((5, 5120, 4096), 5, True), ((16, 14336, 4096), 5, True), ((32, 5112, 4096), 5, False), ((32, 26624, 4096), 5, True),
                 ((2, 1, 4096, 4096), 5, False), ((8, 4, 5112, 4096), 5, False), ((8, 4, 5120, 4096), 5, True)],
    "float32": [((1, 2560, 4096), 4, True), ((1, 2552, 4096), 4, False), ((2, 4096, 4096), 4, True), ((16, 4096, 4096), 5, False), ((4, 14336, 4096), 5, False),
                ((4, 16384, 4096), 5, True), ((8, 4, 8192, 4096), 5, False)],
}


@pytest.mark.parametrize("dtype,problem,kernel,past", [(d, *c) for d in PAST_CACHES for c in PAST_CACHES[d]], ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_matrices_of_few_rows_past_the_caches(dtype, problem, kernel, past):
    *batch, m, n, k = problem
    x, w, y = (descriptor(dtype, s) for s in ((*batch, m, k), (k, n), (*batch, m, n)))
    w.strides.sizes[:2] = 1, k
    assert plan_of(x, w, y)[:2] == (kernel, past)


def test_matrices_of_many_products_count_together():
    """Keys of 32 sequences, 8 heads each: 64 MB, every one its own product's."""
    x, w, y = (descriptor("bfloat16", s) for s in ((32, 8, 4, 1024), (32, 8, 1024, 128), (32, 8, 4, 128)))
    w.strides.sizes[:4] = 8 * 1024 * 128, 1024 * 128, 1, 1024
    assert plan_of(x, w, y)[:2] == (5, 1)


@pytest.mark.parametrize("dtype", list(test_gpu_gemm_rows_dot.SHAPES))
def test_whole_rows_on_the_gpu(dtype):
    """The products of those tests, and the one of slices, are one row's (two of fp32) times whole rows."""
    for m, n, k in test_gpu_gemm_rows_dot.SHAPES[dtype]:
        x, w, y = (descriptor(dtype, s) for s in ((m, k), (k, n), (m, n)))
        w.strides.sizes[:2] = 1, k
        assert plan_of(x, w, y)[0] == 4, (m, n, k)
    x, w, y = (descriptor("float16", s) for s in ((1, 2056), (2056, 34), (1, 34)))
    x.address, w.address = x.address + 16, w.address + 16
    x.strides.sizes[0] = 2072
    w.strides.sizes[:2] = 1, 2072
    assert plan_of(x, w, y)[0] == 4


# one row (two of fp32): the shortest K, x as long as it may be for many and for few columns, and K whose last turn of eight loads would have one to three
WHOLE_ROWS = {
    "bfloat16": [((1, 64, 2048), True), ((1, 64, 2040), False), ((2, 64, 4096), False), ((1, 2056, 8192), True), ((1, 2056, 8200), False), ((1, 2048, 8200), True),
                 ((1, 64, 32768), True), ((1, 64, 32776), False), ((1, 64, 4096), True), ((1, 64, 4160), False), ((1, 64, 5632), False), ((1, 64, 5696), True),
                 ((1, 64, 4104), True), ((1, 64, 16448), True)],
    "float32": [((1, 64, 1024), True), ((1, 64, 1016), False), ((2, 64, 1024), True), ((3, 64, 1024), False), ((2, 2056, 4096), True), ((2, 2056, 4104), False),
                ((2, 64, 8192), True), ((2, 64, 8200), False), ((1, 64, 2080), False), ((1, 64, 2848), True)],
}


@pytest.mark.parametrize("dtype,problem,taken", [(d, *c) for d in WHOLE_ROWS for c in WHOLE_ROWS[d]], ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_whole_rows(dtype, problem, taken):
    m, n, k = problem
    x, w, y = (descriptor(dtype, s) for s in ((m, k), (k, n), (m, n)))
    w.strides.sizes[:2] = 1, k
    assert (plan_of(x, w, y)[0] == 4) == taken
