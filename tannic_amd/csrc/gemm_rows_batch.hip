// Two to four rows times narrow matrices that lie row by row, 16-bit, one product per batch index:
// y[b][m][n] = sum over k of x[b][m][k] * W[b][k][n], N a multiple of 8 up to 256, K of a thousand or more.  (Attention's probabilities times the
// cached values for one new token: a group's query heads are the rows, K is the length of the context, whatever it is.)
//
// The work is reading W once.  A lane owns eight consecutive columns (one 16-byte load per row of W), LN lanes lie side by side
// along the columns and 64 / LN rows of W are one load instruction; a block's wavefronts take turns along K, UNROLL rows per
// lane in flight.  x comes value by value beside it (64 / LN consecutive k per instruction, from the cache), so its row pitch
// and K may be odd, and nothing here needs alignment.  A lane's sums meet the other rows' by halves (a reduce-scatter: 30 exchanges
// for 32 sums over 16 lanes where a butterfly takes 128), then the wavefronts' in LDS, in a fixed order; no scratch, one kernel.
// (src/cpu/matmul.cpp:60-124; fp32 sums, rounded once.)
#include "gemm_common.hpp"

namespace th {

typedef unsigned int uint4r __attribute__((ext_vector_type(4), aligned(2)));

constexpr int kRowsBatchWaves = 16;

// rows of W a lane has in flight: with few blocks a context of a few thousand is one pass
constexpr int rows_batch_unroll(int lanes) { return lanes == 2 ? 8 : 4; }

// The sums over the lanes that differ in bits LAST ... 32 of the lane number (first call: STEP = 32): N values per lane become N * LAST / 64
// finished ones, those whose number has the bits of the lane's (the upper half where the lane has bit STEP, and so on).
template <int N, int STEP, int LAST>
__device__ __forceinline__ void scatter_sums(float* v, uint32_t lane) {
    if constexpr (STEP >= LAST) {
        const bool upper = (lane & STEP) != 0;
#pragma unroll
        for (int i = 0; i < N / 2; ++i) {
            const float keep = upper ? v[i + N / 2] : v[i], send = upper ? v[i] : v[i + N / 2];
            v[i] = keep + __shfl_xor(send, STEP, 64);
        }
        scatter_sums<N / 2, STEP / 2, LAST>(v, lane);
    }
}

template <class T, int LN>
__global__ __launch_bounds__(64 * kRowsBatchWaves) void gemm_rows_batch_kernel(const T* x, const T* w, T* y, GemmProblem p) {
    constexpr int MR = 4;   // rows a lane accumulates, at least M
    constexpr int ROWS = 64 / LN, UNROLL = rows_batch_unroll(LN);
    constexpr int LEFT = MR * 8 / ROWS;   // finished sums per lane
    static_assert(LEFT >= 1, "every lane ends with a sum");
    __shared__ float part[kRowsBatchWaves][64 * LEFT];
    const uint32_t lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), waves = blockDim.x / 64;
    // (workgroups go round the eight dies in turn: with whole eights of products, those that share a product's rows share a die)
    const uint32_t batch = blockIdx.x % p.batches, group = blockIdx.x / p.batches;
    int64_t oa, ob, oc;
    batch_offsets(p, batch, oa, ob, oc);
    const uint32_t col = (group * LN + lane % LN) * 8, row = lane / LN;
    const bool active = col < p.N;   // (N is a multiple of 8)
    const T* wp = w + ob + (active ? col : 0);
    const T* xp[MR];
#pragma unroll
    for (int m = 0; m < MR; ++m) xp[m] = x + oa + static_cast<int64_t>(static_cast<uint32_t>(m) < p.M ? m : 0) * p.a_rs;   // (rows past M are never stored)

    float acc[MR * 8];
#pragma unroll
    for (int i = 0; i < MR * 8; ++i) acc[i] = 0.0f;
    for (uint32_t k0 = wave * ROWS * UNROLL; k0 < p.K; k0 += waves * ROWS * UNROLL) {
        uint4r bits[UNROLL];
        T xv[UNROLL][MR];
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
            const uint32_t k = k0 + u * ROWS + row;
            const bool live = k < p.K;
            bits[u] = uint4r{0, 0, 0, 0};
            if (live) bits[u] = *reinterpret_cast<const uint4r*>(wp + static_cast<int64_t>(k) * p.b_rs);
#pragma unroll
            for (int m = 0; m < MR; ++m) {
                xv[u][m] = T{};
                if (live) xv[u][m] = xp[m][static_cast<int64_t>(k) * p.a_cs];
            }
        }
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
            T e[8];
            __builtin_memcpy(e, &bits[u], 16);
            float wide[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) wide[i] = static_cast<float>(widen(e[i]));
#pragma unroll
            for (int m = 0; m < MR; ++m) {
                const float f = static_cast<float>(widen(xv[u][m]));
#pragma unroll
                for (int i = 0; i < 8; ++i) acc[m * 8 + i] += f * wide[i];
            }
        }
    }
    scatter_sums<MR * 8, 32, LN>(acc, lane);
#pragma unroll
    for (int i = 0; i < LEFT; ++i) part[wave][i * 64 + lane] = acc[i];
    __syncthreads();
    for (uint32_t at = threadIdx.x; at < 64 * LEFT; at += blockDim.x) {
        // sum `at` is the (at / 64)th that lane at % 64 finished: row value / 8, column value % 8 of that lane's eight
        float sum = 0.0f;
        for (uint32_t v = 0; v < waves; ++v) sum += part[v][at];
        const uint32_t from = at % 64;
        uint32_t value = at / 64;
#pragma unroll
        for (int step = 32, half = MR * 4; step >= LN; step /= 2, half /= 2) value += from & step ? half : 0;
        const uint32_t m = value / 8, n = (group * LN + from % LN) * 8 + value % 8;
        if (m < p.M && n < p.N) y[oc + static_cast<int64_t>(m) * p.c_rs + n] = narrow_result<T>(sum);
    }
}

template <class T, int LN>
static int launch_rows_batch(const GemmProblem& p, const void* x, const void* w, void* y, hipStream_t stream) {
    constexpr uint32_t per_wave = 64 / LN * rows_batch_unroll(LN);   // rows of W a wavefront has in flight
    const uint32_t groups = (p.N + 8 * LN - 1) / (8 * LN);
    uint32_t waves = (p.K + per_wave - 1) / per_wave;
    if (waves > kRowsBatchWaves) waves = kRowsBatchWaves;
    hipLaunchKernelGGL((gemm_rows_batch_kernel<T, LN>), dim3(groups * p.batches), dim3(64 * waves), 0, stream, static_cast<const T*>(x), static_cast<const T*>(w),
                       static_cast<T*>(y), p);
    return launch_status("gemm_rows_batch_kernel");
}

// The same for a handful of products (few results: at most 8192), where the latency of one pass over K is the time.  Two lanes side by
// side, so that there are blocks enough; a block's sixteen wavefronts have all of a pass, 4096 rows of W, on their way at once, and x goes
// through LDS meanwhile as [k][row] in fp32: one read per k for the four rows (value by value from the cache, four loads of two bytes
// beside every 16-byte load of W, the path to the cache was as long as the latency).  Eight products of 4 x 128 under 2049: 14.1 us on
// the kernel for few results before (a workgroup per 4 x 4 results, W's lines 32 times), 8.9 here (one lane, twice the blocks: 9.4);
// 4 x 128 under 4001 19.5 / 10.8, sixteen of 4 x 128 under 1025 13.5 / 7.8, one row of 64 columns under 3000 13.6 / 9.1.
constexpr int kRowsFewUnroll = 8;
constexpr uint32_t kRowsFewPass = 32 * kRowsFewUnroll * kRowsBatchWaves;    // rows of W a block has in flight
template <class T>
__global__ __launch_bounds__(64 * kRowsBatchWaves) void gemm_rows_few_kernel(const T* x, const T* w, T* y, GemmProblem p) {
    constexpr int MR = 4, LN = 2, ROWS = 64 / LN, UNROLL = kRowsFewUnroll;
    __shared__ float part[kRowsBatchWaves][64];
    extern __shared__ __align__(16) unsigned char rows_few_lds[];
    float4* values = reinterpret_cast<float4*>(rows_few_lds);
    const uint32_t lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), waves = blockDim.x / 64;
    // (workgroups go round the eight dies in turn: with whole eights of products, those that share a product's lines share a die)
    const uint32_t batch = blockIdx.x % p.batches, group = blockIdx.x / p.batches;
    int64_t oa, ob, oc;
    batch_offsets(p, batch, oa, ob, oc);
    const uint32_t col = (group * LN + lane % LN) * 8, row = lane / LN;
    const T* wp = w + ob + (col < p.N ? col : 0);   // (N is a multiple of 8; columns past it are never stored)
    const T* xp[MR];
#pragma unroll
    for (int m = 0; m < MR; ++m) xp[m] = x + oa + static_cast<int64_t>(static_cast<uint32_t>(m) < p.M ? m : 0) * p.a_rs;   // (rows past M are never stored)
    float acc[MR * 8];
#pragma unroll
    for (int i = 0; i < MR * 8; ++i) acc[i] = 0.0f;
    for (uint32_t first = 0; first < p.K; first += kRowsFewPass) {
        const uint32_t here = p.K - first < kRowsFewPass ? p.K - first : kRowsFewPass;
        const uint32_t k0 = wave * ROWS * UNROLL + row;
        uint4r bits[UNROLL];
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
            const uint32_t k = k0 + u * ROWS;
            bits[u] = uint4r{0, 0, 0, 0};
            if (k < here) bits[u] = *reinterpret_cast<const uint4r*>(wp + static_cast<int64_t>(first + k) * p.b_rs);
        }
        if (first) __syncthreads();     // the pass before has been read
        for (uint32_t k = threadIdx.x; k < here; k += blockDim.x)
            values[k] = float4{static_cast<float>(widen(xp[0][first + k])), static_cast<float>(widen(xp[1][first + k])), static_cast<float>(widen(xp[2][first + k])),
                               static_cast<float>(widen(xp[3][first + k]))};
        __syncthreads();
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
            const uint32_t k = k0 + u * ROWS;
            const float4 v = k < here ? values[k] : float4{0.0f, 0.0f, 0.0f, 0.0f};
            const float f[MR] = {v.x, v.y, v.z, v.w};
            T e[8];
            __builtin_memcpy(e, &bits[u], 16);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float wide = static_cast<float>(widen(e[i]));
#pragma unroll
                for (int m = 0; m < MR; ++m) acc[m * 8 + i] += f[m] * wide;
            }
        }
    }
    scatter_sums<MR * 8, 32, LN>(acc, lane);
    part[wave][lane] = acc[0];
    __syncthreads();
    if (threadIdx.x < 64) {
        float sum = 0.0f;
        for (uint32_t v = 0; v < waves; ++v) sum += part[v][lane];
        uint32_t value = 0;
#pragma unroll
        for (int step = 32, half = MR * 4; step >= LN; step /= 2, half /= 2) value += lane & step ? half : 0;
        const uint32_t m = value / 8, n = (group * LN + lane % LN) * 8 + value % 8;
        if (m < p.M && n < p.N) y[oc + static_cast<int64_t>(m) * p.c_rs + n] = narrow_result<T>(sum);
    }
}

// Few results of row-major matrices under a long K; above 8192 results the tiles and the kernel above have work enough.
static bool rows_few_takes(const GemmProblem& p) {
    if (p.M == 0 || p.M > 4 || p.N == 0 || p.N % 8 != 0 || p.K < 512 || p.K >= (1u << 31) || p.a_cs != 1 || p.b_cs != 1 || p.b_rs == 1 || p.row_bias || p.c_group || p.b_group_stride)
        return false;
    if (static_cast<uint64_t>(p.N) * p.batches * p.M > 8192) return false;
    // Rows of W that are an odd number of 16-byte pieces: a block's 32 bytes of one lie in two lines every other time, and fewer than 64 blocks
    // under a long K are bound by the lines each has on its way (bf16, four rows, us on the kernel for few results / here, W in no cache: 104
    // columns under 8192 22 / 27, 200 under 16384 39 / 50, two products 39 / 49, four 43 / 50; W in the caches 200 under 16384 33.4 / 35.6, 72 32 / 35, but
    // 200 under 4096 14 / 12, 72 under 8192 15 / 13, two products 20 / 13; up to 64 columns from 32768 on, 40 under 65536 75 / 84, under 16384 23 / 19;
    // rows of an even number, under 16384: 192 columns 45 / 46, two products of 128 46 / 44).  And a last pass over less than 1024 rows costs nearly what a whole one does (two products of 72 columns under 4200 13.7 / 15.4, 6 of 40 12.0 / 13.2,
    // two of 88 under 8250 20.2 / 22.2; under 5200 ten of 40 13.7 / 13.7, under 3000 72 12.8 / 11.4).  The kernel for few results does these in one round
    // of workgroups; in two it takes twice as long (five products of 200 under 18417 53 / 57, six 94 / 58; twenty of 56 under 4200 22.2 / 14.6).
    if (p.N % 16 == 0 || p.N == 8 || static_cast<uint64_t>((p.N + 3) / 4) * p.batches > 256) return true;
    const uint32_t last = p.K % kRowsFewPass;
    return p.K < (p.N > 96 ? 6144u : p.N > 64 ? 12288u : 32768u) && (p.K <= kRowsFewPass || last == 0 || last >= 1024);
}

bool gemm_rows_few_takes(const GemmProblem& p, int dtype) {
    return (dtype == TANNIC_FLOAT16 || dtype == TANNIC_BFLOAT16) && rows_few_takes(p);
}

template <class T>
static int run_rows_few(const GemmProblem& p, const void* x, const void* w, void* y, hipStream_t stream) {
    constexpr uint32_t per_wave = 32 * kRowsFewUnroll;
    uint32_t waves = (p.K + per_wave - 1) / per_wave;
    if (waves > kRowsBatchWaves) waves = kRowsBatchWaves;
    const size_t lds = static_cast<size_t>(p.K < kRowsFewPass ? p.K : kRowsFewPass) * 16;
    auto kernel = gemm_rows_few_kernel<T>;
    static std::atomic<uint64_t> configured{0};
    if (int rc = raise_lds_limit(reinterpret_cast<const void*>(kernel), kRowsFewPass * 16, configured)) return rc;
    hipLaunchKernelGGL(kernel, dim3((p.N + 15) / 16 * p.batches), dim3(64 * waves), lds, stream, static_cast<const T*>(x), static_cast<const T*>(w), static_cast<T*>(y), p);
    return launch_status("gemm_rows_few_kernel");
}

int gemm_rows_few(const GemmProblem& p, int dtype, const void* a, const void* b, void* c, hipStream_t stream) {
    if (!rows_few_takes(p)) return TANNIC_UNSUPPORTED_DTYPE;
    if (dtype == TANNIC_FLOAT16) return run_rows_few<f16>(p, a, b, c, stream);
    if (dtype == TANNIC_BFLOAT16) return run_rows_few<bf16>(p, a, b, c, stream);
    return TANNIC_UNSUPPORTED_DTYPE;
}

// Which of the kernels takes a product: its lanes side by side along the columns, or 0 where none does.
//
// They are taken where the tiles would read an operand at any alignment (K, or a pitch or an address of x or W, that no 16 bytes divide)
// and there are more results than the kernel for few results takes, up to one block of 32 columns per compute unit - two where the
// columns are whole blocks of aligned rows.  bf16, four rows, replayed calls, us here / before:
//   one block a unit   32 products of 1001 x 128 7.0 / 15.9, 64 of 2049 x 128 12.6 / 33.2, 128 of 4001 x 64 23.2 / 58.4, 85 of 1001 x 72 10.9 / 16.1,
//                      64 of 1024 x 128 with an odd pitch of x 7.2 / 15.1, of W 7.7 / 15.0
//   ragged, more       113 of 1001 x 72 18.1 / 16.2, 78 of 1001 x 104 18.8 / 16.0
//   two a unit         72 of 2049 x 128 18.5 / 33.4, 96 of it 23.1 / 33.7, 128 of it 23.7 / 34.0, of 1001 x 128 14.4 / 19.0
//   three a unit       192 of 1001 x 128 21.6 / 20.0, of 2049 x 128 38.8 / 34.7
//   aligned, on tiles  64 of 2048 x 128 12.2 / 11.6, of 4000 x 128 21.5 / 16.8
// (Up to 64 columns a tile of the product is half empty, and up to 8192 columns in all are taken: 204 of 1001 x 40 13.4 / 17.3.  A K
// below 1000 is not taken, although 64 of 513 x 128 ran in 6.0 against 11.1.)
// Lanes: four, 64-byte runs of a row (64 of 2049 x 128 12.6, with two 19.2; 85 of 1001 x 72 10.9, 16.6), but two where the columns are no
// more than two lanes', or three times two lanes' in more than a round (131 of 2007 x 48 19.4 against 25.5), or a long K is shared by too
// few blocks (32 of 4001 x 128 14.4 against 19.2, of 2049 x 128 9.2 against 9.4).
static uint32_t rows_batch_lanes(const GemmProblem& p, const void* x, const void* w) {
    if (p.M < 2 || p.M > 4 || p.N == 0 || p.N > 256 || p.N % 8 != 0 || p.K < 1000 || p.K >= (1u << 31)) return 0;
    if (p.a_cs != 1 || p.b_cs != 1 || p.b_rs == 1 || p.row_bias || p.c_group || p.b_group_stride) return 0;
    bool x_aligned = p.a_rs % 8 == 0 && reinterpret_cast<uintptr_t>(x) % 16 == 0, w_aligned = p.b_rs % 8 == 0 && reinterpret_cast<uintptr_t>(w) % 16 == 0;
    for (int d = 0; d < p.batch_rank; ++d) {
        x_aligned = x_aligned && p.a_bs[d] % 8 == 0;
        w_aligned = w_aligned && p.b_bs[d] % 8 == 0;
    }
    if (p.K % 8 == 0 && x_aligned && w_aligned) return 0;
    const uint64_t columns = static_cast<uint64_t>(p.N) * p.batches, blocks = static_cast<uint64_t>((p.N + 31) / 32) * p.batches;
    if (columns * p.M <= 8192) return 0;
    if (blocks > (p.N % 32 == 0 && w_aligned ? 512 : 256) && !(p.N <= 64 && columns <= 8192)) return 0;
    if (p.N > 32 && p.N <= 48 && blocks > 256) return 2;
    return p.N <= 16 || (p.K > 3000 && (p.N + 15) / 16 * static_cast<uint64_t>(p.batches) <= 256) ? 2 : 4;
}

uint32_t gemm_rows_batch_lanes(const GemmProblem& p, int dtype, const void* a, const void* b) {
    return dtype == TANNIC_FLOAT16 || dtype == TANNIC_BFLOAT16 ? rows_batch_lanes(p, a, b) : 0;
}

template <class T>
static int run_rows_batch(const GemmProblem& p, const void* x, const void* w, void* y, hipStream_t stream) {
    const uint32_t lanes = rows_batch_lanes(p, x, w);
    if (lanes == 0) return TANNIC_UNSUPPORTED_DTYPE;
    return lanes == 4 ? launch_rows_batch<T, 4>(p, x, w, y, stream) : launch_rows_batch<T, 2>(p, x, w, y, stream);
}

int gemm_rows_batch(const GemmProblem& p, int dtype, const void* a, const void* b, void* c, hipStream_t stream) {
    if (dtype == TANNIC_FLOAT16) return run_rows_batch<f16>(p, a, b, c, stream);
    if (dtype == TANNIC_BFLOAT16) return run_rows_batch<bf16>(p, a, b, c, stream);
    return TANNIC_UNSUPPORTED_DTYPE;
}

}  // namespace th
