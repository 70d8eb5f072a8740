// One row times a matrix whose rows are contiguous along K (two rows of fp32): y = x * W^T as decoding one sequence runs it.
//
// The work is reading W once.  The kernel beside it (gemm_skinny_stream_kernel) reads 128 bytes of sixteen rows at a time, through LDS into
// matrix fragments of which one row in sixteen is used, with one block of four wavefronts on a compute unit.  Here a wavefront owns a row of W: a load
// instruction is a kilobyte of it, eight of them are on their way while the eight before are multiplied, six blocks (five of two fp32 rows)
// share a compute unit by their registers, and x waits in LDS.  Bound by HBM, 6.5 TB/s of W where it is large (8 multiply-adds and their conversions for 16 bytes are a third of the
// time; two rows of 16-bit values are not worth it: 28672 x 4096 40.8 there, 44.0 here).  One row, W from memory, us there / here: bf16
// 6144 x 4096 13.1 / 10.9, 28672 x 4096 40.5 / 36.0, 32000 x 2048 28.7 / 23.2, 12000 x 5000 30.6 / 22.5, 512 x 16384 12.8 / 8.8, fp32 4096 x 4096
// 18.4 / 14.8, 14336 x 4096 51.0 / 38.3, 1024 x 1024 5.4 / 4.1, two rows 4096 x 4096 18.4 / 16.0.  (src/cpu/matmul.cpp:36-60)
#include "gemm_common.hpp"
#include "lanes.hpp"

namespace th {

typedef unsigned int uint4d __attribute__((ext_vector_type(4)));

struct AddF {
    static __device__ inline float combine(float a, float b) { return a + b; }
};

constexpr int kDotWaves = 4, kDotUnroll = 8;
constexpr size_t kDotLds = 64 * 1024;

// MR rows of x
template <class T, int MR>
__global__ __launch_bounds__(64 * kDotWaves) void gemm_rows_dot_kernel(const T* x, const T* w, T* y, GemmProblem p, bool streamed) {
    constexpr uint32_t CH = 16 / sizeof(T), U = kDotUnroll;
    extern __shared__ __align__(16) unsigned char rows_dot_lds[];
    int64_t ox, ow, oc;
    batch_offsets(p, blockIdx.y, ox, ow, oc);
    const uint32_t lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const uint32_t n = blockIdx.x * kDotWaves + wave;
    const T* const row = w + ow + static_cast<int64_t>(n < p.N ? n : p.N - 1) * p.b_cs;      // (rows past the end are never stored)
    const uint32_t chunks = p.K / CH;      // 16-byte pieces of a row
    auto piece = [&](uint32_t c) { return c + lane < chunks ? c + lane : chunks - 1; };
    auto load = [&](uint4d (&into)[U], uint32_t first) {
        // (the empty statements keep the loads apart, which the compiler would merge into some through the caches)
        if (streamed) {
            asm volatile("");
#pragma unroll
            for (uint32_t u = 0; u < U; ++u) into[u] = __builtin_nontemporal_load(reinterpret_cast<const uint4d*>(row) + piece(first + u * 64));
            asm volatile("");
        } else {
#pragma unroll
            for (uint32_t u = 0; u < U; ++u) into[u] = reinterpret_cast<const uint4d*>(row)[piece(first + u * 64)];
        }
    };
    uint4d bits[U];
    load(bits, 0);
    // x meanwhile
    uint4d* const staged = reinterpret_cast<uint4d*>(rows_dot_lds);
#pragma unroll
    for (int m = 0; m < MR; ++m)
        for (uint32_t c = threadIdx.x; c < chunks; c += 64 * kDotWaves)
            staged[m * chunks + c] = *reinterpret_cast<const uint4d*>(x + ox + static_cast<int64_t>(m) * p.a_rs + static_cast<size_t>(c) * CH);
    __syncthreads();
    float acc[MR];
#pragma unroll
    for (int m = 0; m < MR; ++m) acc[m] = 0.0f;
    for (uint32_t first = 0; first < chunks; first += 64 * U) {
        uint4d next[U];
        if (first + 64 * U < chunks) load(next, first + 64 * U);
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            const uint32_t c = first + u * 64 + lane;
            if (c >= chunks) continue;
            T e[CH];
            __builtin_memcpy(e, &bits[u], 16);
#pragma unroll
            for (int m = 0; m < MR; ++m) {
                const uint4d here = staged[m * chunks + c];
                T f[CH];
                __builtin_memcpy(f, &here, 16);
#pragma unroll
                for (uint32_t j = 0; j < CH; ++j) acc[m] = fmaf(static_cast<float>(widen(f[j])), static_cast<float>(widen(e[j])), acc[m]);
            }
        }
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) bits[u] = next[u];
    }
#pragma unroll
    for (int m = 0; m < MR; ++m) {
        const float sum = wave_reduce<AddF>(acc[m]);
        if (lane == 0 && n < p.N) y[oc + static_cast<int64_t>(m) * p.c_rs + n] = narrow_result<T>(sum);
    }
}

// From 40 MB on.  us through the caches / past them, every W from memory, and the same W again and again: bf16 5248 x 4096 (42 MB) 11.0 / 9.9, 11.1 / 9.0;
// 8576 x 4096 15.2 / 13.7, 14.4 / 12.5; 29440 x 4096 45.3 / 40.2, 37.2 / 36.6; fp32 3072 x 4096 12.9 / 11.8, 11.9 / 10.2; 14336 x 4096 45.7 / 42.5, 37.9 / 39.2.  Below, the same W
// is as fast either way (bf16 2176 x 4096 6.3 / 6.4), and smaller ones may be a whole model's that does stay.
bool rows_dot_past_caches(const GemmProblem& p, size_t esize) { return rows_past_caches(p, esize, 40ull << 20); }

template <class T, int MR>
static int launch_rows_dot(const GemmProblem& p, const void* x, const void* w, void* y, hipStream_t stream) {
    auto kernel = gemm_rows_dot_kernel<T, MR>;
    static std::atomic<uint64_t> configured{0};
    if (int rc = raise_lds_limit(reinterpret_cast<const void*>(kernel), kDotLds, configured)) return rc;
    hipLaunchKernelGGL(kernel, dim3((p.N + kDotWaves - 1) / kDotWaves, p.batches), dim3(64 * kDotWaves), MR * p.K * sizeof(T), stream, static_cast<const T*>(x),
                       static_cast<const T*>(w), static_cast<T*>(y), p, rows_dot_past_caches(p, sizeof(T)));
    return launch_status("gemm_rows_dot_kernel");
}

// Single products.  Below K = 2048 (fp32: 1024) a wavefront's eight loads are not all used (bf16 16384 x 512 7.2 there, 8.4 here, 3072 x 1024 4.8 / 4.9); where x takes
// more than 16 KB and there are rows for every compute unit, LDS holds too few blocks (4096 x 14336 20.2 / 21.6, fp32 42.2 / 47.7).
bool gemm_rows_dot_takes(const GemmProblem& p, size_t esize) {
    if (p.M == 0 || p.M > (esize == 4 ? 2 : 1) || p.batches != 1) return false;
    const uint64_t of_x = static_cast<uint64_t>(p.M) * p.K * esize;
    // (a last turn of one to three loads takes as long as a whole one: 2361 x 4160 6.7 there, 8.1 here; the kernel there for a K of no whole windows is
    // slower still, 4500 x 4200 17.9 / 16.8)
    const uint64_t loads = (p.K * esize + 1023) / 1024, rest = loads % kDotUnroll;
    if (p.K * esize % 128 == 0 && rest > 0 && rest < 4 && loads > kDotUnroll && loads < 4 * kDotUnroll) return false;
    return p.K >= (esize == 4 ? 1024 : 2048) && of_x <= kDotLds && (of_x <= 16 * 1024 * p.M || p.N <= 2048);
}

// (the caller has seen to contiguous rows in 16-byte pieces)
template <class T>
int gemm_rows_dot(const GemmProblem& p, const void* x, const void* w, void* y, hipStream_t stream) {
    if (p.M == 1) return launch_rows_dot<T, 1>(p, x, w, y, stream);
    if constexpr (sizeof(T) == 4) return launch_rows_dot<T, 2>(p, x, w, y, stream);
    return TANNIC_UNSUPPORTED_DTYPE;
}
template int gemm_rows_dot<f16>(const GemmProblem&, const void*, const void*, void*, hipStream_t);
template int gemm_rows_dot<bf16>(const GemmProblem&, const void*, const void*, void*, hipStream_t);
template int gemm_rows_dot<float>(const GemmProblem&, const void*, const void*, void*, hipStream_t);

}  // namespace th
