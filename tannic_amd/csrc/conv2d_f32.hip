// conv2d in fp32 on v_mfma_f32_16x16x4f32: 1x1, 3x3 and 7x7 kernels, any width, alignment, stride and (3x3, 7x7) padding.
//
// The fp32 matrix pipe is sixteen times slower than the 16-bit one (2048 flops in 32 clocks), so a layer is bound by it and by
// nothing else as long as every SIMD has as much of the work as every other, and nothing makes the pipe wait.  A block of
// four wavefronts owns 32 WO output channels x 16 PT (4 / WO) output pixels of the flattened batch (WO = 1, 2 or 4
// wavefronts side by side along the channels, the others along the pixels); a wavefront's tile is 32 channels x 16 PT pixels.
//  * PT and WO are chosen per launch by the time that whole rounds of blocks take: ResNet-like layers have 98 * 2^n pixels,
//    which leaves every power-of-two tile at 49 / 64 of its last round (64 -> 64 3x3 over 56 x 56, batch 32: 3.06 tiles of
//    64 x 128 a compute unit), where PT = 13 gives 242 blocks for 256 compute units.
//  * The signal goes through LDS as it lies in memory, channel by channel, with the padding made real: a channel's plane is the
//    rows its tile touches, W + pad columns each, one pad column (or row) between two rows (images) serving both.  The loads go
//    straight to LDS, a single float per lane (16 bytes where a 1x1 kernel's images allow it); where a lane's float lies
//    is worked out once, padding is an offset past the buffer's end, which arrives as zero.  So nothing is asked of widths and
//    alignments, a tile may run over several images, and an operand value is one ds_read_b32 for any tap, stride or row:
//    no range tests and no masks next to the MFMAs.  A 1x1 kernel's plane is its sampled pixels one after the other.
//  * K = (ci, kh, kw) is walked as the weights lie in memory.  A group of 4 U kernel rows (ci, kh) is U rows for each quarter
//    of a wavefront; the block's rows of weights for a group are 16-byte pieces of OIHW, loaded to LDS beside the planes.
//    Three stages of {planes, weights}: one multiplied, one complete by the middle of the group, one on its way.
//  * Nothing but MFMAs and LDS reads in the loop (see there), and the sums of 36 or 64 products that the smaller tiles add up.
// Pixels are the MFMA's first operand: an accumulator holds four consecutive pixels of the lane's channel, stored as 16 bytes.
// With few tiles the channels are shared between `splits` blocks per tile: partial sums in fp32, added in split order
// by a second kernel.  Accumulation starts from the bias (src/cpu/conv2d.cpp:90).
// Measured, batch 32, us before (gathering tiles; products over images, unfolded or re-pitched) / here, TFLOP/s of 157 here:
//   64 -> 64 3x3 over 56 x 56 104 / 67, 111; 128 -> 128 over 28 x 28 104 / 73, 101; 256 -> 256 over 14 x 14 117 / 87, 85;
//   512 -> 512 over 7 x 7 111 / 77, 96; 64 -> 256 1x1 over 56 x 56 55 / 44, 74; 512 -> 256 over 28 x 28 76 / 61, 108;
//   256 -> 1024 over 14 x 14 44 / 36, 92; 3 -> 261 7x7 s2 over 40 x 42, batch 27, 36 / 19.  One image, 3x3: 21 / 11 ... 26 / 18.
// plan_f32 says which problems are left to the kernels before, with both sides.
// What is left: the last round of tiles, start-up (some 4 us) and the write-out of a round, which a compute unit with one block
// does not overlap with anything.
#include "conv_common.hpp"
#include "gemm_common.hpp"

namespace th {

typedef float float4c __attribute__((ext_vector_type(4)));

constexpr int kF32Threads = 256;
constexpr uint32_t kF32Outside = 0x80000000u;   // byte offset no buffer reaches: loads zero

struct F32Plan {
    uint32_t K;                     // C * KH * KW
    uint32_t pixels;                // N * HO * WO
    uint32_t ptile;                 // pixels per block
    uint32_t co_tiles, splits;
    uint32_t chunks, chunks_per_split;   // groups of kernel rows, which are chunks of channels as well
    uint32_t pitch, plane;          // floats per plane in LDS; elements of it that are loaded
    uint32_t buffer;                // floats per LDS buffer
    uint32_t hp, wp;                // rows of an image and columns of a row with the shared padding
    uint32_t hw;                    // pixels of an image
    uint32_t ragged;                // the last chunk has fewer channels than the others
    uint32_t rows64, rows256;       // whole rows of a plane in 64 and in 256 elements
    FastDiv div_hw, div_wo, div_hp, div_wp, div_pitch, div_co_tiles, div_splits;
};

template <int N, class F, int I = 0>
__device__ __forceinline__ void f32_static_for(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        f32_static_for<N, F, I + 1>(static_cast<F&&>(f));
    }
}

// After how many groups the sums of a kernel start from zero again, their values added to a second set of accumulators (0: never).
// An fp32 sum is off by some 1.8e-8 of the result's norm times the root of the additions that are chained, and the products that
// small problems ran on before share K between four wavefronts or sixteen blocks.  Chains of 36 and 64 products stay below
// theirs (512 -> 512 3x3 over 7 x 7, nine images: 4.1e-7 there, 5.7e-7 as one chain a block, 1.5e-7 here) and cost 2 - 4 % (31.6
// -> 32.7 us; 42.7 there).
// The widest tiles are chosen for problems that are one chain on every path (and have no registers for a second set); a 7x7
// kernel's K is short.
constexpr uint32_t chained_groups(int side, int u, int pt) { return pt >= 10 || side == 7 ? 0 : side == 3 ? 1 : 64 / (4 * u); }

// COUNT consecutive floats at a byte offset (all of it in the offset that the buffer's range check sees)
template <int COUNT>
__device__ inline void f32_load_run(float* out, __amdgpu_buffer_rsrc_t rsrc, uint32_t offset) {
    if constexpr (COUNT >= 4) {
        const auto v = __builtin_amdgcn_raw_buffer_load_b128(rsrc, offset, 0, 0);
        __builtin_memcpy(out, &v, 16);
        f32_load_run<COUNT - 4>(out + 4, rsrc, offset + 16);
    } else if constexpr (COUNT == 3) {
        const auto v = __builtin_amdgcn_raw_buffer_load_b96(rsrc, offset, 0, 0);
        __builtin_memcpy(out, &v, 12);
    } else if constexpr (COUNT == 2) {
        const auto v = __builtin_amdgcn_raw_buffer_load_b64(rsrc, offset, 0, 0);
        __builtin_memcpy(out, &v, 8);
    } else if constexpr (COUNT == 1) {
        const auto v = __builtin_amdgcn_raw_buffer_load_b32(rsrc, offset, 0, 0);
        __builtin_memcpy(out, &v, 4);
    }
}

// KS: the kernel's side; U: kernel rows (ci, kh) a quarter of a wavefront takes per group; PT: 16-pixel tiles per wavefront;
// NL: signal values per thread and chunk; WO: wavefronts along the output channels; WIDE: signal values come four at a time.
// RESIDENT: all channels of the tile are loaded once (few channels, a large kernel), a group is 4 rows of whatever channels,
// weights come straight from memory.  Otherwise a chunk is the channels of one group: 4 U / KS of them.
template <int KS, int U, int PT, int NL, bool RESIDENT, int WO, bool WIDE>
__global__ __launch_bounds__(kF32Threads, PT >= 10 ? 1 : 2) void conv2d_f32_kernel(const float* x, const float* w, const float* bias, float* y, float* partials, ConvProblem p, F32Plan q) {
#if defined(__HIP_DEVICE_COMPILE__)   // the host pass needs the launch stub only (and loses it over the body's device-only builtins)
    static_assert(RESIDENT ? U == 1 : U % KS == 0, "a quarter's rows are whole channels, or one row");
    constexpr int RUN = U * KS;                                   // k steps per group, weights per lane and group
    constexpr uint32_t CHANNELS = RESIDENT ? 0 : 4 * U / KS;       // per chunk
    constexpr int SIGNAL_OPS = WIDE ? NL / 4 : NL;                 // loads per wavefront and chunk
    constexpr int WEIGHT_OPS = (WO * 32 * RUN + 255) / 256;
    constexpr uint32_t SIGNAL = 256 * NL + (KS == 1 ? 0 : 128), STAGE = SIGNAL + 1024 * WEIGHT_OPS;   // floats
    typedef __attribute__((address_space(3))) void* lds_void;
    typedef const __attribute__((address_space(3))) float* lds_float;
    typedef const __attribute__((address_space(3))) float4c* lds_float4;
    extern __shared__ __align__(16) unsigned char f32_lds[];
    float* lds = reinterpret_cast<float*>(f32_lds);
    const uint32_t lds_at = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_void)(f32_lds)));

    uint32_t block = blockIdx.x;
    // workgroups go round the eight dies in turn: tiles next to each other (which share rows of the signal) on one die
    if (gridDim.x % 8 == 0) block = (block % 8) * (gridDim.x / 8) + block / 8;
    uint32_t rest, split, tile, ct;
    q.div_splits.divmod(block, rest, split);
    q.div_co_tiles.divmod(rest, tile, ct);
    const uint32_t p0 = tile * q.ptile;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64;
    const uint32_t column = lane % 16, quarter = lane / 16;
    const uint32_t wave_o = wave % WO, wave_p = wave / WO;
    const uint32_t co0 = (ct * WO + wave_o) * 32;
    const uint32_t chunk0 = split * q.chunks_per_split, chunk1 = chunk0 + q.chunks_per_split < q.chunks ? chunk0 + q.chunks_per_split : q.chunks;

    // ---- where this thread's values of a chunk come from: place `at` of the LDS buffer ----------------------
    uint32_t n0, r0, oh0, ow0;
    q.div_hw.divmod(p0, n0, r0);
    q.div_wo.divmod(r0, oh0, ow0);
    const float* image = x + static_cast<int64_t>(n0) * p.xs[0];
    const int64_t reach = (static_cast<int64_t>(p.N - 1 - n0) * p.xs[0] + static_cast<int64_t>(p.C - 1) * p.xs[1] + static_cast<int64_t>(p.H - 1) * p.xs[2] + p.W) * 4;
    const __amdgpu_buffer_rsrc_t rsrc_x =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(image), 0, static_cast<int>(reach < 0x7FFFFFFF ? reach : 0x7FFFFFFF), 0x00020000);
    // A 1x1 kernel: the sampled pixels of plane c, one after the other; turned by 16 places per quarter of a wavefront, so that
    // the quarters' reads start in different banks
    auto sampled = [&](uint32_t at) -> uint32_t {
        uint32_t c, e;
        q.div_pitch.divmod(at, c, e);
        const uint32_t turn = 16 * (c / U) % q.ptile;
        const uint32_t pixel = p0 + (e >= turn ? e - turn : e + q.ptile - turn);
        if (c >= CHANNELS || pixel >= q.pixels) return kF32Outside;
        uint32_t n, r, oh, ow;
        q.div_hw.divmod(pixel, n, r);
        int64_t offset = static_cast<int64_t>(n - n0) * p.xs[0] + static_cast<int64_t>(c) * p.xs[1];
        if constexpr (WIDE) {
            offset += r;
        } else {
            q.div_wo.divmod(r, oh, ow);
            offset += static_cast<int64_t>(oh * p.stride_h) * p.xs[2] + ow * p.stride_w;
        }
        return static_cast<uint32_t>(offset * 4);
    };
    // Larger kernels: element e of a plane is column e % wp of row e / wp.  A walk over elements `by` apart.
    struct Walk {
        uint32_t col, row, dn, e;
    };
    auto walk_from = [&](uint32_t e) {
        Walk k;
        uint32_t g;
        k.e = e;
        q.div_wp.divmod(e, g, k.col);
        q.div_hp.divmod(oh0 * p.stride_h + g, k.dn, k.row);
        return k;
    };
    auto walk_on = [&](Walk& k, uint32_t by, uint32_t rows, uint32_t cols) {      // by = rows * wp + cols
        k.e += by;
        k.col += cols;
        k.row += rows;
        if (k.col >= q.wp) {
            k.col -= q.wp;
            k.row += 1;
        }
        while (k.row >= q.hp) {
            k.row -= q.hp;
            k.dn += 1;
        }
    };
    auto place = [&](const Walk& k) -> uint32_t {
        const uint32_t ih = k.row - p.pad_h, iw = k.col - p.pad_w;   // unsigned: the padding is huge
        if (!(k.e < q.plane && n0 + k.dn < p.N && ih < p.H && iw < p.W)) return kF32Outside;
        return static_cast<uint32_t>((static_cast<int64_t>(k.dn) * p.xs[0] + static_cast<int64_t>(ih) * p.xs[2] + iw) * 4);
    };

    // ---- weights -----------------------------------------------------------------------------------------------
    const __amdgpu_buffer_rsrc_t rsrc_w = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(w), 0, static_cast<int>(p.O * q.K * 4), 0x00020000);
    float wv[2][RUN];
    // RESIDENT: a group's RUN floats of this lane's channel (of each of the two 16-channel tiles), a group ahead
    uint32_t w_from[2];
    float w_next[2][RESIDENT ? RUN : 1];
    // otherwise 16-byte pieces of the block's rows, RUN of them to a row and chunk
    uint32_t from[RESIDENT ? 1 : SIGNAL_OPS], a_from[RESIDENT ? 1 : WEIGHT_OPS];
    if constexpr (RESIDENT) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t co = co0 + i * 16 + column;
            w_from[i] = ((co < p.O ? co : p.O - 1) * q.K + quarter * RUN) * 4;
            f32_load_run<RUN>(w_next[i], rsrc_w, w_from[i] + chunk0 * (4 * RUN * 4));
        }
    } else {
        if constexpr (KS == 1) {
#pragma unroll
            for (int j = 0; j < SIGNAL_OPS; ++j) from[j] = sampled((wave * SIGNAL_OPS + j) * (WIDE ? 256 : 64) + lane * (WIDE ? 4 : 1));
        } else {
            // wavefront c loads channel c of a chunk
            static_assert(CHANNELS == 4 && !WIDE, "a channel per wavefront");
            Walk k = walk_from(lane);
            const uint32_t rows = q.rows64, cols = 64 - rows * q.wp;
#pragma unroll
            for (int j = 0; j < SIGNAL_OPS; ++j) {
                from[j] = place(k);
                if (from[j] != kF32Outside) from[j] += wave * static_cast<uint32_t>(p.xs[1] * 4);
                walk_on(k, 64, rows, cols);
            }
        }
#pragma unroll
        for (int j = 0; j < WEIGHT_OPS; ++j) {
            const uint32_t piece = (wave * WEIGHT_OPS + j) * 64 + lane, row = piece / RUN, at = piece % RUN, co = ct * (WO * 32) + row;
            a_from[j] = row < WO * 32 && co < p.O ? (co * q.K + at * 4) * 4 : kF32Outside;
        }
    }
    // Load `op` of this wavefront of a chunk into stage `to`, straight to LDS (64 lanes, consecutive places).
    auto fetch = [&](int op, uint32_t chunk, uint32_t to) __attribute__((always_inline)) {
        if (op < WEIGHT_OPS) {
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_w, (lds_void)(lds + to + SIGNAL + (wave * WEIGHT_OPS + op) * 256), 16, a_from[op], chunk * (4 * RUN * 4), 0, 0);
        } else {
            const int j = op - WEIGHT_OPS;
            const uint32_t at = KS == 1 ? (wave * SIGNAL_OPS + j) * (WIDE ? 256 : 64) : wave * q.pitch + j * 64;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_x, (lds_void)(lds + to + at), WIDE ? 16 : 4, from[j], chunk * CHANNELS * static_cast<uint32_t>(p.xs[1] * 4), 0, 0);
        }
    };
    // The last chunk may have fewer channels: what belongs to none of them becomes an offset that no buffer reaches, zero.
    auto end_of_channels = [&] {
        const uint32_t channels = p.C - (q.chunks - 1) * CHANNELS;
        if constexpr (!RESIDENT) {
#pragma unroll
            for (int j = 0; j < SIGNAL_OPS; ++j) {
                const uint32_t at = KS == 1 ? (wave * SIGNAL_OPS + j) * (WIDE ? 256 : 64) + lane * (WIDE ? 4 : 1) : wave * q.pitch;
                if (at >= channels * q.pitch) from[j] = kF32Outside;
            }
#pragma unroll
            for (int j = 0; j < WEIGHT_OPS; ++j)
                if (((wave * WEIGHT_OPS + j) * 64 + lane) % RUN * 4 >= channels * KS * KS) a_from[j] = kF32Outside;
        }
    };
    constexpr int OPS = WEIGHT_OPS + SIGNAL_OPS;
    if constexpr (!RESIDENT) {
        if (q.ragged && chunk0 + 1 == q.chunks) end_of_channels();
#pragma unroll
        for (int op = 0; op < OPS; ++op) fetch(op, chunk0, 0);
        if (chunk0 + 1 < chunk1) {
            if (q.ragged && chunk0 + 2 == q.chunks) end_of_channels();
#pragma unroll
            for (int op = 0; op < OPS; ++op) fetch(op, chunk0 + 1, STAGE);
        }
    }

    // ---- this lane's pixels: where their windows begin in a plane, for every kernel row of a quarter's group (3x3) ---------
    constexpr int ROWS = RESIDENT || KS == 1 ? 1 : KS;
    uint32_t base[ROWS][PT];      // bytes
#pragma unroll
    for (int j = 0; j < PT; ++j) {
        const uint32_t mine = wave_p * (16 * PT) + j * 16 + column;
        uint32_t start;
        if constexpr (KS == 1) {
            const uint32_t turned = mine + 16 * quarter % q.ptile;
            start = (turned < q.ptile ? turned : turned - q.ptile) + quarter * U * q.pitch;
        } else {
            const uint32_t pixel = p0 + mine < q.pixels ? p0 + mine : q.pixels - 1;
            uint32_t n, r, oh, ow;
            q.div_hw.divmod(pixel, n, r);
            q.div_wo.divmod(r, oh, ow);
            start = ((n - n0) * q.hp + oh * p.stride_h - oh0 * p.stride_h) * q.wp + ow * p.stride_w;
            if constexpr (!RESIDENT) start += quarter * (U / KS) * q.pitch;
        }
#pragma unroll
        for (int u = 0; u < ROWS; ++u) base[u][j] = lds_at + (start + u * q.wp) * 4;
    }

    // accumulators start from the bias of their channel: (i, j) -> channel i * 16 + column, value v -> pixel 4 * quarter + v
    float4c acc[2][PT];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const uint32_t co = co0 + i * 16 + column;
        const float b = (p.has_bias && split == 0 && co < p.O) ? bias[static_cast<int64_t>(co) * p.bs] : 0.0f;
#pragma unroll
        for (int j = 0; j < PT; ++j) acc[i][j] = float4c{b, b, b, b};
    }

    if constexpr (RESIDENT) {
        // the last group's rows may lie past the last channel: a plane of zeros
        Walk k = walk_from(threadIdx.x);
        const uint32_t rows = q.rows256, cols = 256 - rows * q.wp;
        for (; k.e < q.pitch; walk_on(k, 256, rows, cols)) {
            const uint32_t offset = place(k);
            for (uint32_t c = 0; c * q.pitch < q.buffer; ++c) {
                const uint32_t at = offset != kF32Outside && c < p.C ? offset + c * static_cast<uint32_t>(p.xs[1] * 4) : kF32Outside;
                lds[c * q.pitch + k.e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc_x, at, 0, 0));
            }
        }
        __syncthreads();
    } else {
        if (chunk0 + 1 < chunk1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(OPS) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    }

    // The loop.  A vector instruction between two fp32 MFMAs of a wavefront holds the matrix pipe up (14 clocks for the
    // first one, 4 for each that follows; measured with a loop of pairs of MFMAs: 66.5 clocks a pair, 80.5 with one addition, 67 with
    // a read of LDS), so the loop has next to none: addresses are registers plus an immediate, moved on to the next stage once a
    // group, all in one place, and operands are replaced in their registers as soon as their last MFMA has been issued: a
    // pixel's value behind that MFMA, a kernel row's (two rows of a 1x1 kernel's) MFMAs before it is needed, the weights at the
    // group's end.
    //   First half of a group: nothing but MFMAs and reads.  In the middle the wavefronts meet: the next chunk is in LDS,
    // and nobody reads the one before any more.  Second half: the loads of the chunk after the next go out into that one's place.
    constexpr int TOGETHER = KS == 1 ? 2 : KS, READS = RUN / TOGETHER;        // values per read; reads per group and pixel
    constexpr uint32_t PTILE = 16 * PT * (4 / WO);
    float b[PT][TOGETHER];
    // value e of a read, from the address of its window
    auto read_at = [&](uint32_t window, int e) -> float { return reinterpret_cast<lds_float>(window)[KS == 1 ? e * PTILE : e]; };
    if constexpr (RESIDENT) {
        auto window = [&](uint32_t group) -> uint32_t {
            const uint32_t row = group * 4 + quarter, c = row / KS, kh = row % KS;
            return (c * q.pitch + kh * q.wp) * 4;
        };
        {
            const uint32_t at = window(chunk0);
#pragma unroll
            for (int j = 0; j < PT; ++j)
#pragma unroll
                for (int e = 0; e < TOGETHER; ++e) b[j][e] = read_at(base[0][j] + at, e);
        }
        for (uint32_t group = chunk0; group < chunk1; ++group) {
            // the vector work of a group in one place
            const uint32_t then = group + 1 < chunk1 ? group + 1 : group, at = window(then);
            uint32_t next[PT];
#pragma unroll
            for (int j = 0; j < PT; ++j) next[j] = base[0][j] + at;
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int e = 0; e < RUN; ++e) wv[i][e] = w_next[i][e];
            if ((group + 1) * (4 * RUN) > q.K) {
                // the last group: rows past the last channel count as zero
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int e = 0; e < RUN; ++e)
                        if ((group * 4 + quarter) * RUN + e >= q.K) wv[i][e] = 0.0f;
            }
#pragma unroll
            for (int i = 0; i < 2; ++i) f32_load_run<RUN>(w_next[i], rsrc_w, w_from[i] + then * (4 * RUN * 4));
            __builtin_amdgcn_sched_barrier(0);
            f32_static_for<KS>([&](auto t_) {
                constexpr int t = decltype(t_)::value;
                f32_static_for<PT>([&](auto j_) {
                    constexpr int j = decltype(j_)::value;
                    acc[0][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[j][t], wv[0][t], acc[0][j], 0, 0, 0);
                    acc[1][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[j][t], wv[1][t], acc[1][j], 0, 0, 0);
                    b[j][t] = read_at(next[j], t);
                    __builtin_amdgcn_sched_barrier(0);
                });
            });
        }
    } else {
        uint32_t w_at = lds_at + (SIGNAL + (wave_o * 32 + column) * (4 * RUN) + quarter * RUN) * 4;      // row `column` of the first tile
        auto read_weight = [&](int k) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                if constexpr (RUN % 4 == 0) {
                    if (k % 4 == 0) {
                        const float4c v = *reinterpret_cast<lds_float4>(w_at + (i * 16 * (4 * RUN) + k) * 4);
#pragma unroll
                        for (int e = 0; e < 4; ++e) wv[i][k + e] = v[e];
                    }
                } else {
                    wv[i][k] = *reinterpret_cast<lds_float>(w_at + (i * 16 * (4 * RUN) + k) * 4);
                }
            }
        };
#pragma unroll
        for (int j = 0; j < PT; ++j)
#pragma unroll
            for (int e = 0; e < TOGETHER; ++e) b[j][e] = read_at(base[0][j], e);
#pragma unroll
        for (int k = 0; k < RUN; ++k) read_weight(k);
        constexpr int HALF = READS > 1 ? READS / 2 : 0;      // the meeting is before read HALF
        constexpr int WEIGHTS = RUN % 4 == 0 ? 4 : 1;         // steps whose weights are read together
        uint32_t chunk = chunk0, current = 0;
        auto run = [&](auto next_, auto more_) __attribute__((always_inline)) {
            constexpr bool NEXT = decltype(next_)::value, MORE = decltype(more_)::value;
            const uint32_t after = current == 2 * STAGE ? 0 : current + STAGE, into = current == 0 ? 2 * STAGE : current - STAGE;
            if constexpr (MORE) {
                if (q.ragged && chunk + 3 == q.chunks) end_of_channels();
            }
            f32_static_for<READS>([&](auto r_) __attribute__((always_inline)) {
                constexpr int r = decltype(r_)::value;
                constexpr bool turn = r + 1 == READS;
                if constexpr (NEXT && r == HALF) {
                    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                    __builtin_amdgcn_s_barrier();
                    asm volatile("" ::: "memory");
                    // the wavefronts run in step and share the path to memory: each a little later than the one before
                    if (MORE && (wave & 1)) asm volatile("s_nop 15\n s_nop 7");
                    if (MORE && (wave & 2)) asm volatile("s_nop 15\n s_nop 15\n s_nop 15");
                }
                if constexpr (NEXT && turn) {
                    // what is read from here on is the next chunk's
                    const uint32_t step = (after - current) * 4;
#pragma unroll
                    for (int j = 0; j < PT; ++j)
#pragma unroll
                        for (int u = 0; u < ROWS; ++u) base[u][j] += step;
                    w_at += step;
                    __builtin_amdgcn_sched_barrier(0);
                }
                f32_static_for<TOGETHER>([&](auto t_) __attribute__((always_inline)) {
                    constexpr int t = decltype(t_)::value, k = r * TOGETHER + t;
                    f32_static_for<PT>([&](auto j_) __attribute__((always_inline)) {
                        constexpr int j = decltype(j_)::value;
                        acc[0][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[j][t], wv[0][k], acc[0][j], 0, 0, 0);
                        acc[1][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[j][t], wv[1][k], acc[1][j], 0, 0, 0);
                        constexpr int r_then = turn ? 0 : r + 1;
                        if constexpr (!turn || NEXT) b[j][t] = read_at(base[KS == 1 ? 0 : r_then][j] + (KS == 1 ? r_then * 2 * PTILE * 4 : 0), t);
                        if constexpr (NEXT && turn && j + 1 == PT) {
                            // the weights whose last step is over: those before the last read's first steps, then the step's own
                            if constexpr (t == 0) {
#pragma unroll
                                for (int e = 0; e + WEIGHTS <= k + 1; e += WEIGHTS) read_weight(e);
                            } else if constexpr ((k + 1) % WEIGHTS == 0) {
                                read_weight(k + 1 - WEIGHTS);
                            }
                        }
                        if constexpr (MORE) {
                            constexpr int PAIRS = (RUN - HALF * TOGETHER) * PT, pair = (k - HALF * TOGETHER) * PT + j;
                            constexpr int first = pair < 0 ? 0 : pair * OPS / PAIRS, end = pair < 0 ? 0 : (pair + 1) * OPS / PAIRS;
                            f32_static_for<end - first>([&](auto o_) __attribute__((always_inline)) { fetch(first + decltype(o_)::value, chunk + 2, into); });
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    });
                });
            });
            current = after;
        };
        using Yes = std::true_type;
        using No = std::false_type;
        constexpr uint32_t GROUPS = chained_groups(KS, U, PT);
        float4c total[2][GROUPS ? PT : 1];
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < (GROUPS ? PT : 1); ++j) total[i][j] = float4c{0.0f, 0.0f, 0.0f, 0.0f};
        uint32_t left = GROUPS;
        auto settle = [&] {
            if constexpr (GROUPS != 0) {
                if (--left != 0) return;
                left = GROUPS;
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < PT; ++j) {
                        total[i][j] += acc[i][j];
                        acc[i][j] = float4c{0.0f, 0.0f, 0.0f, 0.0f};
                    }
            }
        };
        for (; chunk + 2 < chunk1; ++chunk) {
            run(Yes{}, Yes{});
            settle();
        }
        if (chunk + 1 < chunk1) {
            run(Yes{}, No{});
            settle();
            ++chunk;
        }
        run(No{}, No{});
        if constexpr (GROUPS != 0) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < PT; ++j) acc[i][j] = total[i][j] + acc[i][j];
        }
    }

    // ---- results: four consecutive pixels of a channel per lane, as 16 bytes wherever they lie in one image ------------
    typedef float float4any __attribute__((ext_vector_type(4), aligned(4)));
#pragma unroll
    for (int j = 0; j < PT; ++j) {
        const uint32_t pixel = p0 + wave_p * (16 * PT) + j * 16 + quarter * 4;
        if (pixel >= q.pixels) continue;
        uint32_t n, r;
        q.div_hw.divmod(pixel, n, r);
        const bool whole = partials ? pixel + 4 <= q.pixels : r + 4 <= q.hw;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t co = co0 + i * 16 + column;
            if (co >= p.O) continue;
            float* to = partials ? partials + (static_cast<size_t>(split) * p.O + co) * q.pixels + pixel
                                 : y + static_cast<int64_t>(n) * p.ys[0] + static_cast<int64_t>(co) * p.ys[1] + r;
            if (whole) {
                *reinterpret_cast<float4any*>(to) = acc[i][j];
            } else {
                uint32_t at = r;
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    if (pixel + v >= q.pixels) break;
                    *to = acc[i][j][v];
                    ++to;
                    if (!partials && ++at == q.hw) {
                        at = 0;
                        to += p.ys[0] - static_cast<int64_t>(q.hw);
                    }
                }
            }
        }
    }
#endif
}

// y[n][co][r] = the sum over the splits, in split order (split 0 started from the bias)
__global__ __launch_bounds__(256) void conv2d_f32_sum_kernel(const float* partials, float* y, ConvProblem p, uint32_t pixels, uint32_t splits, FastDiv div_pixels, FastDiv div_hw,
                                                             uint32_t total) {
    const uint32_t idx = blockIdx.x * 256 + threadIdx.x;
    if (idx >= total) return;
    float sum = partials[idx];
    for (uint32_t s = 1; s < splits; ++s) sum += partials[static_cast<size_t>(s) * total + idx];
    uint32_t co, pixel, n, r;
    div_pixels.divmod(idx, co, pixel);
    div_hw.divmod(pixel, n, r);
    y[static_cast<int64_t>(n) * p.ys[0] + static_cast<int64_t>(co) * p.ys[1] + r] = sum;
}

template <int KS, int U, int PT, int NL, bool RESIDENT, int WO, bool WIDE>
static int launch_f32(const ConvProblem& p, const F32Plan& q, const float* x, const float* w, const float* bias, float* y, float* partials, hipStream_t stream) {
    auto kernel = conv2d_f32_kernel<KS, U, PT, NL, RESIDENT, WO, WIDE>;
    static std::atomic<uint64_t> configured{0};
    if (int rc = raise_lds_limit(reinterpret_cast<const void*>(kernel), 160 * 1024, configured)) return rc;
    const uint32_t blocks = (q.pixels + q.ptile - 1) / q.ptile * q.co_tiles * q.splits;
    const size_t lds = static_cast<size_t>(q.buffer) * 4;
    hipLaunchKernelGGL(kernel, dim3(blocks), dim3(kF32Threads), lds, stream, x, w, bias, y, partials, p, q);
    return launch_status("conv2d_f32_kernel");
}

// one of the kernels below as a candidate: its plan and the time it is expected to take
template <int KS, int U, int PT, int NL, bool RESIDENT, int WO, bool WIDE>
static void consider_f32(const ConvProblem& p, bool wide, F32Plan& best, double& best_time, int& best_index, int index) {
    constexpr uint32_t COMPUTE_UNITS = 256;
    constexpr uint32_t wo = WO;
    if (WIDE != wide && KS == 1) return;
    if (wo > 1 && p.O <= 16 * wo) return;     // half of the wavefronts would have no channel
    F32Plan q{};
    q.K = p.C * KS * KS;
    // The widest tiles are one block on a compute unit, and nothing runs beside its write-out: not under a short K (K = 60, 187 channels,
    // 4 images of 123 x 124: 31 us with them, 26 before this kernel, 21 with the next narrower; K below 32 in more than three rounds, mean of
    // nine: 1.12 times the time before with them, 0.87 without; K of 64 to 128 in one round or less, mean of thirteen: 0.87 and 0.79).
    if (KS == 1 && PT >= 10 && q.K < 128) return;
    q.pixels = p.N * p.HO * p.WO;
    q.ptile = 16 * PT * (4 / wo);
    q.co_tiles = (p.O + 32 * wo - 1) / (32 * wo);
    // (padding beyond the kernel's height: the images move apart until no image's first window begins above the last of the one
    // before, as a tile's windows are counted from its first row on)
    uint64_t hp = static_cast<uint64_t>(p.H) + p.pad_h;
    if (static_cast<uint64_t>(p.HO - 1) * p.stride_h > hp) hp = static_cast<uint64_t>(p.HO - 1) * p.stride_h;
    const uint64_t wp = static_cast<uint64_t>(p.W) + p.pad_w;
    if (hp >= (1ull << 31) || wp >= (1ull << 31)) return;
    q.hp = static_cast<uint32_t>(hp);
    q.wp = static_cast<uint32_t>(wp);
    // the plane of a tile: its sampled pixels, or the rows its windows touch
    uint64_t plane, images;
    if (KS == 1) {
        plane = q.ptile;
        images = (q.ptile - 2) / (p.HO * p.WO) + 2;
    } else {
        const uint64_t rows = (q.ptile - 2) / p.WO + 2;                // output rows a tile can touch
        images = (rows - 2) / p.HO + 2;
        const int64_t between = static_cast<int64_t>(q.hp) - static_cast<int64_t>(p.HO) * p.stride_h;
        plane = ((rows - 1) * p.stride_h + KS + (between > 0 ? (images - 1) * static_cast<uint64_t>(between) : 0)) * q.wp + p.pad_w + KS;
    }
    if (images > p.N) images = p.N;
    // quarters of a wavefront read planes next to each other: they begin 16 banks apart (17 where columns are two apart)
    const uint32_t residue = p.stride_w == 1 ? 16 : 17;
    // (a wavefront loads a plane 64 places at a time, all of them its own)
    const uint64_t pitch = KS == 1 ? plane : RESIDENT ? plane : 64 * NL + residue;
    if (pitch > (1u << 16)) return;
    q.rows64 = 64 / q.wp;
    q.rows256 = 256 / q.wp;
    q.ragged = p.C * KS % (4 * U) != 0;
    const uint64_t values = RESIDENT ? ((p.C * KS + 3) / 4 * 4 + KS - 1) / KS * pitch : 4 * U / KS * pitch;
    if (RESIDENT ? values * 4 > 64 * 1024 : KS == 1 ? values > 256 * NL : plane > 64 * NL) return;
    q.chunks = (q.K + 4 * U * KS - 1) / (4 * U * KS);
    q.pitch = static_cast<uint32_t>(pitch);
    q.plane = static_cast<uint32_t>(plane);
    q.buffer = RESIDENT ? static_cast<uint32_t>(values) : 3 * (256 * NL + (KS == 1 ? 0 : 128) + 1024 * ((WO * 32 * U * KS + 255) / 256));
    if (q.buffer * 4 > 160 * 1024) return;
    const uint64_t span = (images * p.xs[0] + static_cast<uint64_t>(p.C) * p.xs[1] + static_cast<uint64_t>(p.H) * p.xs[2] + p.W) * 4;
    if (span >= (1ull << 31)) return;
    const uint64_t tiles = (q.pixels + q.ptile - 1) / q.ptile * q.co_tiles;
    // Tiles of 32 pixels under 128 channels (planes so wide that no other tile fits) read the signal often: not beyond half a round of
    // them under a short K or with channels to spare (time against the kernels before: K = 72, 14 rounds 1.53, K = 144, 4 rounds 1.31, K =
    // 2916 with 192 channels in two tiles 1.28; K = 1152 with whole tiles 0.77 - 0.93, below half a round 0.54 - 0.76).
    if (KS == 3 && PT * (4 / WO) == 2 && 2 * tiles > COMPUTE_UNITS && (q.K < 512 || 8 * p.O < 7 * q.co_tiles * 32 * wo)) return;
    const uint32_t resident = PT >= 10 || q.buffer * 4 > 80 * 1024 ? 1 : 2;        // blocks on a compute unit at a time
    for (uint32_t splits = 1; splits <= (RESIDENT ? 1 : q.chunks) && splits <= 32; ++splits) {
        const uint32_t per_split = (q.chunks + splits - 1) / splits;
        if (splits > 1 && (per_split * (splits - 1) >= q.chunks || tiles * (splits - 1) >= 2 * COMPUTE_UNITS)) continue;
        if (splits > 1 && chained_groups(KS, U, PT) == 0) continue;      // (where blocks share the channels, the sums are short chains)
        const uint64_t blocks = tiles * splits;
        if (blocks >= (1ull << 24)) continue;
        // microseconds: a chunk is U * KS steps of 2 PT MFMAs of 32 clocks; start and write-out of a round; the pass over partial sums
        const double rounds = static_cast<double>((blocks + COMPUTE_UNITS - 1) / COMPUTE_UNITS);
        const double work = per_split * ((U * KS) * (2.0 * PT * 32) + 120.0) / 2300.0;
        const double time = rounds * work + 4.0 * (1.0 + (rounds - 1.0) / (2.0 * resident)) + (splits > 1 ? 4.5 + splits * static_cast<double>(q.pixels) * p.O * 8 / 4e6 : 0.0);
        if (time < best_time) {
            best_time = time;
            best = q;
            best.splits = splits;
            best.chunks_per_split = per_split;
            best_index = index;
        }
    }
}

template <class Launch>
static int finish_f32(const ConvProblem& p, F32Plan& q, float* y, hipStream_t stream, Launch&& launch) {
    const uint32_t hw = p.HO * p.WO;
    q.hw = hw;
    q.div_hw = FastDiv(hw);
    q.div_wo = FastDiv(p.WO);
    q.div_hp = FastDiv(q.hp);
    q.div_wp = FastDiv(q.wp);
    q.div_pitch = FastDiv(q.pitch);
    q.div_co_tiles = FastDiv(q.co_tiles);
    q.div_splits = FastDiv(q.splits);
    float* partials = nullptr;
    const uint32_t results = q.pixels * p.O;
    if (q.splits > 1 && scratch_acquire(reinterpret_cast<void**>(&partials), static_cast<size_t>(results) * q.splits * 4, stream) != TANNIC_SUCCESS) return TANNIC_ERROR;
    int status = launch(partials);
    if (partials) {
        if (status == TANNIC_SUCCESS) {
            hipLaunchKernelGGL(conv2d_f32_sum_kernel, dim3((results + 255) / 256), dim3(256), 0, stream, partials, y, p, q.pixels, q.splits, FastDiv(q.pixels), FastDiv(hw), results);
            status = launch_status("conv2d_f32_sum_kernel");
        }
        scratch_release(partials, stream);
    }
    return status;
}

// The kernels compiled: F(KS, U, PT, NL, RESIDENT, WO, WIDE).  (Three more shapes were the plan of 110 of 295 000 random problems.)
#define TH_F32_K1W(F, WIDE) F(1, 4, 2, 8, false, 1, WIDE) F(1, 4, 2, 4, false, 2, WIDE) F(1, 8, 2, 4, false, 4, WIDE) F(1, 4, 4, 8, false, 2, WIDE) \
    F(1, 8, 4, 8, false, 4, WIDE) F(1, 4, 6, 12, false, 2, WIDE) F(1, 8, 6, 12, false, 4, WIDE) F(1, 8, 8, 16, false, 4, WIDE) F(1, 4, 7, 8, false, 4, WIDE) F(1, 4, 7, 16, false, 2, WIDE) \
    F(1, 4, 13, 16, false, 4, WIDE) F(1, 4, 13, 28, false, 2, WIDE)
#define TH_F32_K1(F) TH_F32_K1W(F, true) TH_F32_K1W(F, false)
#define TH_F32_K3(F) F(3, 3, 2, 8, false, 1, false) F(3, 3, 2, 8, false, 2, false) F(3, 3, 2, 8, false, 4, false) F(3, 3, 4, 8, false, 2, false) F(3, 3, 4, 8, false, 4, false) F(3, 3, 5, 8, false, 2, false) \
    F(3, 3, 5, 8, false, 4, false) F(3, 3, 7, 8, false, 2, false) F(3, 3, 7, 6, false, 4, false) F(3, 3, 7, 12, false, 4, false) F(3, 3, 7, 16, false, 2, false) F(3, 3, 10, 10, false, 2, false) F(3, 3, 10, 12, false, 4, false) F(3, 3, 4, 12, false, 2, false) \
    F(3, 3, 13, 12, false, 2, false) F(3, 3, 13, 10, false, 4, false)
#define TH_F32_K7(F) F(7, 1, 2, 1, true, 1, false) F(7, 1, 2, 1, true, 2, false) F(7, 1, 4, 1, true, 2, false) F(7, 1, 7, 1, true, 2, false)

#define TH_F32_CONSIDER(KS, U, PT, NL, RES, WO, WIDE) consider_f32<KS, U, PT, NL, RES, WO, WIDE>(p, wide, q, time, index, counter++);
#define TH_F32_LAUNCH(KS, U, PT, NL, RES, WO, WIDE) \
    if (index == counter++) return launch_f32<KS, U, PT, NL, RES, WO, WIDE>(p, q, x, w, bias, y, partials, stream);

#define TH_F32_DESCRIBE(KS, U, PT, NL, RES, WO, WIDE) \
    if (index == counter++) {                         \
        const uint32_t of[7] = {KS, U, PT, NL, RES, WO, WIDE}; \
        for (int i = 0; i < 7; ++i) out[1 + i] = of[i];        \
    }

// The index of the kernel that takes the problem, with its plan and the time (us) it is expected to take; -1 if none does
static int plan_f32(const ConvProblem& p, int dtype, const void* x, const void* w, F32Plan& q, double& time) {
    if (dtype != TANNIC_FLOAT32 || p.KH != p.KW || p.C == 0) return -1;
    const uint64_t K = static_cast<uint64_t>(p.C) * p.KH * p.KW, pixels = static_cast<uint64_t>(p.N) * p.HO * p.WO;
    // contiguous OIHW weights (K runs through memory in order), rows of single floats, results contiguous within an image
    if (p.ws[3] != 1 || p.ws[2] != p.KW || p.ws[1] != static_cast<int64_t>(p.KH) * p.KW || p.ws[0] != static_cast<int64_t>(K) || reinterpret_cast<uintptr_t>(w) % 4 != 0) return -1;
    if (p.xs[3] != 1 || p.xs[0] < 0 || p.xs[1] < 0 || p.xs[2] < 0 || p.ys[3] != 1 || p.ys[2] != static_cast<int64_t>(p.WO)) return -1;
    if (p.KH == 1 && (p.pad_h || p.pad_w)) return -1;
    if (K * p.O * 4 >= (1ull << 31) || pixels >= (1ull << 28) || pixels * p.O >= (1ull << 31)) return -1;
    const bool dense = p.stride_h == 1 && p.stride_w == 1;
    // 16-byte pieces of the weights (7x7 takes single floats), and of a 1x1 kernel's signal where an image is whole pieces
    if (p.KH != 7 && (K % 4 != 0 || reinterpret_cast<uintptr_t>(w) % 16 != 0)) return -1;
    const bool wide = dense && p.xs[2] == static_cast<int64_t>(p.W) && (static_cast<uint64_t>(p.H) * p.W) % 4 == 0 && p.xs[0] % 4 == 0 && p.xs[1] % 4 == 0 &&
                      reinterpret_cast<uintptr_t>(x) % 16 == 0;
    // Few results go to the products that share K more finely than the groups here do, and so round less: 1x1 kernels to the product of
    // small matrices, which is faster too (512 -> 256 over 20 x 20, two images: 8.6 us and 2.1e-7 there, 12.9 and 4.1e-7 as one chain
    // here), with a stride, whose samples that product needs copied, under fewer than 256 channels (128 -> 64 over 56 x 56, two images:
    // 7.2 us and 1.1e-7 there, 8.1 here; under 512 the groups round less, 1.6e-7 against 2.1e-7); 3x3 kernels with at most 8192 results to
    // the product with a workgroup per 4 x 4 results, unfolded (304 -> 3 over 35 x 37, two images: 1.0e-7 there, 2.9e-7 as chains shared
    // by eleven blocks here, although in 13 us instead of 49).
    const uint64_t image = static_cast<uint64_t>(p.HO) * p.WO;
    if (p.KH == 1 && image % 4 == 0 && (dense ? p.xs[2] == static_cast<int64_t>(p.W) : p.WO % 4 == 0 && p.C < 256) && gemm_small_f32_takes(p.O, image, p.C, p.N)) return -1;
    if (p.KH == 3 && K >= 320 && (image + 3) / 4 * 4 * p.N * p.O <= 8192) return -1;
    // Very many results under a short K are bound by writing them, behind the sums of a block here and beside those of others in the products
    // over images (29 images of 122 x 122, 20 -> 991: 544 us there, 717 here; 24 of 84 x 84, 32 -> 437 with a stride: 111 / 149; but 4 -> 739
    // 640 / 543 and 16 -> 286 307 / 279).
    if (p.KH == 1 && image % 4 == 0 && K >= 8 && K < 64 && p.O >= 400 && pixels * p.O >= (1ull << 26)) return -1;
    time = 1e30;
    int index = -1, counter = 0;
    if (p.KH == 1) {
        TH_F32_K1(TH_F32_CONSIDER)
    } else if (p.KH == 3) {
        TH_F32_K3(TH_F32_CONSIDER)
    } else if (p.KH == 7) {
        TH_F32_K7(TH_F32_CONSIDER)
        // Wide rows: what a tile loads grows beyond what it multiplies (three channels, stride 2, 64 channels, mean of the time against the
        // gathering tiles by the LDS of a block: up to 32 KB 0.81, to 40 KB 0.88, to 44 KB 0.95, to 50 KB 1.01, to 60 KB 1.2).
        if (q.buffer * 4 > 40 * 1024) return -1;
    }
    return index;
}

double conv2d_f32_expected(const ConvProblem& p, int dtype, const void* x, const void* w) {
    F32Plan q{};
    double time;
    return plan_f32(p, dtype, x, w, q, time) < 0 ? -1.0 : time;
}

bool conv2d_f32_plan(const ConvProblem& p, int dtype, const void* x, const void* w, uint32_t out[kConvPlanValues]) {
    if (p.N == 0 || p.O == 0 || p.HO == 0 || p.WO == 0) return false;
    F32Plan q{};
    double time;
    const int index = plan_f32(p, dtype, x, w, q, time);
    if (index < 0) return false;
    int counter = 0;
    if (p.KH == 1) {
        TH_F32_K1(TH_F32_DESCRIBE)
    } else if (p.KH == 3) {
        TH_F32_K3(TH_F32_DESCRIBE)
    } else {
        TH_F32_K7(TH_F32_DESCRIBE)
    }
    out[0] = 1;
    const uint32_t plan[9] = {q.ptile, q.co_tiles, q.splits, q.chunks, q.chunks_per_split, q.pitch, q.plane, q.hp, q.wp};
    for (int i = 0; i < 9; ++i) out[8 + i] = plan[i];
    return true;
}

int conv2d_f32(const ConvProblem& p, int dtype, const void* x_, const void* w_, const void* bias_, void* y_, hipStream_t stream) {
    if (dtype != TANNIC_FLOAT32 || p.KH != p.KW) return TANNIC_UNSUPPORTED_DTYPE;
    if (p.N == 0 || p.O == 0 || p.HO == 0 || p.WO == 0) return TANNIC_SUCCESS;
    F32Plan q{};
    double time;
    const int index = plan_f32(p, dtype, x_, w_, q, time);
    if (index < 0) return TANNIC_UNSUPPORTED_DTYPE;
    const float* x = static_cast<const float*>(x_);
    const float* w = static_cast<const float*>(w_);
    const float* bias = static_cast<const float*>(bias_);
    float* y = static_cast<float*>(y_);
    return finish_f32(p, q, y, stream, [&](float* partials) -> int {
        int counter = 0;
        if (p.KH == 1) {
            TH_F32_K1(TH_F32_LAUNCH)
        } else if (p.KH == 3) {
            TH_F32_K3(TH_F32_LAUNCH)
        } else {
            TH_F32_K7(TH_F32_LAUNCH)
        }
        return TANNIC_UNSUPPORTED_DTYPE;
    });
}

}  // namespace th
