// conv2d in fp32 on the 16-bit matrix pipe: every value is the sum of three bfloat16 values, 1x1 and 3x3 kernels.
//
// The fp32 matrix pipe does 32 multiply-adds a clock and SIMD, the bfloat16 one 512.  A float is exactly the sum of three bfloat16 values
// (24 bits of mantissa, three times eight; each part the nearest to what the ones before left), and of the nine products of parts the
// six largest carry everything above 2^-24 of the product: x0 w0, x0 w1, x1 w0, x1 w1, x0 w2, x2 w0, each exact, summed in fp32.  Six MFMAs of
// 16 x 16 x 32 take the place of eight of 16 x 16 x 4 of twice the length: 2.7 times the rate of the fp32 pipe, 1.5 times after the clock that
// this much work leaves (1.4 PFLOP/s of bfloat16 products, the rate of the large products, are 233 TFLOP/s of fp32; the fp32 pipe does 157).
// The error against 64 bits is below that of the fp32 pipe, which rounds after every product where this rounds after 32: the five small
// products have accumulators of their own (a rounding there is 2^-8 of one beside the large ones), and the large ones' sums are
// chains of nine taps (1x1: of 512 products).  256 -> 256 3x3 over 14 x 14: 1.07e-7 of the result's norm, 1.80e-7 on the fp32 pipe;
// 512 -> 512 over 7 x 7 1.18e-7 / 1.63e-7; 1x1 512 -> 128 1.28e-7 / 1.55e-7, 1024 -> 256 1.3e-7 / 1.64e-7.
//  * The weights are split by a kernel of their own, into the order in which the MFMAs want them; wavefronts load them straight into
//    registers, 16 bytes a lane.  The signal is split on its way into LDS: a lane takes eight channels of a place of the tile's plane (the
//    rows that the tile touches, padding made real, as in conv2d_f32.hip), eight loads of one float each, whole lines for the
//    wavefront, and writes 16 bytes to each of three planes of 32 channels.  So nothing is asked of the signal's widths, alignment or
//    strides.  Of the weights plan_split asks what conv2d_f32.hip does (whole 16-byte pieces, a K that four divides): that kernel's
//    expected time is what this one's is held against.
//  * A wavefront's tile is 32 output channels by 16 PT pixels of the flattened batch; WO wavefronts of a block's four lie along the
//    channels.  A tap of 32 channels is 12 PT MFMAs for six loads of weights and 3 PT reads of LDS.
//  * Both operands are split 2^24 times as large as they are, so that the last bit of the smallest fp32 value (2^-149) is a normal bfloat16: no
//    part of any value is denormal, whatever lies beside it, and the sums are 2^48 times the results (powers of two change no rounding).
//    What that puts out of range (values from 2^103 on, results from 2^79 on), infinities and NaNs leave a sum that is not finite: the wavefront
//    does those sixteen pixels over again in fp32, straight from memory, thirty-six products at a time.  (Slow, and only there: 128 -> 256 3x3 over
//    20 x 20, sixteen images, 35 us; one infinity 178, one in every ninth value of a channel 320; 52 on the fp32 pipe.  Weights or signals of 1e-37
//    beside ordinary ones 1.1e-7 of their own results, 1.5e-7 on the fp32 pipe.)
// With few tiles the channels are shared between `splits` blocks per tile, partial sums in fp32, added in split order by a second kernel.
// Measured, 53 convolutions of a ResNet-50 and their additions, batch 32: 3350 -> 2740 .. 2880 us by the card (the layers: plan_split).
// What is left: the weights' kernel (3 - 5 us of a layer's 30 - 50), a block's start and end (some 9 us), the last round of tiles.
#include "conv_common.hpp"

namespace th {

typedef __bf16 split8 __attribute__((ext_vector_type(8)));
typedef __bf16 split2 __attribute__((ext_vector_type(2)));
typedef float float2s __attribute__((ext_vector_type(2)));
typedef float float4s __attribute__((ext_vector_type(4)));
typedef unsigned int uint4s __attribute__((ext_vector_type(4)));
typedef unsigned short ushort2s __attribute__((ext_vector_type(2)));

constexpr int kSplitThreads = 256;
constexpr uint32_t kSplitOutside = 0x80000000u;   // byte offset no buffer reaches: loads zero
constexpr uint32_t kSplitChannels = 32;           // per chunk: the K of one MFMA
// the operands are split so many times as large as they are, and the sums brought back by the square of it
constexpr float kSplitUp = 0x1p24f, kSplitSumUp = 0x1p48f, kSplitSumDown = 0x1p-48f;

// The high products of so many chunks of a 1x1 kernel (the nine taps of one chunk of a 3x3 kernel) are one chain of additions, the chains'
// sums added to a third set of accumulators.  The chain rounds as much as the square root of its length (K = 1024, 1024 -> 256 over 14 x 14:
// 1.87e-7 of the result's norm as one chain, 1.3e-7 as two; the fp32 matrix pipe's chains of 64 products 1.64e-7).
constexpr uint32_t kSplitChained = 16;

struct SplitPlan {
    uint32_t pixels, ptile;              // N * HO * WO; pixels per block
    uint32_t co_tiles, splits;
    uint32_t chunks, chunks_per_split;
    uint32_t plane;                      // places of a tile's plane that hold something
    uint32_t hp, wp;                     // rows of an image and columns of a row with the shared padding
    uint32_t hw;
    uint32_t weight_bytes;
    FastDiv div_hw, div_wo, div_hp, div_wp, div_co_tiles, div_splits;
};

template <int N, class F, int I = 0>
__device__ __forceinline__ void split_static_for(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        split_static_for<N, F, I + 1>(static_cast<F&&>(f));
    }
}

// a = the sum of the low halves, b = that of the high halves, to 2^-24 and better of the value: each part is the nearest bfloat16 to what the
// ones before left, and both differences are exact
__device__ __forceinline__ void split_pair(float a, float b, uint32_t part[3]) {
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const split2 rounded = __builtin_convertvector(float2s{a, b}, split2);
        __builtin_memcpy(&part[i], &rounded, 4);
        a -= __builtin_bit_cast(float, part[i] << 16);
        b -= __builtin_bit_cast(float, part[i] & 0xFFFF0000u);
    }
}

__device__ __forceinline__ float4s split_mfma(const uint4s& a, const uint4s& b, const float4s& c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(split8, a), __builtin_bit_cast(split8, b), c, 0, 0, 0);
}

// The weights as MFMA operands: [16 channels out][32 channels in][tap][part][lane][8].
// A block per 16 x 32 channels, whose weights are sixteen runs of 32 TAPS floats, through LDS; a wavefront per tap (1x1: four, of which
// one goes on), as there is nothing here but the latency of one load, one pass through LDS and one store.
template <int TAPS> constexpr int split_weight_threads = TAPS == 1 ? 256 : 64 * TAPS;
template <int TAPS>
__global__ __launch_bounds__(split_weight_threads<TAPS>) void conv2d_split_weights_kernel(const float* w, uint4s* planes, uint32_t O, uint32_t C, FastDiv div_chunks) {
    constexpr uint32_t RUN = kSplitChannels * TAPS, PITCH = RUN + 1, THREADS = split_weight_threads<TAPS>;
    __shared__ float held[16 * PITCH];
    const uint32_t tap = threadIdx.x / 64, lane = threadIdx.x % 64;
    uint32_t tile, chunk;
    div_chunks.divmod(blockIdx.x, tile, chunk);
    const uint32_t c0 = chunk * kSplitChannels, live = (C - c0 < kSplitChannels ? C - c0 : kSplitChannels) * TAPS;
    float v[16 * RUN / THREADS];
#pragma unroll
    for (uint32_t i = 0; i < 16 * RUN / THREADS; ++i) {
        const uint32_t at = i * THREADS + threadIdx.x, row = at / RUN, e = at % RUN, o = tile * 16 + row;
        v[i] = o < O && e < live ? w[(o * C + c0) * TAPS + e] : 0.0f;
    }
#pragma unroll
    for (uint32_t i = 0; i < 16 * RUN / THREADS; ++i) {
        const uint32_t at = i * THREADS + threadIdx.x;
        held[at / RUN * PITCH + at % RUN] = v[i];
    }
    __syncthreads();
    if (tap >= TAPS) return;
    const float* mine = held + lane % 16 * PITCH + lane / 16 * (8 * TAPS) + tap;
    uint32_t part[4][3];
#pragma unroll
    for (int e = 0; e < 4; ++e) split_pair(mine[2 * e * TAPS] * kSplitUp, mine[(2 * e + 1) * TAPS] * kSplitUp, part[e]);
    const uint32_t fragment = blockIdx.x * TAPS + tap;
#pragma unroll
    for (int i = 0; i < 3; ++i) planes[(fragment * 3 + i) * 64 + lane] = uint4s{part[0][i], part[1][i], part[2][i], part[3][i]};
}

// KS: the kernel's side; PT: 16-pixel tiles per wavefront; WO: wavefronts along the output channels (32 each), the others along the
// pixels; NL: places of a plane per lane.
template <int KS, int PT, int WO, int NL>
__global__ __launch_bounds__(kSplitThreads, NL <= 3 && (KS == 1 || PT <= 2) ? 2 : 1) void conv2d_split_kernel(const float* x, const float* w, const uint4s* planes, const float* bias, float* y,
                                                                                   float* partials, ConvProblem p, SplitPlan q) {
#if defined(__HIP_DEVICE_COMPILE__)   // the host pass needs the launch stub only (and loses it over the body's device-only builtins)
    constexpr int TAPS = KS * KS;
    // Bytes.  A place's 32 channels are 64, every 80, so that sixteen places' reads are in all banks without any arithmetic; in three parts
    constexpr uint32_t PLACE = 80, PLANE = NL * 64 * PLACE, STAGE = 3 * PLANE;
    typedef const __attribute__((address_space(3))) uint4s* lds_read;
    typedef __attribute__((address_space(3))) uint4s* lds_write;
    typedef __attribute__((address_space(3))) void* lds_void;
    extern __shared__ __align__(16) unsigned char split_lds[];
    const uint32_t lds_at = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_void)(split_lds)));

    uint32_t block = blockIdx.x;
    // workgroups go round the eight dies in turn: tiles next to each other (which share rows of the signal) on one die
    if (gridDim.x % 8 == 0) block = (block % 8) * (gridDim.x / 8) + block / 8;
    uint32_t rest, split, tile, ct;
    q.div_splits.divmod(block, rest, split);
    q.div_co_tiles.divmod(rest, tile, ct);
    const uint32_t p0 = tile * q.ptile;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64;
    const uint32_t column = lane % 16, quarter = lane / 16;
    const uint32_t wave_o = wave % WO, wave_p = wave / WO;
    const uint32_t co0 = (ct * WO + wave_o) * 32;
    const uint32_t chunk0 = split * q.chunks_per_split, chunk1 = chunk0 + q.chunks_per_split < q.chunks ? chunk0 + q.chunks_per_split : q.chunks;

    // ---- where this lane's places of a plane come from: channel 8 * wave of a chunk --------------------------
    uint32_t n0, r0, oh0, ow0;
    q.div_hw.divmod(p0, n0, r0);
    q.div_wo.divmod(r0, oh0, ow0);
    const float* image = x + static_cast<int64_t>(n0) * p.xs[0];
    const int64_t reach = (static_cast<int64_t>(p.N - 1 - n0) * p.xs[0] + static_cast<int64_t>(p.C - 1) * p.xs[1] + static_cast<int64_t>(p.H - 1) * p.xs[2] + p.W) * 4;
    const __amdgpu_buffer_rsrc_t rsrc_x =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(image), 0, static_cast<int>(reach < 0x7FFFFFFF ? reach : 0x7FFFFFFF), 0x00020000);
    uint32_t from[NL];
#pragma unroll
    for (int t = 0; t < NL; ++t) {
        const uint32_t e = t * 64 + lane;
        from[t] = kSplitOutside;
        if constexpr (KS == 1) {
            // the sampled pixels, one after the other
            const uint32_t pixel = p0 + e;
            if (e < q.plane && pixel < q.pixels) {
                uint32_t n, r, oh, ow;
                q.div_hw.divmod(pixel, n, r);
                q.div_wo.divmod(r, oh, ow);
                from[t] = static_cast<uint32_t>((static_cast<int64_t>(n - n0) * p.xs[0] + static_cast<int64_t>(oh * p.stride_h) * p.xs[2] + ow * p.stride_w) * 4);
            }
        } else {
            // the rows that the tile touches, W + pad columns each, the padding between rows and images shared by both
            uint32_t g, col, dn, row;
            q.div_wp.divmod(e, g, col);
            q.div_hp.divmod(oh0 * p.stride_h + g, dn, row);
            const uint32_t ih = row - p.pad_h, iw = col - p.pad_w;   // unsigned: the padding is huge
            if (e < q.plane && n0 + dn < p.N && ih < p.H && iw < p.W) from[t] = static_cast<uint32_t>((static_cast<int64_t>(dn) * p.xs[0] + static_cast<int64_t>(ih) * p.xs[2] + iw) * 4);
        }
    }
    const uint32_t channel_step = static_cast<uint32_t>(p.xs[1] * 4);
    float held[NL][8];
    auto fetch = [&](int t, uint32_t chunk) __attribute__((always_inline)) {
        const uint32_t c0 = chunk * kSplitChannels + wave * 8;
        if (c0 + 8 <= p.C) {
#pragma unroll
            for (int e = 0; e < 8; ++e) held[t][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc_x, from[t], (c0 + e) * channel_step, 0));
        } else {
            // the last chunk may have fewer channels: the others are zero
#pragma unroll
            for (int e = 0; e < 8; ++e) held[t][e] = c0 + e < p.C ? __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc_x, from[t], (c0 + e) * channel_step, 0)) : 0.0f;
        }
    };
    // two of a place's eight channels, split; all eight to LDS
    uint32_t part[4][3];
    auto split_two = [&](int t, int e) __attribute__((always_inline)) { split_pair(held[t][2 * e] * kSplitUp, held[t][2 * e + 1] * kSplitUp, part[e]); };
    const uint32_t keep_at = lds_at + lane * PLACE + wave * 16;
    auto keep = [&](int t, uint32_t stage) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 3; ++i) *reinterpret_cast<lds_write>(keep_at + stage + t * (64 * PLACE) + i * PLANE) = uint4s{part[0][i], part[1][i], part[2][i], part[3][i]};
    };

    // ---- weights: a fragment of three parts for each of the two 16-channel tiles, a tap ahead --------------
    uint32_t w_at[2];       // bytes
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        uint32_t of = (co0 / 16) + i;
        const uint32_t last = (p.O + 15) / 16 - 1;
        of = of < last ? of : last;
        w_at[i] = (of * q.chunks + chunk0) * (TAPS * 3 * 1024);
    }
    const __amdgpu_buffer_rsrc_t rsrc_w = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint4s*>(planes), 0, static_cast<int>(q.weight_bytes), 0x00020000);
    constexpr int AHEAD = KS == 1 ? 1 : 2;      // taps that the weights are loaded ahead of their use
    uint4s wv[AHEAD + 1][2][3];
    auto fetch_weights = [&](int into) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
#pragma unroll
            for (int s = 0; s < 3; ++s) {
                const auto v = __builtin_amdgcn_raw_buffer_load_b128(rsrc_w, lane * 16 + s * 1024, w_at[i], 0);
                __builtin_memcpy(&wv[into][i][s], &v, 16);
            }
            w_at[i] += 3 * 1024;
        }
    };
#pragma unroll
    for (int a = 0; a < AHEAD; ++a) fetch_weights(a);
#pragma unroll
    for (int t = 0; t < NL; ++t) fetch(t, chunk0);

    // ---- this lane's pixels: where their windows begin in LDS, for each row of the kernel ------------------------
    uint32_t window[KS][PT];
#pragma unroll
    for (int j = 0; j < PT; ++j) {
        const uint32_t mine = wave_p * (16 * PT) + j * 16 + column;
        uint32_t first = mine;
        if constexpr (KS != 1) {
            const uint32_t pixel = p0 + mine < q.pixels ? p0 + mine : q.pixels - 1;
            uint32_t n, r, oh, ow;
            q.div_hw.divmod(pixel, n, r);
            q.div_wo.divmod(r, oh, ow);
            first = ((n - n0) * q.hp + oh * p.stride_h - oh0 * p.stride_h) * q.wp + ow * p.stride_w;
        }
#pragma unroll
        for (int kh = 0; kh < KS; ++kh) window[kh][j] = lds_at + (first + kh * q.wp) * PLACE + quarter * 16;
    }
    auto start_value = [&](int i) -> float {
        const uint32_t co = co0 + i * 16 + column;
        return p.has_bias && split == 0 && co < p.O ? bias[static_cast<int64_t>(co) * p.bs] : 0.0f;
    };
    // (i, j) -> channel i * 16 + column, value v -> pixel 4 * quarter + v
    constexpr bool SETTLES = KS != 1 || PT <= 4;       // (the widest tile of a 1x1 kernel has no registers for the third set, and K up to 512)
    float4s high[2][PT], low[2][PT], total[2][SETTLES ? PT : 1];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const float b = start_value(i) * kSplitSumUp;
#pragma unroll
        for (int j = 0; j < PT; ++j) {
            high[i][j] = SETTLES ? float4s{0.0f, 0.0f, 0.0f, 0.0f} : float4s{b, b, b, b};
            low[i][j] = float4s{0.0f, 0.0f, 0.0f, 0.0f};
            if constexpr (SETTLES) total[i][j] = float4s{b, b, b, b};
        }
    }
    auto meet = [] {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
#pragma unroll
    for (int t = 0; t < NL; ++t) {
#pragma unroll
        for (int e = 0; e < 4; ++e) split_two(t, e);
        keep(t, 0);
    }
    if (chunk0 + 1 < chunk1) {
#pragma unroll
        for (int t = 0; t < NL; ++t) fetch(t, chunk0 + 1);
    }
    meet();

    // The loop, a tap of sixteen pixels of the wavefront at a time: twelve MFMAs, six products of parts for each of the two channel
    // tiles, and between them what comes next: the signal's fragment of the step after (three reads of LDS), the weights of the tap after
    // the next (six loads), a quarter of the work of splitting a place of the next chunk, and loads of the chunk after it.  An MFMA keeps the
    // pipe busy for 16 clocks and a wavefront issues an instruction every 4: three fit behind each, and nothing may stand in a row.
    uint32_t stage = 0;
    uint4s b[2][3];
    auto read = [&](uint32_t at, int into) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < 3; ++s) b[into][s] = *reinterpret_cast<lds_read>(at + s * PLANE);
    };
    constexpr int STEPS = TAPS * PT, UNITS = 4 * NL;
    for (uint32_t chunk = chunk0; chunk < chunk1; ++chunk) {
        const bool more = chunk + 2 < chunk1;
        read(window[0][0], 0);
        split_static_for<STEPS>([&](auto step_) __attribute__((always_inline)) {
            constexpr int step = decltype(step_)::value, tap = step / PT, j = step % PT, now = step % 2, set = TAPS == 1 ? 0 : tap % (AHEAD + 1);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (j == 0) fetch_weights((set + AHEAD) % (AHEAD + 1));     // (behind the block's last tap: what lies there, never multiplied)
            if constexpr (step + 1 < STEPS) {
                constexpr int tap_then = (step + 1) / PT;
                read(window[tap_then / KS][(step + 1) % PT] + tap_then % KS * PLACE, 1 - now);
            }
            // (behind the last chunk: the same values once more, never read)
            constexpr int unit = (step * UNITS + STEPS - 1) / STEPS, units = ((step + 1) * UNITS + STEPS - 1) / STEPS - unit;
            split_static_for<units>([&](auto u_) __attribute__((always_inline)) {
                constexpr int u = unit + decltype(u_)::value;
                split_two(u / 4, u % 4);
                if constexpr (u % 4 == 3) keep(u / 4, STAGE - stage);
            });
            // of the nine products of parts the six that reach the result, the small ones in a sum of their own
            auto multiply = [&](auto& sum, int of_b, int of_w) __attribute__((always_inline)) {
#pragma unroll
                for (int i = 0; i < 2; ++i) sum[i][j] = split_mfma(b[now][of_b], wv[set][i][of_w], sum[i][j]);
            };
            multiply(low, 2, 0);
            multiply(low, 0, 2);
            multiply(low, 1, 1);
            multiply(low, 1, 0);
            multiply(low, 0, 1);
            multiply(high, 0, 0);
#pragma unroll
            for (int m = 0; m < 12; ++m) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                if (m < 3) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                if (j == 0) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
                if (units) __builtin_amdgcn_sched_group_barrier(0x002, 2 * units, 0);
                if (m >= 9) __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            split_static_for<units>([&](auto u_) __attribute__((always_inline)) {
                constexpr int u = unit + decltype(u_)::value;
                if constexpr (u % 4 == 3) {
                    if (more) fetch(u / 4, chunk + 2);
                }
            });
        });
        if constexpr (TAPS % (AHEAD + 1) != 0) {
            // the sets move up
            uint4s moved[AHEAD + 1][2][3];
#pragma unroll
            for (int a = 0; a <= AHEAD; ++a)
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int s = 0; s < 3; ++s) moved[a][i][s] = wv[(a + TAPS) % (AHEAD + 1)][i][s];
#pragma unroll
            for (int a = 0; a <= AHEAD; ++a)
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int s = 0; s < 3; ++s) wv[a][i][s] = moved[a][i][s];
        }
        if (SETTLES && (KS != 1 || (chunk - chunk0) % kSplitChained == kSplitChained - 1)) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < PT; ++j) {
                    total[i][j] += high[i][j];
                    high[i][j] = float4s{0.0f, 0.0f, 0.0f, 0.0f};
                }
        }
        meet();
        stage = STAGE - stage;
        const uint32_t turn = stage ? STAGE : 0u - STAGE;
#pragma unroll
        for (int kh = 0; kh < KS; ++kh)
#pragma unroll
            for (int j = 0; j < PT; ++j) window[kh][j] += turn;
    }
    uint32_t redo = 0;       // bit j: a sum of the pixels j is not finite
#pragma unroll
    for (int j = 0; j < PT; ++j) {
        bool finite = true;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            high[i][j] += low[i][j];
            if constexpr (SETTLES) high[i][j] += total[i][j];
#pragma unroll
            for (int v = 0; v < 4; ++v) finite = finite && __builtin_isfinite(high[i][j][v]);
            high[i][j] *= kSplitSumDown;
        }
        if (__builtin_amdgcn_ballot_w64(!finite)) redo |= 1u << j;
    }

    // ---- values and sums beyond the range: these pixels over again, in fp32 --------------------------------------
    if (redo) {
        constexpr int CHAIN = 9;        // MFMAs of four products, the loads of all on their way together
        const uint32_t k_first = chunk0 * kSplitChannels * TAPS, k_end = (chunk1 * kSplitChannels < p.C ? chunk1 * kSplitChannels : p.C) * TAPS;
#pragma unroll 1
        for (int j = 0; j < PT; ++j) {
            if (!(redo >> j & 1)) continue;
            const uint32_t pixel = p0 + wave_p * (16 * PT) + j * 16 + column;
            uint32_t n, r, oh, ow;
            q.div_hw.divmod(pixel < q.pixels ? pixel : q.pixels - 1, n, r);
            q.div_wo.divmod(r, oh, ow);
            const float* from_image = x + static_cast<int64_t>(n) * p.xs[0];
            float4s all[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const float b = start_value(i);
                all[i] = float4s{b, b, b, b};
            }
#pragma unroll 1
            for (uint32_t k0 = k_first; k0 < k_end; k0 += 4 * CHAIN) {
                float xv[CHAIN], wk[CHAIN][2];
#pragma unroll
                for (int u = 0; u < CHAIN; ++u) {
                    const uint32_t k = k0 + 4 * u + quarter, c = k / TAPS, tap = k % TAPS;
                    const uint32_t ih = oh * p.stride_h + tap / KS - p.pad_h, iw = ow * p.stride_w + tap % KS - p.pad_w;
                    // (what is not there is the first element, and then zero)
                    const bool there = k < k_end && pixel < q.pixels && ih < p.H && iw < p.W;
                    const float value = from_image[there ? static_cast<int64_t>(c) * p.xs[1] + static_cast<int64_t>(ih) * p.xs[2] + iw : 0];
                    xv[u] = there ? value : 0.0f;
#pragma unroll
                    for (int i = 0; i < 2; ++i) {
                        const uint32_t co = co0 + i * 16 + column;
                        const bool weighs = k < k_end && co < p.O;
                        const float weight = w[weighs ? static_cast<size_t>(co) * p.C * TAPS + k : 0];
                        wk[u][i] = weighs ? weight : 0.0f;
                    }
                }
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    float4s sum = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                    for (int u = 0; u < CHAIN; ++u) sum = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[u], wk[u][i], sum, 0, 0, 0);
                    all[i] += sum;
                }
            }
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int to = 0; to < PT; ++to)
                    if (to == j) high[i][to] = all[i];
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
                *reinterpret_cast<float4any*>(to) = high[i][j];
            } else {
                uint32_t at = r;
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    if (pixel + v >= q.pixels) break;
                    *to = high[i][j][v];
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
__global__ __launch_bounds__(256) void conv2d_split_sum_kernel(const float* partials, float* y, ConvProblem p, uint32_t splits, FastDiv div_pixels, FastDiv div_hw, uint32_t total) {
    const uint32_t idx = blockIdx.x * 256 + threadIdx.x;
    if (idx >= total) return;
    float sum = partials[idx];
    for (uint32_t s = 1; s < splits; ++s) sum += partials[static_cast<size_t>(s) * total + idx];
    uint32_t co, pixel, n, r;
    div_pixels.divmod(idx, co, pixel);
    div_hw.divmod(pixel, n, r);
    y[static_cast<int64_t>(n) * p.ys[0] + static_cast<int64_t>(co) * p.ys[1] + r] = sum;
}

struct SplitOperands {
    const float *x, *w, *bias;
    const uint4s* planes;
    float *y, *partials;
};

template <int KS, int PT, int WO, int NL>
static int launch_split(const ConvProblem& p, const SplitPlan& q, const SplitOperands& o, hipStream_t stream) {
    auto kernel = conv2d_split_kernel<KS, PT, WO, NL>;
    static std::atomic<uint64_t> configured{0};
    constexpr size_t lds = 2 * 3 * NL * 64 * 80;
    if (int rc = raise_lds_limit(reinterpret_cast<const void*>(kernel), lds, configured)) return rc;
    const uint32_t blocks = (q.pixels + q.ptile - 1) / q.ptile * q.co_tiles * q.splits;
    hipLaunchKernelGGL(kernel, dim3(blocks), dim3(kSplitThreads), lds, stream, o.x, o.w, o.planes, o.bias, o.y, o.partials, p, q);
    return launch_status("conv2d_split_kernel");
}

// one of the kernels below as a candidate: its plan and the time it is expected to take
template <int KS, int PT, int WO, int NL>
static void consider_split(const ConvProblem& p, SplitPlan& best, double& best_time, int& best_index, int index) {
    constexpr uint32_t COMPUTE_UNITS = 256;
    SplitPlan q{};
    q.pixels = p.N * p.HO * p.WO;
    q.ptile = 16 * PT * (4 / WO);
    q.co_tiles = (p.O + 32 * WO - 1) / (32 * WO);
    q.chunks = (p.C + kSplitChannels - 1) / kSplitChannels;
    // (padding beyond the kernel's height: the images move apart until no image's first window begins above the last of the one before)
    uint64_t hp = static_cast<uint64_t>(p.H) + p.pad_h;
    if (static_cast<uint64_t>(p.HO - 1) * p.stride_h > hp) hp = static_cast<uint64_t>(p.HO - 1) * p.stride_h;
    const uint64_t wp = static_cast<uint64_t>(p.W) + p.pad_w;
    if (hp >= (1ull << 31) || wp >= (1ull << 31)) return;
    q.hp = static_cast<uint32_t>(hp);
    q.wp = static_cast<uint32_t>(wp);
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
    if (plane > 64 * NL) return;
    q.plane = static_cast<uint32_t>(plane);
    if (images > p.N) images = p.N;
    const uint64_t span = (images * p.xs[0] + static_cast<uint64_t>(p.C) * p.xs[1] + static_cast<uint64_t>(p.H) * p.xs[2] + p.W) * 4;
    if (span >= (1ull << 31)) return;
    const uint64_t tiles = (q.pixels + q.ptile - 1) / q.ptile * q.co_tiles;
    for (uint32_t splits = 1; splits <= q.chunks && splits <= 16; ++splits) {
        const uint32_t per_split = (q.chunks + splits - 1) / splits;
        if (splits > 1 && (per_split * (splits - 1) >= q.chunks || tiles * (splits - 1) >= 2 * COMPUTE_UNITS)) continue;
        if (KS == 1 && PT > 4 && per_split > kSplitChained) continue;
        const uint64_t blocks = tiles * splits;
        if (blocks >= (1ull << 24)) continue;
        // Microseconds.  A tap of 32 channels is 12 PT MFMAs of 16 clocks for every wavefront, at the 1.45 GHz that is left of the clock under
        // them, and what splitting a tile's places does not hide behind them (a second block on the compute unit hides some of it); a
        // round's start and end; the weights' kernel and the launches; the pass over partial sums.
        const double rounds = static_cast<double>((blocks + COMPUTE_UNITS - 1) / COMPUTE_UNITS);
        const double work = per_split * (KS * KS * (12.0 * PT * 16) + NL * 300.0 + 150.0) / 1450.0 * (KS == 1 && rounds > 1.0 ? 0.82 : 1.0);
        const double time = rounds * (work + 3.0) + 13.0 + (splits > 1 ? 4.0 + splits * static_cast<double>(q.pixels) * p.O * 8 / 4e6 : 0.0);
        if (time < best_time) {
            best_time = time;
            best = q;
            best.splits = splits;
            best.chunks_per_split = per_split;
            best_index = index;
        }
    }
}

// The kernels compiled: F(KS, PT, WO, NL)
#define TH_SPLIT_K1(F) F(1, 4, 2, 2) F(1, 4, 4, 1) F(1, 7, 4, 2)
#define TH_SPLIT_K3(F) F(3, 2, 2, 2) F(3, 2, 2, 3) F(3, 4, 2, 4) F(3, 4, 2, 5) F(3, 4, 4, 2) F(3, 4, 4, 3) F(3, 4, 4, 4) F(3, 7, 4, 4) F(3, 7, 4, 5)

#define TH_SPLIT_CONSIDER(KS, PT, WO, NL) consider_split<KS, PT, WO, NL>(p, q, time, index, counter++);
#define TH_SPLIT_LAUNCH(KS, PT, WO, NL) \
    if (index == counter++) return launch_split<KS, PT, WO, NL>(p, q, o, stream);

// The index of the kernel that takes the problem, with its plan; -1 if none does
static int plan_split(const ConvProblem& p, int dtype, const void* x, const void* w, SplitPlan& q) {
    if (dtype != TANNIC_FLOAT32 || p.KH != p.KW || (p.KH != 1 && p.KH != 3)) return -1;
    const uint64_t K = static_cast<uint64_t>(p.C) * p.KH * p.KW, pixels = static_cast<uint64_t>(p.N) * p.HO * p.WO;
    // contiguous OIHW weights, rows of single floats, results contiguous within an image
    if (p.ws[3] != 1 || p.ws[2] != p.KW || p.ws[1] != static_cast<int64_t>(p.KH) * p.KW || p.ws[0] != static_cast<int64_t>(K) || reinterpret_cast<uintptr_t>(w) % 4 != 0) return -1;
    if (p.xs[3] != 1 || p.xs[0] < 0 || p.xs[1] < 0 || p.xs[2] < 0 || p.ys[3] != 1 || p.ys[2] != static_cast<int64_t>(p.WO) || reinterpret_cast<uintptr_t>(x) % 4 != 0) return -1;
    if (p.KH == 1 && (p.pad_h || p.pad_w)) return -1;
    if (K * p.O * 4 >= (1ull << 31) || pixels >= (1ull << 28) || pixels * p.O >= (1ull << 31)) return -1;
    // what is addressed is the weights as parts, six bytes a value with both kinds of channels rounded up: 32-bit byte offsets, two fragments ahead
    const uint64_t fragments = (static_cast<uint64_t>(p.O) + 15) / 16 * ((static_cast<uint64_t>(p.C) + kSplitChannels - 1) / kSplitChannels) * (p.KH * p.KW);
    if ((fragments + 2) * 3 * 1024 >= (1ull << 32)) return -1;
    // (few channels are a short K: what a tile starts and ends with counts, and 1x1 kernels are bound by their tensors; small problems by launches)
    if (p.KH == 1 ? p.C < (p.O >= 128 ? 100u : 140u) : p.C < 32) return -1;
    if (2.0 * K * p.O * pixels < 1.2e9) return -1;
    const double before = conv2d_f32_expected(p, dtype, x, w);
    if (before < 0) return -1;
    double time = 1e30;
    int index = -1, counter = 0;
    if (p.KH == 1) {
        TH_SPLIT_K1(TH_SPLIT_CONSIDER)
    } else {
        TH_SPLIT_K3(TH_SPLIT_CONSIDER)
    }
    // What the fp32 kernel takes is 1.2 to 1.5 times its expectation (us there / here, in a network of such layers: 3x3 128 -> 128 over 28 x 28,
    // batch 32, 75 / 50; 256 -> 256 over 14 x 14 86 / 53, alone with sixteen images 61 / 40, eight 35 / 34; 1x1 512 -> 256 over 28 x 28
    // 62 / 51, 1024 -> 512 over 14 x 14 72 / 54, 2048 -> 512 over 7 x 7 56 / 37, 512 -> 128 over 28 x 28 44 / 40, eight images of it 19 / 23).
    return index >= 0 && time < before * (p.KH == 3 ? 1.15 : 1.4) ? index : -1;
}

#define TH_SPLIT_DESCRIBE(KS, PT, WO, NL)          \
    if (index == counter++) {                     \
        const uint32_t of[4] = {KS, PT, WO, NL};    \
        for (int i = 0; i < 4; ++i) out[1 + i] = of[i]; \
    }

bool conv2d_split_plan(const ConvProblem& p, int dtype, const void* x, const void* w, uint32_t out[kConvPlanValues]) {
    if (p.N == 0 || p.O == 0 || p.HO == 0 || p.WO == 0) return false;
    SplitPlan q{};
    const int index = plan_split(p, dtype, x, w, q);
    if (index < 0) return false;
    int counter = 0;
    if (p.KH == 1) {
        TH_SPLIT_K1(TH_SPLIT_DESCRIBE)
    } else {
        TH_SPLIT_K3(TH_SPLIT_DESCRIBE)
    }
    out[0] = 3;
    const uint32_t plan[8] = {q.ptile, q.co_tiles, q.splits, q.chunks, q.chunks_per_split, q.plane, q.hp, q.wp};
    for (int i = 0; i < 8; ++i) out[5 + i] = plan[i];
    return true;
}

int conv2d_split(const ConvProblem& p, int dtype, const void* x, const void* w, const void* bias, void* y, hipStream_t stream) {
    if (dtype != TANNIC_FLOAT32 || p.KH != p.KW) return TANNIC_UNSUPPORTED_DTYPE;
    if (p.N == 0 || p.O == 0 || p.HO == 0 || p.WO == 0) return TANNIC_SUCCESS;
    SplitPlan q{};
    const int index = plan_split(p, dtype, x, w, q);
    if (index < 0) return TANNIC_UNSUPPORTED_DTYPE;
    q.hw = p.HO * p.WO;
    q.div_hw = FastDiv(q.hw);
    q.div_wo = FastDiv(p.WO);
    q.div_hp = FastDiv(q.hp);
    q.div_wp = FastDiv(q.wp);
    q.div_co_tiles = FastDiv(q.co_tiles);
    q.div_splits = FastDiv(q.splits);
    const uint32_t taps = p.KH * p.KW, fragments = (p.O + 15) / 16 * q.chunks * taps, results = q.pixels * p.O;
    // (a block's weights are loaded a tap ahead, the last ones behind the end)
    const size_t plane_bytes = (static_cast<size_t>(fragments) + 2) * 3 * 1024;
    char* scratch = nullptr;
    if (scratch_acquire(reinterpret_cast<void**>(&scratch), plane_bytes + (q.splits > 1 ? static_cast<size_t>(results) * q.splits * 4 : 0), stream) != TANNIC_SUCCESS) {
        (void)hipGetLastError();
        return TANNIC_UNSUPPORTED_DTYPE;      // no memory for the split weights: conv2d_f32 needs none, or less
    }
    q.weight_bytes = static_cast<uint32_t>(plane_bytes);
    uint4s* planes = reinterpret_cast<uint4s*>(scratch);
    const SplitOperands o{static_cast<const float*>(x), static_cast<const float*>(w), static_cast<const float*>(bias), planes, static_cast<float*>(y),
                          q.splits > 1 ? reinterpret_cast<float*>(scratch + plane_bytes) : nullptr};
    const uint32_t weight_blocks = (p.O + 15) / 16 * q.chunks;
    if (taps == 1) hipLaunchKernelGGL((conv2d_split_weights_kernel<1>), dim3(weight_blocks), dim3(split_weight_threads<1>), 0, stream, o.w, planes, p.O, p.C, FastDiv(q.chunks));
    else hipLaunchKernelGGL((conv2d_split_weights_kernel<9>), dim3(weight_blocks), dim3(split_weight_threads<9>), 0, stream, o.w, planes, p.O, p.C, FastDiv(q.chunks));
    int status = launch_status("conv2d_split_weights_kernel");
    if (status == TANNIC_SUCCESS) {
        status = [&]() -> int {
            int counter = 0;
            if (p.KH == 1) {
                TH_SPLIT_K1(TH_SPLIT_LAUNCH)
            } else {
                TH_SPLIT_K3(TH_SPLIT_LAUNCH)
            }
            return TANNIC_ERROR;
        }();
    }
    if (status == TANNIC_SUCCESS && q.splits > 1) {
        hipLaunchKernelGGL(conv2d_split_sum_kernel, dim3((results + 255) / 256), dim3(256), 0, stream, o.partials, o.y, p, q.splits, FastDiv(q.pixels), FastDiv(q.hw), results);
        status = launch_status("conv2d_split_sum_kernel");
    }
    scratch_release(scratch, stream);
    return status;
}

}  // namespace th
