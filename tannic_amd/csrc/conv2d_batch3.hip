// conv2d with a 3x3 kernel, 16-bit, a batch of small maps under many channels: pixels of the flattened batch, weights as MFMA operands.
//
// The patch kernel (conv2d_k3.hip) gives a block whole rows of one image: maps of 14 x 14 leave it 128 blocks for 256 compute units, and every
// block brings its weights through registers and LDS.  Here a block takes 16 PT (4 / WO) consecutive pixels of the flattened batch, whatever
// images they lie in, and 32 WO output channels.
//  * The weights are put into the order in which the MFMAs want them by a kernel of their own; wavefronts load them straight into registers,
//    16 bytes a lane, each tap's set a whole chunk of 32 channels before its use.
//  * The signal goes through LDS in two stages as the plane of rows that the tile touches, padding made real, 32 channels a place: a lane
//    takes eight channels of a place, eight loads of one element, whole lines for the wavefront.  So nothing is asked of widths,
//    alignments, strides or channels.
//  * A wavefront's tile is 32 channels by 16 PT pixels; a tap of 32 channels is 2 PT MFMAs for two loads of weights and PT reads of LDS, made
//    while the tap before is multiplied.
// With few tiles the channels are shared between `splits` blocks per tile, partial sums in fp32, added in split order by a second kernel.
// fp16, batch 32, us before / now, the weights' kernel (4 us) included: 256 -> 256 over 14 x 14 29.4 / 23.6 (16 images 30.9 / 20.4), 384 -> 256 over
// 13 x 13 54 / 30, 256 -> 256 from 28 x 28 with a stride 37 / 29; plan_batch3 has more.  Bound by what a compute unit loads, 64 bytes a clock
// (a chunk's weights, 73 KB, take as long as 64 pixels' MFMAs; the signal is loaded element by element), by as many LDS reads, and by start and end.
// Loading a chunk ahead of the MFMAs and no branch around a load: 32.1 -> 23.5 us for the first of these layers.
#include "conv_common.hpp"

namespace th {

typedef _Float16 half8b __attribute__((ext_vector_type(8)));
typedef __bf16 bfloat8b __attribute__((ext_vector_type(8)));
typedef float float4b __attribute__((ext_vector_type(4)));
typedef unsigned int uint4b __attribute__((ext_vector_type(4)));

constexpr int kBatch3Threads = 256;
constexpr int kBatch3Taps = 9;
constexpr uint32_t kBatch3Outside = 0x80000000u;   // byte offset no buffer reaches: loads zero
constexpr uint32_t kBatch3Channels = 32;           // per chunk: the K of one MFMA

struct Batch3Plan {
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
__device__ __forceinline__ void batch3_static_for(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        batch3_static_for<N, F, I + 1>(static_cast<F&&>(f));
    }
}

template <class T> __device__ __forceinline__ float4b batch3_mfma(const uint4b& a, const uint4b& b, const float4b& c) {
    if constexpr (std::is_same_v<T, f16>) return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8b, a), __builtin_bit_cast(half8b, b), c, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bfloat8b, a), __builtin_bit_cast(bfloat8b, b), c, 0, 0, 0);
}

// The weights as MFMA operands: [16 channels out][32 channels in][tap][lane][8].  A block per 16 x 32 channels, whose weights are sixteen runs
// of 288 elements, through LDS; a wavefront per tap.
__global__ __launch_bounds__(64 * kBatch3Taps) void conv2d_batch3_weights_kernel(const uint16_t* w, uint4b* out, uint32_t O, uint32_t C, FastDiv div_chunks) {
    constexpr uint32_t RUN = kBatch3Channels * kBatch3Taps, PITCH = RUN + 2, THREADS = 64 * kBatch3Taps;
    __shared__ uint16_t held[16 * PITCH];
    uint32_t tile, chunk;
    div_chunks.divmod(blockIdx.x, tile, chunk);
    const uint32_t c0 = chunk * kBatch3Channels, live = (C - c0 < kBatch3Channels ? C - c0 : kBatch3Channels) * kBatch3Taps;
    uint16_t v[16 * RUN / THREADS];
#pragma unroll
    for (uint32_t i = 0; i < 16 * RUN / THREADS; ++i) {
        const uint32_t at = i * THREADS + threadIdx.x, row = at / RUN, e = at % RUN, o = tile * 16 + row;
        v[i] = o < O && e < live ? w[(o * C + c0) * kBatch3Taps + e] : static_cast<uint16_t>(0);
    }
#pragma unroll
    for (uint32_t i = 0; i < 16 * RUN / THREADS; ++i) {
        const uint32_t at = i * THREADS + threadIdx.x;
        held[at / RUN * PITCH + at % RUN] = v[i];
    }
    __syncthreads();
    const uint32_t tap = threadIdx.x / 64, lane = threadIdx.x % 64;
    const uint16_t* mine = held + lane % 16 * PITCH + lane / 16 * (8 * kBatch3Taps) + tap;
    uint32_t pair[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) pair[e] = mine[2 * e * kBatch3Taps] | static_cast<uint32_t>(mine[(2 * e + 1) * kBatch3Taps]) << 16;
    out[(blockIdx.x * kBatch3Taps + tap) * 64 + lane] = uint4b{pair[0], pair[1], pair[2], pair[3]};
}

// PT: 16-pixel tiles per wavefront; WO: wavefronts along the output channels (32 each), the others along the pixels; NL: places of a plane per lane.
template <class T, int PT, int WO, int NL>
__global__ __launch_bounds__(kBatch3Threads, PT <= 4 ? 2 : 1) void conv2d_batch3_kernel(const T* x, const uint4b* weights, const T* bias, T* y, float* partials, ConvProblem p, Batch3Plan q) {
#if defined(__HIP_DEVICE_COMPILE__)   // the host pass needs the launch stub only (and loses it over the body's device-only builtins)
    // Bytes.  A place's 32 channels are 64, every 80, so that sixteen places' reads are in all banks without any arithmetic
    constexpr uint32_t PLACE = 80, STAGE = NL * 64 * PLACE;
    constexpr int TAPS = kBatch3Taps, KS = 3, ES = sizeof(T);
    typedef const __attribute__((address_space(3))) uint4b* lds_read;
    typedef __attribute__((address_space(3))) uint4b* lds_write;
    typedef __attribute__((address_space(3))) void* lds_void;
    extern __shared__ __align__(16) unsigned char batch3_lds[];
    const uint32_t lds_at = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_void)(batch3_lds)));

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

    // ---- weights: a fragment for each of the two 16-channel tiles and each tap, a chunk ahead -----------------
    uint32_t w_at[2];       // bytes
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        uint32_t of = (co0 / 16) + i;
        const uint32_t last = (p.O + 15) / 16 - 1;
        of = of < last ? of : last;
        w_at[i] = (of * q.chunks + chunk0) * (TAPS * 1024);
    }
    const __amdgpu_buffer_rsrc_t rsrc_w = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint4b*>(weights), 0, static_cast<int>(q.weight_bytes), 0x00020000);
    uint4b wv[TAPS][2];
    auto fetch_weights = [&](int tap) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const auto v = __builtin_amdgcn_raw_buffer_load_b128(rsrc_w, lane * 16, w_at[i] + tap * 1024, 0);
            __builtin_memcpy(&wv[tap][i], &v, 16);
        }
    };

    // ---- where this lane's places of a plane come from: channel 8 * wave of a chunk --------------------------
    uint32_t n0, r0, oh0, ow0;
    q.div_hw.divmod(p0, n0, r0);
    q.div_wo.divmod(r0, oh0, ow0);
    const T* image = x + static_cast<int64_t>(n0) * p.xs[0];
    const int64_t reach = (static_cast<int64_t>(p.N - 1 - n0) * p.xs[0] + static_cast<int64_t>(p.C - 1) * p.xs[1] + static_cast<int64_t>(p.H - 1) * p.xs[2] + p.W) * ES;
    const __amdgpu_buffer_rsrc_t rsrc_x =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(image), 0, static_cast<int>(reach < 0x7FFFFFFF ? reach : 0x7FFFFFFF), 0x00020000);
    uint32_t from[NL];
#pragma unroll
    for (int t = 0; t < NL; ++t) {
        // the rows that the tile touches, W + pad columns each, the padding between rows and images shared by both
        const uint32_t e = t * 64 + lane;
        uint32_t g, col, dn, row;
        q.div_wp.divmod(e, g, col);
        q.div_hp.divmod(oh0 * p.stride_h + g, dn, row);
        const uint32_t ih = row - p.pad_h, iw = col - p.pad_w;   // unsigned: the padding is huge
        from[t] = kBatch3Outside;
        if (e < q.plane && n0 + dn < p.N && ih < p.H && iw < p.W) from[t] = static_cast<uint32_t>((static_cast<int64_t>(dn) * p.xs[0] + static_cast<int64_t>(ih) * p.xs[2] + iw) * ES);
    }
    const uint32_t channel_step = static_cast<uint32_t>(p.xs[1] * ES);
    uint32_t held[NL][8];
    // A value waits in a register of its own, above it zeros or copies of its sign: were it the same in the loop and before it, the compiler would
    // keep halves of registers from one chunk to the next, and to put them together wait for the loads where they are made.
    auto fetch = [&](int t, uint32_t chunk, auto signs) __attribute__((always_inline)) {
        // (no branch around loads: the wait for one counts those behind it.  The last chunk may have fewer channels: the others are zero)
        const uint32_t c0 = chunk * kBatch3Channels + wave * 8;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const uint16_t v = __builtin_amdgcn_raw_buffer_load_b16(rsrc_x, c0 + e < p.C ? from[t] : kBatch3Outside, c0 + e < p.C ? (c0 + e) * channel_step : 0, 0);
            held[t][e] = decltype(signs)::value ? static_cast<uint32_t>(static_cast<int32_t>(static_cast<int16_t>(v))) : v;
        }
    };
    const uint32_t keep_at = lds_at + lane * PLACE + wave * 16;
    auto keep = [&](int t, uint32_t stage) __attribute__((always_inline)) {
        uint4b v;
#pragma unroll
        for (int e = 0; e < 8; ++e) asm volatile("" : "+v"(held[t][e]));     // (nor may the pairs be made before)
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = (held[t][2 * e] & 0xFFFF) | held[t][2 * e + 1] << 16;
        *reinterpret_cast<lds_write>(keep_at + stage + t * (64 * PLACE)) = v;
    };
#pragma unroll
    for (int t = 0; t < NL; ++t) fetch(t, chunk0, std::true_type{});
#pragma unroll
    for (int tap = 0; tap < TAPS; ++tap) fetch_weights(tap);

    // ---- this lane's pixels: where their windows begin in LDS, for each row of the kernel ------------------------
    uint32_t window[KS][PT];
#pragma unroll
    for (int j = 0; j < PT; ++j) {
        const uint32_t mine = wave_p * (16 * PT) + j * 16 + column;
        const uint32_t pixel = p0 + mine < q.pixels ? p0 + mine : q.pixels - 1;
        uint32_t n, r, oh, ow;
        q.div_hw.divmod(pixel, n, r);
        q.div_wo.divmod(r, oh, ow);
        const uint32_t first = ((n - n0) * q.hp + oh * p.stride_h - oh0 * p.stride_h) * q.wp + ow * p.stride_w;
#pragma unroll
        for (int kh = 0; kh < KS; ++kh) window[kh][j] = lds_at + (first + kh * q.wp) * PLACE + quarter * 16;
    }
    // (i, j) -> channel i * 16 + column, value v -> pixel 4 * quarter + v
    float4b sum[2][PT];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const uint32_t co = co0 + i * 16 + column;
        const float b = p.has_bias && split == 0 && co < p.O ? static_cast<float>(widen(bias[static_cast<int64_t>(co) * p.bs])) : 0.0f;
#pragma unroll
        for (int j = 0; j < PT; ++j) sum[i][j] = float4b{b, b, b, b};
    }
    auto meet = [] {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
#pragma unroll
    for (int t = 0; t < NL; ++t) keep(t, 0);
#pragma unroll
    for (int t = 0; t < NL; ++t) fetch(t, chunk0 + 1 < chunk1 ? chunk0 + 1 : chunk0, std::true_type{});
    meet();

    // The loop, a tap of the wavefront's pixels at a time: 2 PT MFMAs, and between them what comes next: the signal's fragments of the tap after
    // (PT reads of LDS), this tap's weights of the next chunk (two loads), places of the next chunk into the other stage, and behind them
    // loads of the chunk after it.
    uint32_t stage = 0;
    uint4b b[2][PT];
    auto read = [&](int tap, int into) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < PT; ++j) b[into][j] = *reinterpret_cast<lds_read>(window[tap / KS][j] + tap % KS * PLACE);
    };
    for (uint32_t chunk = chunk0; chunk < chunk1; ++chunk) {
        const uint32_t after = chunk + 2 < chunk1 ? chunk + 2 : chunk;     // (behind the last chunk: one that is in the caches, never read)
        read(0, 0);
#pragma unroll
        for (int i = 0; i < 2; ++i) w_at[i] += TAPS * 1024;
        batch3_static_for<TAPS>([&](auto tap_) __attribute__((always_inline)) {
            constexpr int tap = decltype(tap_)::value, now = tap % 2;
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (tap + 1 < TAPS) read(tap + 1, 1 - now);
            constexpr int unit = (tap * NL + TAPS - 1) / TAPS, units = ((tap + 1) * NL + TAPS - 1) / TAPS - unit;
            batch3_static_for<units>([&](auto u_) __attribute__((always_inline)) { keep(unit + decltype(u_)::value, STAGE - stage); });
#pragma unroll
            for (int j = 0; j < PT; ++j)
#pragma unroll
                for (int i = 0; i < 2; ++i) sum[i][j] = batch3_mfma<T>(b[now][j], wv[tap][i], sum[i][j]);
#pragma unroll
            for (int m = 0; m < 2 * PT; ++m) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                if (m < PT) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                if (units && m >= PT) __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            fetch_weights(tap);                // (behind the block's last chunk: what lies there, never multiplied)
            batch3_static_for<units>([&](auto u_) __attribute__((always_inline)) { fetch(unit + decltype(u_)::value, after, std::false_type{}); });
        });
        meet();
        stage = STAGE - stage;
        const uint32_t turn = stage ? STAGE : 0u - STAGE;
#pragma unroll
        for (int kh = 0; kh < KS; ++kh)
#pragma unroll
            for (int j = 0; j < PT; ++j) window[kh][j] += turn;
    }

    // ---- results: four consecutive pixels of a channel per lane, in one piece wherever they lie in one image ------------
    typedef float float4any __attribute__((ext_vector_type(4), aligned(4)));
    typedef unsigned int uint2any __attribute__((ext_vector_type(2), aligned(2)));
#pragma unroll
    for (int j = 0; j < PT; ++j) {
        const uint32_t pixel = p0 + wave_p * (16 * PT) + j * 16 + quarter * 4;
        if (pixel >= q.pixels) continue;
        uint32_t n, r;
        q.div_hw.divmod(pixel, n, r);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t co = co0 + i * 16 + column;
            if (co >= p.O) continue;
            if (partials) {
                float* to = partials + (static_cast<size_t>(split) * p.O + co) * q.pixels + pixel;
                if (pixel + 4 <= q.pixels) {
                    *reinterpret_cast<float4any*>(to) = sum[i][j];
                } else {
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        if (pixel + v < q.pixels) to[v] = sum[i][j][v];
                }
                continue;
            }
            T* to = y + static_cast<int64_t>(n) * p.ys[0] + static_cast<int64_t>(co) * p.ys[1] + r;
            T rounded[4];
#pragma unroll
            for (int v = 0; v < 4; ++v) rounded[v] = narrow_result<T>(sum[i][j][v]);
            if (r + 4 <= q.hw) {
                uint2any bits;
                __builtin_memcpy(&bits, rounded, 8);
                *reinterpret_cast<uint2any*>(to) = bits;
            } else {
                uint32_t at = r;
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    if (pixel + v >= q.pixels) break;
                    *to = rounded[v];
                    ++to;
                    if (++at == q.hw) {
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
template <class T>
__global__ __launch_bounds__(256) void conv2d_batch3_sum_kernel(const float* partials, T* y, ConvProblem p, uint32_t splits, FastDiv div_pixels, FastDiv div_hw, uint32_t total) {
    const uint32_t idx = blockIdx.x * 256 + threadIdx.x;
    if (idx >= total) return;
    float sum = partials[idx];
    for (uint32_t s = 1; s < splits; ++s) sum += partials[static_cast<size_t>(s) * total + idx];
    uint32_t co, pixel, n, r;
    div_pixels.divmod(idx, co, pixel);
    div_hw.divmod(pixel, n, r);
    y[static_cast<int64_t>(n) * p.ys[0] + static_cast<int64_t>(co) * p.ys[1] + r] = narrow_result<T>(sum);
}

template <class T, int PT, int WO, int NL>
static int launch_batch3(const ConvProblem& p, const Batch3Plan& q, const void* x, const uint4b* weights, const void* bias, void* y, float* partials, hipStream_t stream) {
    auto kernel = conv2d_batch3_kernel<T, PT, WO, NL>;
    static std::atomic<uint64_t> configured{0};
    constexpr size_t lds = 2 * NL * 64 * 80;
    if (int rc = raise_lds_limit(reinterpret_cast<const void*>(kernel), lds, configured)) return rc;
    const uint32_t blocks = (q.pixels + q.ptile - 1) / q.ptile * q.co_tiles * q.splits;
    hipLaunchKernelGGL(kernel, dim3(blocks), dim3(kBatch3Threads), lds, stream, static_cast<const T*>(x), weights, static_cast<const T*>(bias), static_cast<T*>(y), partials, p, q);
    return launch_status("conv2d_batch3_kernel");
}

constexpr uint32_t COMPUTE_UNITS = 256;

// one of the kernels below as a candidate: its plan and the time it is expected to take
template <int PT, int WO, int NL>
static void consider_batch3(const ConvProblem& p, Batch3Plan& best, double& best_time, int& best_index, int index) {
    Batch3Plan q{};
    q.pixels = p.N * p.HO * p.WO;
    q.ptile = 16 * PT * (4 / WO);
    q.co_tiles = (p.O + 32 * WO - 1) / (32 * WO);
    q.chunks = (p.C + kBatch3Channels - 1) / kBatch3Channels;
    // (padding beyond the kernel's height: the images move apart until no image's first window begins above the last of the one before)
    uint64_t hp = static_cast<uint64_t>(p.H) + p.pad_h;
    if (static_cast<uint64_t>(p.HO - 1) * p.stride_h > hp) hp = static_cast<uint64_t>(p.HO - 1) * p.stride_h;
    const uint64_t wp = static_cast<uint64_t>(p.W) + p.pad_w;
    if (hp >= (1ull << 31) || wp >= (1ull << 31)) return;
    q.hp = static_cast<uint32_t>(hp);
    q.wp = static_cast<uint32_t>(wp);
    const uint64_t rows = (q.ptile - 2) / p.WO + 2;                // output rows a tile can touch
    uint64_t images = (rows - 2) / p.HO + 2;
    const int64_t between = static_cast<int64_t>(q.hp) - static_cast<int64_t>(p.HO) * p.stride_h;
    const uint64_t plane = ((rows - 1) * p.stride_h + 3 + (between > 0 ? (images - 1) * static_cast<uint64_t>(between) : 0)) * q.wp + p.pad_w + 3;
    if (plane > 64 * NL) return;
    q.plane = static_cast<uint32_t>(plane);
    if (images > p.N) images = p.N;
    const uint64_t span = (images * p.xs[0] + static_cast<uint64_t>(p.C) * p.xs[1] + static_cast<uint64_t>(p.H) * p.xs[2] + p.W) * 2;
    if (span >= (1ull << 31)) return;
    const uint64_t tiles = (q.pixels + q.ptile - 1) / q.ptile * q.co_tiles;
    for (uint32_t splits = 1; splits <= q.chunks && splits <= 8; ++splits) {
        const uint32_t per_split = (q.chunks + splits - 1) / splits;
        if (splits > 1 && (per_split * (splits - 1) >= q.chunks || tiles * (splits - 1) >= 2 * COMPUTE_UNITS)) continue;
        const uint64_t blocks = tiles * splits;
        if (blocks >= (1ull << 24)) continue;
        // Microseconds, within 4 % of 606 problems of one round and 8 % of 167 of more: a chunk of a block, alone on its compute unit with its loads'
        // latency to wait for, or beside and behind others; launches, a block's start and end; the pass over partial sums.  (Before, a chunk alone was
        // priced at two thirds of its time, and few blocks were left to walk all channels: 320 -> 512 over 20 x 24, one image, 64 blocks 23.5 us,
        // with shares of K 20.9; 448 -> 624 over 13 x 16, three images, 100 blocks 31.7 / 25.2.)
        const double rounds = static_cast<double>((blocks + COMPUTE_UNITS - 1) / COMPUTE_UNITS), results = static_cast<double>(q.pixels) * p.O;
        double time;
        if (rounds == 1.0) {
            time = per_split * (0.113 * PT + 0.156 * NL + 0.4) + 8.4 + (splits > 1 ? 3.0 + 1.8e-6 * splits * results : 0.0);
        } else {
            const double chunk = (9.0 * 2 * PT * 16 + 600.0 + NL * 100.0) / 2100.0 * (PT <= 4 ? 0.9 : 1.0);
            time = (PT <= 4 ? 1.35 : 1.35 + 0.05 * rounds) * (rounds * (per_split * chunk + 2.0) + 8.0 + (splits > 1 ? 4.0 + 2e-6 * splits * results : 0.0));
        }
        if (time < best_time) {
            best_time = time;
            best = q;
            best.splits = splits;
            best.chunks_per_split = per_split;
            best_index = index;
        }
    }
}

// The kernels compiled: F(PT, WO, NL)
#define TH_BATCH3(F) F(2, 2, 2) F(2, 2, 3) F(4, 2, 4) F(4, 2, 5) F(4, 2, 6) F(4, 4, 2) F(4, 4, 3) F(4, 4, 4) F(4, 4, 5) F(4, 4, 7) F(7, 4, 3) F(7, 4, 4) F(7, 4, 5)

#define TH_BATCH3_CONSIDER(PT, WO, NL) consider_batch3<PT, WO, NL>(p, q, time, index, counter++);
#define TH_BATCH3_LAUNCH(PT, WO, NL) \
    if (index == counter++) return launch_batch3<T, PT, WO, NL>(p, q, x, weights, bias, y, partials, stream);
#define TH_BATCH3_DESCRIBE(PT, WO, NL)          \
    if (index == counter++) {                  \
        const uint32_t of[3] = {PT, WO, NL};    \
        for (int i = 0; i < 3; ++i) out[2 + i] = of[i]; \
    }

// The index of the kernel that takes the problem, with its plan; -1 if none does
static int plan_batch3(const ConvProblem& p, int dtype, const void* x, const void* w, Batch3Plan& q) {
    if ((dtype != TANNIC_FLOAT16 && dtype != TANNIC_BFLOAT16) || p.KH != 3 || p.KW != 3) return -1;
    const uint64_t K = static_cast<uint64_t>(p.C) * 9, pixels = static_cast<uint64_t>(p.N) * p.HO * p.WO;
    // contiguous OIHW weights, rows of single elements, results contiguous within an image
    if (p.ws[3] != 1 || p.ws[2] != 3 || p.ws[1] != 9 || p.ws[0] != static_cast<int64_t>(K) || reinterpret_cast<uintptr_t>(w) % 2 != 0) return -1;
    if (p.xs[3] != 1 || p.xs[0] < 0 || p.xs[1] < 0 || p.xs[2] < 0 || p.ys[3] != 1 || p.ys[2] != static_cast<int64_t>(p.WO) || reinterpret_cast<uintptr_t>(x) % 2 != 0) return -1;
    if (K * p.O * 2 >= (1ull << 30) || pixels >= (1ull << 28) || pixels * p.O >= (1ull << 31)) return -1;
    // (the ordered weights, both kinds of channels rounded up and a chunk ahead, are addressed by 32-bit byte offsets)
    const uint64_t weight_blocks = (static_cast<uint64_t>(p.O) + 15) / 16 * ((static_cast<uint64_t>(p.C) + kBatch3Channels - 1) / kBatch3Channels);
    if ((weight_blocks + 1) * kBatch3Taps * 1024 >= (1ull << 32)) return -1;
    // Where it is the faster one (fp16, us before / here, weights' kernel included; before: the patch kernel, or the unfolded batch as a product for
    // few pixels an image and for channels that are not whole chunks):
    //  * small problems are launches (256 -> 256, six images of 12 x 12 18.6 / 19.1, 128 -> 128, six of 24 x 24 16.2 / 13.4); 64 channels are two
    //    chunks, all start and end (64 -> 64 over 56 x 56, batch 32, 19 / 43)
    const uint64_t image = static_cast<uint64_t>(p.HO) * p.WO;
    const bool whole_chunks = p.C % kBatch3Channels == 0;
    if (p.C < 64 || (whole_chunks && p.C < 96) || 2.0 * K * p.O * pixels < 5e8) return -1;
    //  * few pixels an image: the weights are brought into order for few pixels (512 -> 512 over 7 x 7: sixteen images 29 / 30, 32 images 32.5 / 31;
    //    with a stride, which leaves the unfolded operand small, from 14 x 14 32 / 37, 256 -> 256 from 28 x 28 32 images 37 / 29, eight 26.6 / 27.1)
    if (pixels < p.C || (image < 100 && pixels < 3ull * p.C)) return -1;
    // (few pixels in all, where the unfolded batch is as small as the weights: 320 -> 512 over 20 x 24, one image, 18.6 / 20.9, 272 -> 592 over 19 x 18
    // 16.8 / 18.7, 200 -> 560 over 12 x 9, four images, 16.2 / 17.2, 256 -> 736 over 25 x 22 19.7 / 21.5; but 136 -> 448 over 13 x 10, four images, 15.2 / 14.5,
    // channels that eight does not divide, whose weights the product wants padded, 278 -> 512 over 22 x 24 25.2 / 21.7, and from 600 pixels on
    // 448 -> 192 over 19 x 16, two images, 18.8 / 17.2)
    const bool strided = p.stride_h > 1 || p.stride_w > 1;
    if (!strided && pixels < 560 && p.C % 8 == 0 && p.C >= 150) return -1;
    if (strided && (image < 100 || pixels < 3000)) return -1;
    //  * many pixels: the patch kernel fills the chip too.  While there is not a block here for every compute unit this one is ahead
    //    (256 -> 256, 32 images of 14 x 14 29.4 / 23.6, sixteen 30.9 / 20.4, sixteen of 20 x 20 35.9 / 22.3, 24 of 16 x 16 24.7 / 22.4; 128 -> 128, eight of
    //    28 x 28 19.4 / 15.3), beyond only where rows are no whole vectors (128 -> 128, 32 of 28 x 28 21.8 / 20.3, 512 -> 512, eight of 28 x 28
    //    65.6 / 49; but 24 of 30 x 30 20.7 / 21.1, 24 of 32 x 32 18.1 / 21.9, 256 -> 256, eight of 56 x 56 46 / 70) or channels no whole chunks (72 -> 72, 32 of
    //    30 x 30 36.8 / 20.5, 130 -> 200, 32 of 19 x 19 40.3 / 22.3)
    const bool room = (pixels + 63) / 64 * ((p.O + 127) / 128) <= 256;
    if (whole_chunks && !room && (p.W % 8 == 0 || p.C < 128 || image > 800)) return -1;
    double time = 1e30;
    int index = -1, counter = 0;
    TH_BATCH3(TH_BATCH3_CONSIDER)
    if (index < 0) return -1;
    //  * the patch kernel in one round that is more than half full, where this one takes two or more (192 -> 512, nineteen images of 22 x 20
    //    30.2 / 37.6, 128 -> 768, fifteen, 26.8 / 30.5, 576 -> 816, seven of 28 x 28 75 / 87, with a stride 480 -> 16, 42 images of 45 x 46 41.7 / 58;
    //    less than half full 256 -> 278, 25 of 20 x 20 36.6 / 32.3, in two rounds 192 -> 691, twenty of 24 x 22 81 / 47); rows of an odd number of pixels
    //    lie at odd addresses there (128 -> 816, twelve of 24 x 25 46 / 35, 160 -> 816, 53 of 16 x 19 83 / 71; but 576 -> 816, seven of 26 x 29, 78 / 87)
    const uint64_t blocks = (pixels + q.ptile - 1) / q.ptile * q.co_tiles * q.splits;
    if (whole_chunks && p.W % 2 == 0) {
        const K3Load there = conv2d_k3_load(p, x, w);
        if (blocks > COMPUTE_UNITS && there.blocks && there.blocks <= there.at_once && there.blocks * 100 >= there.at_once * 58ull) return -1;
        //  * with a stride: rows in whole vectors of larger images there (160 -> 32, sixteen of 45 x 48 18.4 / 20, 224 -> 32 22.9 / 24.2; smaller ones
        //    416 -> 128, thirty of 30 x 32, 0.90), and three or four chunks in one round, with whole vectors or two blocks on a compute unit (96 -> 28,
        //    49 of 32 x 30 13.8 / 15.5, 128 -> 512, 27 of 23 x 20, 18.6 / 21.2, 128 -> 188, sixteen of 35 x 32, 17.1 / 18.1)
        if (strided && there.blocks && ((!there.flat && image > 500) || (p.C <= 128 && blocks <= COMPUTE_UNITS && (!there.flat || there.at_once > COMPUTE_UNITS)))) return -1;
    }
    //  * with a stride, more than one round where the unfolded batch has up to 4096 pixels (320 -> 693, nineteen of 24 x 27, 40 / 51, 408 -> 576 of
    //    27 x 25 52 / 60, 615 -> 528, 29 of 20 x 23, 73 / 86; in one round 384 -> 560 of 26 x 26 49 / 37)
    if (strided && blocks > COMPUTE_UNITS && pixels <= 4096 && K >= 2304) return -1;
    return index;
}

bool conv2d_batch3_plan(const ConvProblem& p, int dtype, const void* x, const void* w, uint32_t out[kConvPlanValues]) {
    if (p.N == 0 || p.O == 0 || p.HO == 0 || p.WO == 0) return false;
    Batch3Plan q{};
    const int index = plan_batch3(p, dtype, x, w, q);
    if (index < 0) return false;
    int counter = 0;
    out[0] = 4;
    out[1] = 3;
    TH_BATCH3(TH_BATCH3_DESCRIBE)
    const uint32_t plan[8] = {q.ptile, q.co_tiles, q.splits, q.chunks, q.chunks_per_split, q.plane, q.hp, q.wp};
    for (int i = 0; i < 8; ++i) out[5 + i] = plan[i];
    return true;
}

template <class T>
static int run_batch3(const ConvProblem& p, Batch3Plan& q, int index, const void* x, const void* w, const void* bias, void* y, hipStream_t stream) {
    q.hw = p.HO * p.WO;
    q.div_hw = FastDiv(q.hw);
    q.div_wo = FastDiv(p.WO);
    q.div_hp = FastDiv(q.hp);
    q.div_wp = FastDiv(q.wp);
    q.div_co_tiles = FastDiv(q.co_tiles);
    q.div_splits = FastDiv(q.splits);
    const uint32_t weight_blocks = (p.O + 15) / 16 * q.chunks, results = q.pixels * p.O;
    // (a block's weights are loaded a chunk ahead, the last ones behind the end)
    const size_t weight_bytes = (static_cast<size_t>(weight_blocks) + 1) * kBatch3Taps * 1024;
    char* scratch = nullptr;
    if (scratch_acquire(reinterpret_cast<void**>(&scratch), weight_bytes + (q.splits > 1 ? static_cast<size_t>(results) * q.splits * 4 : 0), stream) != TANNIC_SUCCESS) {
        (void)hipGetLastError();
        return TANNIC_UNSUPPORTED_DTYPE;      // no memory for the ordered weights: the kernels that come after need none, or less
    }
    q.weight_bytes = static_cast<uint32_t>(weight_bytes);
    uint4b* weights = reinterpret_cast<uint4b*>(scratch);
    float* partials = q.splits > 1 ? reinterpret_cast<float*>(scratch + weight_bytes) : nullptr;
    hipLaunchKernelGGL(conv2d_batch3_weights_kernel, dim3(weight_blocks), dim3(64 * kBatch3Taps), 0, stream, static_cast<const uint16_t*>(w), weights, p.O, p.C, FastDiv(q.chunks));
    int status = launch_status("conv2d_batch3_weights_kernel");
    if (status == TANNIC_SUCCESS) {
        status = [&]() -> int {
            int counter = 0;
            TH_BATCH3(TH_BATCH3_LAUNCH)
            return TANNIC_ERROR;
        }();
    }
    if (status == TANNIC_SUCCESS && q.splits > 1) {
        hipLaunchKernelGGL((conv2d_batch3_sum_kernel<T>), dim3((results + 255) / 256), dim3(256), 0, stream, partials, static_cast<T*>(y), p, q.splits, FastDiv(q.pixels), FastDiv(q.hw), results);
        status = launch_status("conv2d_batch3_sum_kernel");
    }
    scratch_release(scratch, stream);
    return status;
}

int conv2d_batch3(const ConvProblem& p, int dtype, const void* x, const void* w, const void* bias, void* y, hipStream_t stream) {
    if (p.N == 0 || p.O == 0 || p.HO == 0 || p.WO == 0) return TANNIC_UNSUPPORTED_DTYPE;
    Batch3Plan q{};
    const int index = plan_batch3(p, dtype, x, w, q);
    if (index < 0) return TANNIC_UNSUPPORTED_DTYPE;
    if (dtype == TANNIC_FLOAT16) return run_batch3<f16>(p, q, index, x, w, bias, y, stream);
    return run_batch3<bf16>(p, q, index, x, w, bias, y, stream);
}

}  // namespace th
