// 3x3 conv2d of 16-bit types over few output pixels, from 64 channels (a multiple of 32) and 32 output channels on.
//
// The layers of one image, or of a handful: 0.1 to 0.9 billion multiply-adds under up to five megabytes of weights.  A block owns 8, 16 or
// 32 output channels x 16 to 64 pixels of one image and its wavefronts split the channels, 32 at a time; no copy in front, no pass behind,
// some hundred blocks.  What the kernel in conv2d_few.hip spends these layers' time on is how it loads: a signal value per lane and tap,
// two bytes at a time (72 load instructions for 16 pixels and 32 channels), and weights of which every lane reads its own 144 bytes, so that each
// instruction touches 64 lines and each line is asked for by up to nine of them.  Here
//   * the signal's rows under the tile are one run of memory in every channel's plane: it is loaded once in pieces of eight elements at any
//     alignment, transposed in registers (eight channels x eight elements), and put channels last into LDS, where a tap of 16 pixels x 32
//     channels is ONE 16-byte read per lane at an address that never changes; a tap beside the image reads a slot of zeros;
//   * a wavefront's weights, 576 bytes of every row, go straight into LDS in whole kilobytes (the pieces of every fourth row turned by one, so that the
//     reads of 16 rows fall on all banks) and are regrouped into a fragment per tap from there.
// Bound by bytes through the L2s - the weights come once per tile of pixels, 0.17 us for 32 channels of a block of 16 x 16 - and by start and
// end, about 3.5 us.  fp16, recorded calls, weights from memory, us before / here: one image 64 -> 64 over 56 x 56 6.4 / 5.7, 128 -> 128 over 28 x 28
// 7.5 / 5.0, 256 -> 256 over 14 x 14 9.0 / 5.1, 512 -> 512 over 7 x 7 14.7 / 7.1, with stride 2 128 at 56 9.3 / 6.6, 256 at 28 10.3 / 6.6, 512 at 14 16.9 / 6.4;
// four images of 256 -> 256 15.2 / 7.4, of 512 -> 512 22.6 / 8.1, eight of them 19.0 / 12.8 and 21.1 / 10.0.
// (src/cpu/conv2d.cpp:17-64; sums in fp32, the wavefronts' shares of the channels in a fixed order, rounded once; with another number of wavefronts than
// conv2d_few.hip takes for the same problem the order is another.)
#include "conv_few.hpp"

namespace th {

typedef __attribute__((address_space(3))) void* lds_void3;

struct Few3Plan {
    uint32_t units;              // blocks of 32 channels
    uint32_t per_image, tiles;   // tiles of pixels of an image, of all of them
    uint32_t pitch;              // 16-byte slots of a group of eight channels in LDS: the longest run of the signal and a slot of zeros
    uint32_t w_records;          // bytes of the weights
    FastDiv div_tiles, div_image, div_wo;
};

// element `pos` of a run lies in slot: eight neighbours, which one lane writes, and eight lanes' first elements both fall on different banks
__device__ inline uint32_t few3_slot(uint32_t pos) { return (pos & ~7u) | ((pos ^ (pos >> 3)) & 7u); }

template <int ROWS> constexpr uint32_t few3_weight_bytes() { return (ROWS * 36 + 63) / 64 * 1024; }

template <class T, int ROWS, int NP, int WAVES, int PASSES>
__global__ __launch_bounds__(64 * WAVES) void conv2d_few3_kernel(const T* x, const T* w, const T* bias, T* y, ConvProblem p, Few3Plan q) {
#if defined(__HIP_DEVICE_COMPILE__)
    constexpr int MO = (ROWS + 15) / 16, LOADS = (ROWS * 36 + 63) / 64;
    constexpr uint32_t W_BYTES = few3_weight_bytes<ROWS>();
    extern __shared__ __align__(16) unsigned char lds[];
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64, r = lane % 16, kc = lane / 16;
    // blocks that share weights run on one die
    const uint32_t die = blockIdx.x % 8, more = gridDim.x % 8;
    const uint32_t id = die * (gridDim.x / 8) + (die < more ? die : more) + blockIdx.x / 8;
    uint32_t tile_o, tile_p, n, in_image;
    q.div_tiles.divmod(id, tile_o, tile_p);
    q.div_image.divmod(tile_p, n, in_image);
    const uint32_t o0 = tile_o * ROWS, pixel0 = in_image * 16 * NP, pixels = p.HO * p.WO;
    const uint32_t last = pixel0 + 16 * NP < pixels ? pixel0 + 16 * NP - 1 : pixels - 1;
    // the rows of the signal under the tile: one run of a channel's plane
    const int32_t top = static_cast<int32_t>(q.div_wo.div(pixel0) * p.stride_h) - static_cast<int32_t>(p.pad_h);
    const int32_t bottom = static_cast<int32_t>(q.div_wo.div(last) * p.stride_h) - static_cast<int32_t>(p.pad_h) + 3;
    const uint32_t row0 = top > 0 ? top : 0, row_end = bottom < static_cast<int32_t>(p.H) ? (bottom > 0 ? bottom : 0) : p.H;
    const uint32_t run = row_end > row0 ? (row_end - row0) * p.W : 0, pieces = (run + 7) / 8;

    unsigned char* const w_lds = lds + wave * (W_BYTES + 64 * q.pitch);
    unsigned char* const s_lds = w_lds + W_BYTES + kc * 16 * q.pitch;
    const uint32_t zeros = q.pitch - 1;
    uint32_t at[NP][9];
#pragma unroll
    for (int g = 0; g < NP; ++g) {
        const uint32_t pixel = pixel0 + g * 16 + r <= last ? pixel0 + g * 16 + r : last;
        uint32_t ho, wo;
        q.div_wo.divmod(pixel, ho, wo);
#pragma unroll
        for (int t = 0; t < 9; ++t) {
            // (unsigned: a coordinate before the image wraps and is past its end)
            const uint32_t h = ho * p.stride_h + t / 3 - p.pad_h, v = wo * p.stride_w + t % 3 - p.pad_w;
            at[g][t] = 16 * (h < p.H && v < p.W ? few3_slot((h - row0) * p.W + v) : zeros);
        }
    }
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(w), 0, q.w_records, 0x00020000);
    uint32_t from[LOADS];
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
        const uint32_t slot = i * 64 + lane, row = slot / 36 < ROWS ? slot / 36 : ROWS - 1, turned = slot % 36 + 36 - (row >> 2) % 4;
        const uint32_t o = o0 + row < p.O ? o0 + row : p.O - 1;
        from[i] = o * static_cast<uint32_t>(p.ws[0]) * sizeof(T) + (turned < 36 ? turned : turned - 36) * 16;
    }
    uint32_t of_weights[9];
#pragma unroll
    for (int j = 0; j < 9; ++j) {
        const uint32_t turned = 9 * kc + j + ((ROWS == 8 ? r % 8 : r) >> 2);
        of_weights[j] = 16 * ((ROWS == 8 ? r % 8 : r) * 36 + (turned < 36 ? turned : turned - 36));
    }
    if (r == 0) *reinterpret_cast<uint4f*>(s_lds + 16 * zeros) = uint4f{0, 0, 0, 0};

    float4f acc[MO][NP];
#pragma unroll
    for (int m = 0; m < MO; ++m)
#pragma unroll
        for (int g = 0; g < NP; ++g) acc[m][g] = float4f{0.0f, 0.0f, 0.0f, 0.0f};
    const T* const plane0 = x + n * p.xs[0] + 8 * kc * p.xs[1] + static_cast<size_t>(row0) * p.W;
    for (uint32_t u = wave; u < q.units; u += WAVES) {
        const T* const plane = plane0 + u * 32 * p.xs[1];
        uint4f_any v[PASSES][8];
        // (lanes past the run's last piece do it over)
        auto start_of = [&](uint32_t piece) {
            const uint32_t mine = piece < pieces ? piece : pieces - 1;
            return 8 * mine + 8 <= run ? 8 * mine : run - 8;
        };
        auto load = [&](uint32_t first) {
#pragma unroll
            for (int i = 0; i < PASSES; ++i) {
                const T* const here = plane + start_of(first + i * 16 + r);
#pragma unroll
                for (int e = 0; e < 8; ++e) v[i][e] = *reinterpret_cast<const uint4f_any*>(here + e * p.xs[1]);
            }
        };
        auto put = [&](uint32_t first) {
#pragma unroll
            for (int i = 0; i < PASSES; ++i) {
                const uint32_t start = start_of(first + i * 16 + r);
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    uint4f column;
#pragma unroll
                    for (int k = 0; k < 4; ++k) column[k] = __builtin_amdgcn_perm(v[i][2 * k + 1][j / 2], v[i][2 * k][j / 2], j % 2 ? 0x07060302u : 0x05040100u);
                    *reinterpret_cast<uint4f*>(s_lds + 16 * few3_slot(start + j)) = column;
                }
            }
        };
        if (pieces) load(0);
#pragma unroll
        for (int i = 0; i < LOADS; ++i) __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_void3)(w_lds + i * 1024), 16, from[i], u * 576, 0, 0);
        if (pieces) put(0);
        for (uint32_t first = 16 * PASSES; first < pieces; first += 16 * PASSES) {
            load(first);
            put(first);
        }
        // the weights are in; what this wavefront wrote it reads in order
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        uint32_t raw[MO][36];
#pragma unroll
        for (int m = 0; m < MO; ++m)
#pragma unroll
            for (int j = 0; j < 9; ++j) {
                const uint4f piece = *reinterpret_cast<const uint4f*>(w_lds + m * (16 * 576) + of_weights[j]);
#pragma unroll
                for (int e = 0; e < 4; ++e) raw[m][4 * j + e] = piece[e];
            }
#pragma unroll
        for (int t = 0; t < 9; ++t) {
            uint4f signal[NP];
#pragma unroll
            for (int g = 0; g < NP; ++g) signal[g] = *reinterpret_cast<const uint4f*>(s_lds + at[g][t]);
#pragma unroll
            for (int m = 0; m < MO; ++m) {
                // element e of the fragment is channel e's tap t: half (9 e + t) of the lane's run
                uint4f fragment;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int i = 18 * e + t, j = 18 * e + 9 + t;
                    fragment[e] = __builtin_amdgcn_perm(raw[m][j / 2], raw[m][i / 2], (j % 2 ? 0x07060000u : 0x05040000u) | (i % 2 ? 0x0302u : 0x0100u));
                }
#pragma unroll
                for (int g = 0; g < NP; ++g) acc[m][g] = few_mfma<T>(fragment, signal[g], acc[m][g]);
            }
        }
        // nothing of this turn is read any more when the next one's pieces arrive
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
    // The wavefronts' tiles meet, in a fixed order.  Accumulator: lane -> pixel lane % 16, value v -> output channel 4 (lane / 16) + v
    __syncthreads();
    float* const partial = reinterpret_cast<float*>(lds);
    constexpr uint32_t SHARE = ROWS * NP * kFewPitch;
#pragma unroll
    for (int m = 0; m < MO; ++m)
#pragma unroll
        for (int g = 0; g < NP; ++g)
#pragma unroll
            for (int v = 0; v < 4; ++v)
                if (ROWS != 8 || kc < 2) partial[wave * SHARE + ((m * 16 + 4 * kc + v) * NP + g) * kFewPitch + r] = acc[m][g][v];
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < 16 * ROWS * NP; i += 64 * WAVES) {
        const uint32_t in_tile = i % (16 * NP), row = i / (16 * NP), o = o0 + row, pixel = pixel0 + in_tile;
        if (o >= p.O || pixel >= pixels) continue;
        float sum = p.has_bias ? static_cast<float>(widen(bias[o * p.bs])) : 0.0f;
#pragma unroll
        for (int k = 0; k < WAVES; ++k) sum += partial[k * SHARE + (row * NP + in_tile / 16) * kFewPitch + in_tile % 16];
        uint32_t ho, wo;
        q.div_wo.divmod(pixel, ho, wo);
        y[n * p.ys[0] + o * p.ys[1] + ho * p.ys[2] + wo * p.ys[3]] = narrow_result<T>(sum);
    }
#endif
}

// A block: output channels, tiles of 16 pixels, wavefronts; how often it loads signal pieces (16 lanes of eight elements); its LDS
struct Few3Shape {
    uint32_t rows, pixel_tiles, waves, passes;
    size_t lds;
    uint64_t blocks;
    Few3Plan plan;
};

// The shape with `rows` and `pixel_tiles`, and the time (us) it is expected to take; negative where LDS does not hold it.  Fitted to
// 370 timed calls (11 % off in the mean; the shape it picks 0.2 % slower than the best of them): start and end; every round of blocks waits
// for its loads and its own products; and what a compute unit loads for 32 channels of a block, weights and pieces of the signal.  (The blocks at once
// are counted by LDS and by eight wavefronts on a SIMD; registers hold two to four there, fewer blocks where a block is two wavefronts with little LDS.  The constants were fitted
// with that count.)
static double few3_expected(const ConvProblem& p, uint32_t rows, uint32_t pixel_tiles, Few3Shape& s) {
    const uint32_t pixels = p.HO * p.WO, units = p.C / 32, in_tile = 16 * pixel_tiles;
    s.rows = rows;
    s.pixel_tiles = pixel_tiles;
    const uint64_t per_image = (pixels + in_tile - 1) / in_tile, tiles = per_image * p.N;
    s.blocks = tiles * ((static_cast<uint64_t>(p.O) + rows - 1) / rows);
    // rows of the result that a tile touches at most, of the signal under them
    const uint64_t out_rows = std::min<uint64_t>((in_tile + p.WO - 2) / p.WO + 1, p.HO), in_rows = std::min<uint64_t>((out_rows - 1) * p.stride_h + 3, p.H);
    if (s.blocks >= (1ull << 31) || in_rows * p.W > 2048) return -1.0;
    const uint32_t run = static_cast<uint32_t>(in_rows * p.W);
    s.passes = ((run + 7) / 8 + 15) / 16;
    Few3Plan& q = s.plan;
    q.units = units;
    q.per_image = static_cast<uint32_t>(per_image);
    q.tiles = static_cast<uint32_t>(tiles);
    q.pitch = (run + 7) / 8 * 8 + 1;
    const size_t of_wave = (rows * 36 + 63) / 64 * 1024 + 64 * static_cast<size_t>(q.pitch);
    s.waves = units >= 16 && rows == 8 ? 16 : units >= 8 ? 8 : units >= 4 ? 4 : 2;
    while (s.waves > 2 && s.waves * of_wave > kFew3Lds) s.waves /= 2;
    s.lds = s.waves * of_wave;
    if (s.lds > kFew3Lds) return -1.0;
    const uint64_t at_once = 256 * std::min<uint64_t>(kFew3Lds / s.lds, 32 / s.waves), rounds = (s.blocks + at_once - 1) / at_once, load = (s.blocks + 255) / 256;
    const double turns = (units + s.waves - 1) / s.waves, passes = s.passes;
    const double products = std::max(1.0, rows / 16.0) * pixel_tiles, work = 0.047 * rows / 16 + 0.126 * passes + 0.141 * std::max(0.0, passes - 2);
    return 2.1 + rounds * (1.46 + 0.395 * turns * products) + load * units * work;
}

template <class T, int ROWS, int NP, int WAVES, int PASSES>
static int launch_few3(const ConvProblem& p, Few3Shape& s, const void* x, const void* w, const void* bias, void* y, hipStream_t stream) {
    s.plan.div_tiles = FastDiv(s.plan.tiles);
    s.plan.div_image = FastDiv(s.plan.per_image);
    s.plan.div_wo = FastDiv(p.WO);
    auto kernel = conv2d_few3_kernel<T, ROWS, NP, WAVES, PASSES>;
    static std::atomic<uint64_t> configured{0};
    if (int rc = raise_lds_limit(reinterpret_cast<const void*>(kernel), kFew3Lds, configured)) return rc;
    hipLaunchKernelGGL(kernel, dim3(static_cast<uint32_t>(s.blocks)), dim3(64 * WAVES), s.lds, stream, static_cast<const T*>(x), static_cast<const T*>(w),
                       static_cast<const T*>(bias), static_cast<T*>(y), p, s.plan);
    return launch_status("conv2d_few3_kernel");
}

template <class T, int ROWS, int NP>
static int launch_few3_waves(const ConvProblem& p, Few3Shape& s, const void* x, const void* w, const void* bias, void* y, hipStream_t stream) {
    const bool one = s.passes == 1;
    if constexpr (ROWS == 8) {
        if (s.waves == 16) return launch_few3<T, ROWS, NP, 16, 1>(p, s, x, w, bias, y, stream);      // (LDS holds no longer runs)
    }
    if constexpr (ROWS == 32) {
        if (s.waves == 8) return launch_few3<T, ROWS, NP, 8, 1>(p, s, x, w, bias, y, stream);        // (likewise)
    }
    else if (s.waves == 8) return one ? launch_few3<T, ROWS, NP, 8, 1>(p, s, x, w, bias, y, stream) : launch_few3<T, ROWS, NP, 8, 2>(p, s, x, w, bias, y, stream);
    if (s.waves == 4) return one ? launch_few3<T, ROWS, NP, 4, 1>(p, s, x, w, bias, y, stream) : launch_few3<T, ROWS, NP, 4, 2>(p, s, x, w, bias, y, stream);
    return one ? launch_few3<T, ROWS, NP, 2, 1>(p, s, x, w, bias, y, stream) : launch_few3<T, ROWS, NP, 2, 2>(p, s, x, w, bias, y, stream);
}

template <class T>
static int run_few3(const ConvProblem& p, const void* x, const void* w, const void* bias, void* y, hipStream_t stream, uint32_t* plan) {
    if (p.O < 32 || p.C < 64 || p.xs[3] != 1 || p.xs[2] != static_cast<int64_t>(p.W)) return TANNIC_UNSUPPORTED_DTYPE;
    // a run of at least eight elements under every tile that has any
    if (p.W < 8 && (p.pad_h > 1 || p.H < 2 || p.W < 4)) return TANNIC_UNSUPPORTED_DTYPE;
    if (p.H >= (1u << 20) || p.pad_h >= (1u << 20) || p.pad_w >= (1u << 20) || p.stride_h >= (1u << 20)) return TANNIC_UNSUPPORTED_DTYPE;
    // the weights are loaded into LDS in pieces of 16 bytes at multiples of four
    if (p.ws[0] % 2 != 0 || reinterpret_cast<uintptr_t>(w) % 4 != 0) return TANNIC_UNSUPPORTED_DTYPE;
    const uint64_t w_bytes = ((static_cast<uint64_t>(p.O) - 1) * p.ws[0] + static_cast<uint64_t>(p.C) * 9) * sizeof(T);
    if (p.ws[0] >= (1ll << 30) || w_bytes >= (1ull << 31)) return TANNIC_UNSUPPORTED_DTYPE;
    static constexpr uint32_t kShapes[5][2] = {{8, 1}, {16, 1}, {16, 2}, {32, 2}, {16, 4}};
    Few3Shape best{}, s{};
    double least = 1e30;
    for (auto& shape : kShapes) {
        const double expected = few3_expected(p, shape[0], shape[1], s);
        if (expected >= 0.0 && expected < least) { least = expected; best = s; }
    }
    // What the others would take, roughly (86 timed problems, a quarter off in the mean): a start, a chain over the channels, the multiply-adds, output
    // channels in tiles of 64.  Beyond 18 us, 9 under few channels, their larger tiles are mostly the faster ones, whatever this says (fp16, us there /
    // here: 22 images of 96 -> 608 over 12 x 12 15.2 / 23.0, 7 of 192 -> 160 over 31 x 31 19.6 / 27.5, 6 of 64 -> 285 over 34 x 34 15.8 / 20.5, 4 of 64 -> 64
    // over 56 x 56 10.0 / 12.8; but 28 of 704 -> 160 over 8 x 8 34.5 / 20.1).  140 drawn problems that it takes: 0.62 of the time in the mean.
    const double macs = 9.0 * p.N * p.HO * p.WO * p.C * ((p.O + 63) / 64 * 64);
    if (least > (p.C < 128 ? 9.0 : 18.0) || least > 4.26 + 0.0198 * p.C + 9.4e-9 * macs) return TANNIC_UNSUPPORTED_DTYPE;
    if (plan) {      // (only asked for)
        const uint32_t values[8] = {2, 3, (best.rows + 15) / 16, best.pixel_tiles, best.waves, static_cast<uint32_t>(best.blocks), best.rows, best.passes == 1 ? 1u : 2u};
        for (int i = 0; i < 8; ++i) plan[i] = values[i];
        return TANNIC_SUCCESS;
    }
    best.plan.w_records = static_cast<uint32_t>(w_bytes);
    if (best.rows == 8) return launch_few3_waves<T, 8, 1>(p, best, x, w, bias, y, stream);
    if (best.rows == 32) return launch_few3_waves<T, 32, 2>(p, best, x, w, bias, y, stream);
    if (best.pixel_tiles == 1) return launch_few3_waves<T, 16, 1>(p, best, x, w, bias, y, stream);
    if (best.pixel_tiles == 2) return launch_few3_waves<T, 16, 2>(p, best, x, w, bias, y, stream);
    return launch_few3_waves<T, 16, 4>(p, best, x, w, bias, y, stream);
}

// (the sizes that conv2d_few checks first, for its callers and for those that come here directly)
int conv2d_few3(const ConvProblem& p, int dtype, const void* x, const void* w, const void* bias, void* y, hipStream_t stream, uint32_t* plan) {
    const uint64_t pixels = static_cast<uint64_t>(p.N) * p.HO * p.WO;
    if (p.KH != 3 || p.KW != 3 || p.C % 32 != 0 || pixels == 0 || pixels >= (1ull << 24) || p.O == 0) return TANNIC_UNSUPPORTED_DTYPE;
    if (p.ws[3] != 1 || p.ws[2] != 3 || p.ws[1] != 9 || p.ws[0] < 0 || p.xs[0] < 0 || p.xs[1] < 0) return TANNIC_UNSUPPORTED_DTYPE;
    if (dtype == TANNIC_FLOAT16) return run_few3<f16>(p, x, w, bias, y, stream, plan);
    if (dtype == TANNIC_BFLOAT16) return run_few3<bf16>(p, x, w, bias, y, stream, plan);
    return TANNIC_UNSUPPORTED_DTYPE;
}

}  // namespace th
