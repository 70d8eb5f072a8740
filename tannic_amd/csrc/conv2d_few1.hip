// 1x1 conv2d of 16-bit types over few output pixels, stride 1 without padding, from 32 output channels on, C a multiple of 32: the layers
// of one image or of a handful.
//
// The split of conv2d_few.hip - a block owns 16 or 32 output channels x 16 or 32 pixels of one image, its wavefronts split the channels, 32 at a time,
// and meet in LDS - without its two-byte loads: the pixels of a tile are one run of memory in every channel's plane, so that 32 channels
// of 16 pixels are ONE load instruction (16 bytes a lane at any alignment, eight before) that goes to LDS as it is, rows of pixels, and comes back
// as a fragment through two transposing reads (ds_read_b64_tr_b16).  A wavefront that has several turns has the loads of two of
// them on their way.  Bound by start and end, some 2.5 us, then by weights and signal that cross the L2s once per tile of the
// other.  fp16, recorded calls, weights from memory, us before / here: one image 256 -> 1024 over 14 x 14 4.7 / 3.7, 1024 -> 256 5.5 / 4.5, 512 -> 128 over
// 28 x 28 4.8 / 3.7, 512 -> 2048 over 7 x 7 5.2 / 4.3, 2048 -> 512 8.8 / 6.4; four images of 1024 -> 256 9.3 / 7.0, of 2048 -> 512 10.5 / 7.1.
// (src/cpu/conv2d.cpp:17-64; sums in fp32, rounded once.)
#include "conv_few.hpp"

namespace th {

struct Few1Plan {
    uint32_t units;              // blocks of 32 channels
    uint32_t per_image, tiles;   // tiles of pixels of an image, of all of them
    FastDiv div_tiles, div_image, div_wo;
};

typedef short short4f __attribute__((ext_vector_type(4)));

template <class T, int MO, int NP, int WAVES, int TURNS>
__global__ __launch_bounds__(64 * WAVES) void conv2d_few1_kernel(const T* x, const T* w, const T* bias, T* y, ConvProblem p, Few1Plan q) {
#if defined(__HIP_DEVICE_COMPILE__)
    constexpr uint32_t ROW = 16 * NP;      // pixels of a channel in LDS
    extern __shared__ __align__(16) unsigned char lds[];
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64, r = lane % 16, kc = lane / 16;
    // blocks that share weights run on one die
    const uint32_t die = blockIdx.x % 8, more = gridDim.x % 8;
    const uint32_t id = die * (gridDim.x / 8) + (die < more ? die : more) + blockIdx.x / 8;
    uint32_t tile_o, tile_p, n, in_image;
    q.div_tiles.divmod(id, tile_o, tile_p);
    q.div_image.divmod(tile_p, n, in_image);
    const uint32_t o0 = tile_o * 16 * MO, pixels = p.HO * p.WO;
    // (an image's last tile ends with it: what it has in common with the one before is computed twice, to the same bits)
    const uint32_t pixel0 = in_image * ROW + ROW <= pixels ? in_image * ROW : pixels - ROW;

    T* const mine = reinterpret_cast<T*>(lds) + wave * (TURNS * 32 * ROW);
    const T* from[NP];
#pragma unroll
    for (int j = 0; j < NP; ++j) {
        const uint32_t piece = j * 64 + lane;
        from[j] = x + n * p.xs[0] + piece / (2 * NP) * p.xs[1] + pixel0 + piece % (2 * NP) * 8;
    }
    const T* weights[MO];
#pragma unroll
    for (int m = 0; m < MO; ++m) {
        const uint32_t o = o0 + m * 16 + r < p.O ? o0 + m * 16 + r : p.O - 1;
        weights[m] = w + o * p.ws[0] + 8 * kc;
    }
    // the transposing reads: lane 16 g + m points at channel 8 g + m / 4 (+ 4) and pixels 4 (m % 4) .. + 3, and has pixel m of channels 8 g .. 8 g + 7 then
    const T* const read_from = mine + (8 * kc + r / 4) * ROW + 4 * (r % 4);

    float4f acc[MO][NP];
#pragma unroll
    for (int m = 0; m < MO; ++m)
#pragma unroll
        for (int g = 0; g < NP; ++g) acc[m][g] = float4f{0.0f, 0.0f, 0.0f, 0.0f};
    for (uint32_t u = wave; u < q.units; u += TURNS * WAVES) {
        uint4f_any signal[TURNS][NP], raw[TURNS][MO];
#pragma unroll
        for (int t = 0; t < TURNS; ++t) {
            if (t > 0 && u + t * WAVES >= q.units) break;
            const uint32_t here = u + t * WAVES;
#pragma unroll
            for (int j = 0; j < NP; ++j) signal[t][j] = *reinterpret_cast<const uint4f_any*>(from[j] + here * 32 * p.xs[1]);
#pragma unroll
            for (int m = 0; m < MO; ++m) raw[t][m] = *reinterpret_cast<const uint4f_any*>(weights[m] + here * 32);
        }
#pragma unroll
        for (int t = 0; t < TURNS; ++t) {
            if (t > 0 && u + t * WAVES >= q.units) break;
#pragma unroll
            for (int j = 0; j < NP; ++j) *reinterpret_cast<uint4f*>(mine + t * (32 * ROW) + (j * 64 + lane) * 8) = signal[t][j];
        }
        asm volatile("" ::: "memory");      // (a wavefront reads what it wrote in order)
#pragma unroll
        for (int t = 0; t < TURNS; ++t) {
            if (t > 0 && u + t * WAVES >= q.units) break;
#pragma unroll
            for (int g = 0; g < NP; ++g) {
                using Lds = __attribute__((address_space(3))) short4f;
                const T* const at = read_from + t * (32 * ROW) + g * 16;
                const short4f low = __builtin_amdgcn_ds_read_tr16_b64_v4i16((Lds*)at), high = __builtin_amdgcn_ds_read_tr16_b64_v4i16((Lds*)(at + 4 * ROW));
                uint4f fragment;
                __builtin_memcpy(&fragment, &low, 8);
                __builtin_memcpy(reinterpret_cast<char*>(&fragment) + 8, &high, 8);
#pragma unroll
                for (int m = 0; m < MO; ++m) acc[m][g] = few_mfma<T>(raw[t][m], fragment, acc[m][g]);
            }
        }
        asm volatile("" ::: "memory");
    }
    // The wavefronts' tiles meet, in a fixed order.  Accumulator: lane -> pixel lane % 16, value v -> output channel 4 (lane / 16) + v
    __syncthreads();
    float* const partial = reinterpret_cast<float*>(lds);
    constexpr uint32_t SHARE = 16 * MO * NP * kFewPitch;
#pragma unroll
    for (int m = 0; m < MO; ++m)
#pragma unroll
        for (int g = 0; g < NP; ++g)
#pragma unroll
            for (int v = 0; v < 4; ++v) partial[wave * SHARE + ((m * 16 + 4 * kc + v) * NP + g) * kFewPitch + r] = acc[m][g][v];
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < 256 * MO * NP; i += 64 * WAVES) {
        const uint32_t in_tile = i % ROW, row = i / ROW, o = o0 + row;
        if (o >= p.O) continue;
        float sum = p.has_bias ? static_cast<float>(widen(bias[o * p.bs])) : 0.0f;
#pragma unroll
        for (int k = 0; k < WAVES; ++k) sum += partial[k * SHARE + (row * NP + in_tile / 16) * kFewPitch + in_tile % 16];
        uint32_t ho, wo;
        q.div_wo.divmod(pixel0 + in_tile, ho, wo);
        y[n * p.ys[0] + o * p.ys[1] + ho * p.ys[2] + wo * p.ys[3]] = narrow_result<T>(sum);
    }
#endif
}

template <class T, int MO, int NP, int WAVES, int TURNS>
static int launch_few1(const ConvProblem& p, Few1Plan q, const void* x, const void* w, const void* bias, void* y, hipStream_t stream) {
    constexpr size_t staged = WAVES * TURNS * NP * 1024, partial = WAVES * MO * NP * 16 * kFewPitch * 4, lds = staged > partial ? staged : partial;
    static_assert(lds <= 160 * 1024, "a block's LDS");
    const uint64_t blocks = static_cast<uint64_t>((p.O + 16 * MO - 1) / (16 * MO)) * q.tiles;
    auto kernel = conv2d_few1_kernel<T, MO, NP, WAVES, TURNS>;
    static std::atomic<uint64_t> configured{0};
    if (int rc = raise_lds_limit(reinterpret_cast<const void*>(kernel), lds, configured)) return rc;
    hipLaunchKernelGGL(kernel, dim3(static_cast<uint32_t>(blocks)), dim3(64 * WAVES), lds, stream, static_cast<const T*>(x), static_cast<const T*>(w),
                       static_cast<const T*>(bias), static_cast<T*>(y), p, q);
    return launch_status("conv2d_few1_kernel");
}

// A block's tiles of 16 output channels and pixels, its wavefronts
struct Few1Shape {
    uint32_t channel_tiles, pixel_tiles, waves;
    uint64_t blocks;
};

// The shape's expected time (us), negative where an image has fewer pixels than a tile.  Fitted to 1020 timed calls (12 % off in the
// mean; the shape it picks 0.3 % slower than the best of them).
static double few1_expected(const ConvProblem& p, uint32_t channel_tiles, uint32_t pixel_tiles, Few1Shape& s) {
    const uint32_t pixels = p.HO * p.WO, units = p.C / 32, products = channel_tiles * pixel_tiles;
    if (pixels < 16 * pixel_tiles) return -1.0;
    s.channel_tiles = channel_tiles;
    s.pixel_tiles = pixel_tiles;
    s.waves = units > 8 ? 16 : units > 4 ? 8 : units > 2 ? 4 : 2;      // (a wavefront without channels costs less than a second turn)
    s.blocks = static_cast<uint64_t>((pixels + 16 * pixel_tiles - 1) / (16 * pixel_tiles)) * p.N * ((static_cast<uint64_t>(p.O) + 16 * channel_tiles - 1) / (16 * channel_tiles));
    const uint32_t turns = units > s.waves ? 2 : 1, lds = s.waves * std::max(turns * pixel_tiles * 1024, products * 1280);
    const uint64_t at_once = 256 * std::min<uint64_t>(kFew3Lds / lds, 32 / s.waves), rounds = (s.blocks + at_once - 1) / at_once, load = (s.blocks + 255) / 256;
    const double pairs = (units + 2 * s.waves - 1) / (2 * s.waves);
    return 1.81 + rounds * (0.05 + 0.296 * products + 0.262 * pairs) + load * (units * (0.027 * channel_tiles + 0.0156 * pixel_tiles) + s.waves * (0.0016 * products + 0.012));
}

template <class T, int MO, int NP>
static int few1_waves(const ConvProblem& p, const Few1Shape& s, Few1Plan q, const void* x, const void* w, const void* bias, void* y, hipStream_t stream) {
    q.per_image = (p.HO * p.WO + 16 * NP - 1) / (16 * NP);
    q.tiles = q.per_image * p.N;
    q.div_tiles = FastDiv(q.tiles);
    q.div_image = FastDiv(q.per_image);
    q.div_wo = FastDiv(p.WO);
    if (s.waves == 16) return q.units <= 16 ? launch_few1<T, MO, NP, 16, 1>(p, q, x, w, bias, y, stream) : launch_few1<T, MO, NP, 16, 2>(p, q, x, w, bias, y, stream);
    if (s.waves == 8) return launch_few1<T, MO, NP, 8, 1>(p, q, x, w, bias, y, stream);
    if (s.waves == 4) return launch_few1<T, MO, NP, 4, 1>(p, q, x, w, bias, y, stream);
    return launch_few1<T, MO, NP, 2, 1>(p, q, x, w, bias, y, stream);
}

template <class T>
static int run_few1(const ConvProblem& p, bool few, const void* x, const void* w, const void* bias, void* y, hipStream_t stream, uint32_t* plan) {
    if (p.O < 32 || p.xs[3] != 1 || (p.xs[2] != static_cast<int64_t>(p.W) && p.H > 1)) return TANNIC_UNSUPPORTED_DTYPE;
    static constexpr uint32_t kShapes[3][2] = {{1, 1}, {1, 2}, {2, 2}};
    Few1Shape best{}, s{};
    double least = 1e30;
    for (auto& shape : kShapes) {
        const double expected = few1_expected(p, shape[0], shape[1], s);
        if (expected >= 0.0 && expected < least) { least = expected; best = s; }
    }
    // What is left to the others (366 drawn problems, fp16; us there / here).
    const double pixels = static_cast<double>(p.N) * p.HO * p.WO;
    const uint32_t in_image = p.HO * p.WO;
    if (few) {
        // Below conv2d_few's line: over images of whole 16 bytes nothing (44 problems 0.85 of the time in the mean, the worst 1.02).  Over others what a rough estimate of
        // that kernel's time (12 % off) puts at not much more than this one's: many results under channels that leave wavefronts idle (179 problems that
        // stay here 0.82, the worst 1.09; 5 of 320 -> 1920 over 6 x 6 5.9 / 7.1, 2 of 416 -> 288 over 30 x 30 6.8 / 7.8).
        const double there = 2.9 + 0.00152 * p.C + 2.04e-8 * pixels * p.C * ((p.O + 63) / 64 * 64) + 4.4e-7 * pixels * (p.C + p.O);
        if (least > 1e29 || (in_image % 8 != 0 && least > 0.9 * there)) return TANNIC_UNSUPPORTED_DTYPE;
    } else {
        // Beyond it: images of whole 16 bytes stay where they are (45 problems 1.06, the worst 2.1), and so does what the direct-to-LDS tiles over
        // images read, an even number of pixels under whole steps of 64 channels (6 of 320 -> 960 over 14 x 14 5.9 / 10.8), but for few results under many
        // channels (4 of 1024 -> 256 over 14 x 14 9.2 / 7.0), and 64 channels or fewer (2 of 64 -> 928 over 51 x 51 8.4 / 10.7).  The rest was on rows copied
        // into an aligned pitch or on loaders for any alignment (24 of 640 -> 32 over 25 x 25 17.9 / 8.3, 20 of 224 -> 207 over 13 x 13 10.4 / 6.1, 4 of
        // 2048 -> 512 over 7 x 7 10.5 / 7.1), up to 12.5 us (29 of 1152 -> 704 over 5 x 5 16.3 / 24.3).
        const bool tiles = in_image % 2 == 0 && p.C % 64 == 0 && !(p.C >= 512 && pixels * p.O <= 262144.0);
        if (in_image % 8 == 0 || tiles || p.C <= 64 || least > 12.5) return TANNIC_UNSUPPORTED_DTYPE;
    }
    if (plan) {      // (only asked for)
        const uint32_t values[8] = {2, 1, best.channel_tiles, best.pixel_tiles, best.waves, static_cast<uint32_t>(best.blocks), 16 * best.channel_tiles, p.C / 32 > best.waves ? 2u : 1u};
        for (int i = 0; i < 8; ++i) plan[i] = values[i];
        return TANNIC_SUCCESS;
    }
    Few1Plan q{};
    q.units = p.C / 32;
    if (best.channel_tiles == 2) return few1_waves<T, 2, 2>(p, best, q, x, w, bias, y, stream);
    if (best.pixel_tiles == 2) return few1_waves<T, 1, 2>(p, best, q, x, w, bias, y, stream);
    return few1_waves<T, 1, 1>(p, best, q, x, w, bias, y, stream);
}

int conv2d_few1(const ConvProblem& p, int dtype, bool few, const void* x, const void* w, const void* bias, void* y, hipStream_t stream, uint32_t* plan) {
    const uint64_t pixels = static_cast<uint64_t>(p.N) * p.HO * p.WO;
    if (p.KH != 1 || p.KW != 1 || p.C % 32 != 0 || pixels == 0 || pixels >= (1ull << 24) || p.O == 0 || p.C == 0) return TANNIC_UNSUPPORTED_DTYPE;
    if (p.stride_h != 1 || p.stride_w != 1 || p.pad_h || p.pad_w) return TANNIC_UNSUPPORTED_DTYPE;
    if (p.ws[1] != 1 || p.ws[0] < 0 || p.xs[0] < 0 || p.xs[1] < 0) return TANNIC_UNSUPPORTED_DTYPE;
    if (dtype == TANNIC_FLOAT16) return run_few1<f16>(p, few, x, w, bias, y, stream, plan);
    if (dtype == TANNIC_BFLOAT16) return run_few1<bf16>(p, few, x, w, bias, y, stream, plan);
    return TANNIC_UNSUPPORTED_DTYPE;
}

}  // namespace th
