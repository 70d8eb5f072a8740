// conv2d of 16-bit types over few output pixels (one image, or a handful): 1x1 and 3x3 kernels, C a multiple of 32 (3x3 from 64 channels
// and 1x1 with stride 1, over plain rows and from 32 output channels on, mostly go on to conv2d_few3.hip and conv2d_few1.hip from here).
//
// With one image a layer's work is some 0.1 - 0.2 GFLOP and a megabyte of weights: a microsecond of the chip, if all of it
// takes part.  The tiles of the other kernels (64 output channels x up to 512 pixels, or 64 x 128 of a product) leave four
// to thirty-two blocks, each of which walks all channels alone, or need a copy in front and a pass over partial sums
// behind.  Here a block owns 16 MO output channels x 16 NP pixels of the flattened batch and its wavefronts split the
// channels, 32 at a time: no copy, no second kernel, and hundreds of blocks for one image.
//
// v_mfma_f32_16x16x32: a lane holds eight channels 8 (lane / 16) .. + 7 of one tap, of output channel lane % 16 and of pixel
// lane % 16.  The weights of its eight channels are 8 KS KS consecutive elements of OIHW, loaded as 16-byte pieces and
// regrouped into a fragment per tap in registers.  The signal is loaded value by value: pixels of a 16-lane group lie side by
// side in a row, the tap's byte offset is computed once per lane (one past every buffer where the tap falls beside the image or the
// pixel past the batch: the buffer resource's range check then gives the zero), and channels move by a scalar offset.
// So any pixel count, row width, stride and alignment of the signal runs at the same rate: one load instruction per 64
// values, and those instructions - O / (16 MO) x pixels x C KH KW / 64 of them - are what bounds the kernel.  The wavefronts'
// tiles meet in LDS, in a fixed order.  The 53 convolutions and 16 additions of a ResNet-50 over one image, recorded: 867 -> 405 us
// (512 -> 512 3x3 over 7 x 7 59 -> 13, 256 -> 256 over 14 x 14 26.7 -> 8.2, 256 -> 1024 1x1 10.7 -> 4.1).
// (src/cpu/conv2d.cpp:17-64; sums in fp32, rounded once.)
#include "conv_few.hpp"

namespace th {

struct FewPlan {
    uint32_t pixels, units, pixel_tiles, records;   // of the flattened batch; blocks of 32 channels; bytes of the signal
    FastDiv div_hw, div_wo, div_tiles;
};

constexpr uint32_t kFewOutside = 0x80000000u;   // not below any signal's bytes that this kernel takes (records <= 2^31): the load gives zero

template <class T, int KS, int MO, int NP, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void conv2d_few_kernel(const T* x, const T* w, const T* bias, T* y, ConvProblem p, FewPlan q) {
#if defined(__HIP_DEVICE_COMPILE__)
    constexpr int TAPS = KS * KS;
    __shared__ float partial[WAVES][MO][NP][16 * kFewPitch];
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64, r = lane % 16, kc = lane / 16;
    // neighbouring blocks share their output channels' weights
    uint32_t tile_o, tile_p;
    q.div_tiles.divmod(blockIdx.x, tile_o, tile_p);
    const uint32_t o0 = tile_o * 16 * MO, pixel0 = tile_p * 16 * NP;

    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(x), 0, q.records, 0x00020000);
    uint32_t at[NP][TAPS];
#pragma unroll
    for (int g = 0; g < NP; ++g) {
        const uint32_t pixel = pixel0 + g * 16 + r;
        uint32_t n, rest, ho, wo;
        q.div_hw.divmod(pixel < q.pixels ? pixel : 0, n, rest);
        q.div_wo.divmod(rest, ho, wo);
#pragma unroll
        for (int t = 0; t < TAPS; ++t) {
            // (unsigned: a coordinate before the image wraps and is past its end)
            const uint32_t h = ho * p.stride_h + t / KS - p.pad_h, v = wo * p.stride_w + t % KS - p.pad_w;
            const uint32_t offset = static_cast<uint32_t>(n * p.xs[0] + 8 * kc * p.xs[1] + h * p.xs[2] + v * p.xs[3]) * sizeof(T);
            at[g][t] = pixel < q.pixels && h < p.H && v < p.W ? offset : kFewOutside;
        }
    }
    // rows past the end read the last one: they only feed results that are never stored
    const T* weights[MO];
#pragma unroll
    for (int m = 0; m < MO; ++m) {
        const uint32_t o = o0 + m * 16 + r < p.O ? o0 + m * 16 + r : p.O - 1;
        weights[m] = w + o * p.ws[0] + 8 * kc * TAPS;
    }
    const uint32_t channel_bytes = static_cast<uint32_t>(p.xs[1]) * sizeof(T);

    float4f acc[MO][NP];
#pragma unroll
    for (int m = 0; m < MO; ++m)
#pragma unroll
        for (int g = 0; g < NP; ++g) acc[m][g] = float4f{0.0f, 0.0f, 0.0f, 0.0f};
    for (uint32_t u = wave; u < q.units; u += WAVES) {
        uint32_t raw[MO][4 * TAPS];
#pragma unroll
        for (int m = 0; m < MO; ++m)
#pragma unroll
            for (int i = 0; i < TAPS; ++i) {
                const uint4f_any piece = *reinterpret_cast<const uint4f_any*>(weights[m] + static_cast<size_t>(u) * 32 * TAPS + i * 8);
#pragma unroll
                for (int e = 0; e < 4; ++e) raw[m][4 * i + e] = piece[e];
            }
        const uint32_t base = u * 32 * channel_bytes;
#pragma unroll
        for (int t = 0; t < TAPS; ++t) {
            uint4f signal[NP];
#pragma unroll
            for (int g = 0; g < NP; ++g)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const uint32_t low = static_cast<uint16_t>(__builtin_amdgcn_raw_buffer_load_b16(rsrc, at[g][t], base + 2 * e * channel_bytes, 0));
                    const uint32_t high = static_cast<uint16_t>(__builtin_amdgcn_raw_buffer_load_b16(rsrc, at[g][t], base + (2 * e + 1) * channel_bytes, 0));
                    signal[g][e] = low | high << 16;
                }
#pragma unroll
            for (int m = 0; m < MO; ++m) {
                // element e of the fragment is channel e's tap t: half (TAPS e + t) of the lane's run
                uint4f fragment;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int i = TAPS * 2 * e + t, j = TAPS * (2 * e + 1) + t;
                    const uint32_t low = i % 2 ? raw[m][i / 2] >> 16 : raw[m][i / 2] & 0xFFFFu;
                    const uint32_t high = j % 2 ? raw[m][j / 2] & 0xFFFF0000u : raw[m][j / 2] << 16;
                    fragment[e] = low | high;
                }
#pragma unroll
                for (int g = 0; g < NP; ++g) acc[m][g] = few_mfma<T>(fragment, signal[g], acc[m][g]);
            }
        }
    }
    // accumulator: lane -> pixel lane % 16, value v -> output channel 4 (lane / 16) + v
#pragma unroll
    for (int m = 0; m < MO; ++m)
#pragma unroll
        for (int g = 0; g < NP; ++g)
#pragma unroll
            for (int v = 0; v < 4; ++v) partial[wave][m][g][(4 * kc + v) * kFewPitch + r] = acc[m][g][v];
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < 256 * MO * NP; i += 64 * WAVES) {
        const uint32_t in_tile = i % (16 * NP), row = i / (16 * NP), o = o0 + row, pixel = pixel0 + in_tile;
        if (o >= p.O || pixel >= q.pixels) continue;
        float sum = p.has_bias ? static_cast<float>(widen(bias[o * p.bs])) : 0.0f;
#pragma unroll
        for (int k = 0; k < WAVES; ++k) sum += partial[k][row / 16][in_tile / 16][row % 16 * kFewPitch + in_tile % 16];
        uint32_t n, rest, ho, wo;
        q.div_hw.divmod(pixel, n, rest);
        q.div_wo.divmod(rest, ho, wo);
        y[n * p.ys[0] + o * p.ys[1] + ho * p.ys[2] + wo * p.ys[3]] = narrow_result<T>(sum);
    }
#endif
}

template <class T, int KS, int MO, int NP, int WAVES>
static int launch_few(const ConvProblem& p, FewPlan q, const void* x, const void* w, const void* bias, void* y, hipStream_t stream, uint32_t* plan) {
    q.pixel_tiles = (q.pixels + 16 * NP - 1) / (16 * NP);
    q.div_tiles = FastDiv(q.pixel_tiles);
    const uint64_t blocks = static_cast<uint64_t>((p.O + 16 * MO - 1) / (16 * MO)) * q.pixel_tiles;
    if (blocks >= (1ull << 31)) return TANNIC_UNSUPPORTED_DTYPE;
    if (plan) {      // (only asked for)
        const uint32_t values[6] = {2, KS, MO, NP, WAVES, static_cast<uint32_t>(blocks)};
        for (int i = 0; i < 6; ++i) plan[i] = values[i];
        return TANNIC_SUCCESS;
    }
    hipLaunchKernelGGL((conv2d_few_kernel<T, KS, MO, NP, WAVES>), dim3(static_cast<uint32_t>(blocks)), dim3(64 * WAVES), 0, stream, static_cast<const T*>(x),
                       static_cast<const T*>(w), static_cast<const T*>(bias), static_cast<T*>(y), p, q);
    return launch_status("conv2d_few_kernel");
}

// Multiply-adds up to which this kernel is taken, its output channels counted in whole tiles of 16 (a tile costs its loads whatever it
// holds): its loads grow with the work from the first pixel on, the other kernels' time hardly does while their blocks are few.
// Where the lines lie (fp16, replayed calls on one box, us, this kernel / the others; from before conv2d_few3.hip and conv2d_few1.hip, which now have
// most of what lies below them and are faster there):
//   3x3, C = 64 or 128 with a stride   240 M   64 @56: batch 1 6.5 / 10.0, 2 8.7 / 10.1, 4 12.3 / 10.3; 128 @56 s2: 8.7 / 13.2, 11.3 / 16.6, 19.4 / 16.8
//   other 3x3                          470 M   128 @28: batch 1 6.7 / 13.2, 4 12.7 / 19.3, 8 21.4 / 18.8; 256 @14: 8.2 / 26.7, 14.4 / 17.5, 26.8 / 24.8;
//                                              512 @7: 13.0 / 58.9, 22.5 / 60.6, 37.5 / 20.0
//   ... C > 512 (a wavefront's second turn), s2 150 M   1248->39 @11x12, batch 9, 175 M: 32.8 / 22.3; 1024->100 @5x7, batch 27, 334 M: 39.3 / 22.6
//   1x1, images of whole 16 bytes, C < 128      20 M   64->64 @56: batch 1 3.6 / 4.4, 2 4.0 / 3.9, 4 4.5 / 4.0
//   ... C < 256                                 80 M   128->512 @28: batch 1 4.2 / 4.5, 2 5.1 / 4.6
//   ... more channels                          110 M   512->128 @28: batch 1 4.2 / 6.7, 2 5.0 / 6.8; 256->128 @56: 4.8 / 5.3, 6.1 / 5.4; 512->256 @28: 5.1 / 6.8, 7.4 / 6.9
//   1x1, other images, with a stride           210 M   512->1024 @28 s2: batch 1 6.7 / 10.5, 2 10.6 / 10.9, 4 17.5 / 11.4
//   ... without one                            300 M   256->1024 @14: batch 1 4.1 / 10.7, 4 6.6 / 10.5, 8 9.5 / 10.6; 1024->512 @14: 5.2 / 11.7, 11.1 / 15.1,
//                                                      20.2 / 16.5; 2048->512 @7: 7.9 / 11.7, 9.3 / 13.6, 15.8 / 16.1
//   ... without one, C < 256                   140 M   192->51 @140x29, batch 5, 250 M: 13.8 / 10.3; 128->54 @79, batch 3, 153 M: 8.4 / 7.2
//   ... without one, C < 128                   100 M   64->64 @37, batch 32, 179 M: 11.5 / 6.5; 64->109 @83x84, batch 3, 150 M: 8.6 / 6.6
// Up to 16 output channels under 256 or more channels are worth half a tile (the others' tiles are as empty, and their blocks fewer: 3x3 over
// 1, 1.4, 2 and 3 times the line, median of the time here over the time there 0.64, 0.60, 0.77 and 1.1; 1x1 over ragged images 0.74, 0.76, 0.80), but not
// in a 1x1 kernel over whole images (0.77, 1.41 and 1.51).
// (Before output channels counted in tiles, an output head of one channel came here with sixteen times the loads: 512->1 3x3 @65x112,
// batch 12, 202 us here, 64 there.)
static bool few_work(const ConvProblem& p, uint64_t pixels) {
    const bool strided = p.stride_h > 1 || p.stride_w > 1, whole = static_cast<uint64_t>(p.HO) * p.WO % 8 == 0;
    double most = strided ? 210e6 : p.C < 128 ? 100e6 : p.C < 256 ? 140e6 : 300e6;
    if (p.KH == 3) most = p.C < 128 || (strided && p.C < 256) ? 240e6 : strided && p.C > 512 && p.O > 16 ? 150e6 : 470e6;
    else if (whole) most = p.C < 128 ? 20e6 : p.C < 256 ? 80e6 : 110e6;
    double channels = (static_cast<uint64_t>(p.O) + 15) / 16 * 16;
    if (p.O <= 16 && p.C >= 256 && (p.KH == 3 || strided || !whole)) channels = 8;
    return static_cast<double>(pixels) * channels * p.C * (p.KH * p.KW) <= most;
}

// Tiles per block: one while there are fewer than some 300, so that every compute unit has a block; then two (output channels where
// the signal is expensive - nine taps, or every other pixel of a row - and pixels where the weights are), then four, whose
// accumulated tiles fit the static LDS up to eight wavefronts (us with 1, 2 channels, 4 tiles: 3x3 256 @14 batch 1 8.2, 10.1, 13.7, batch 2
// 13.3, 10.4, 13.8, batch 4 23.4, 17.9, 14.4; 1x1 1024->512 @14 with 1 and 2 pixels 5.8, 5.2, batch 4 14.3, 11.1).  Up to 16 output
// channels are never two tiles of them.
template <class T, int KS, int WAVES>
static int few_shape(const ConvProblem& p, const FewPlan& q, uint64_t tiles, const void* x, const void* w, const void* bias, void* y, hipStream_t stream, uint32_t* plan) {
    const bool strided = p.stride_h > 1 || p.stride_w > 1;
    if (tiles < 300 || (p.O <= 16 && (KS == 3 || strided))) return launch_few<T, KS, 1, 1, WAVES>(p, q, x, w, bias, y, stream, plan);
    if constexpr (WAVES <= 8) {
        if (tiles >= 700 && p.O > 16 && (KS == 3 || strided || WAVES == 8)) return launch_few<T, KS, 2, 2, WAVES>(p, q, x, w, bias, y, stream, plan);
    }
    if constexpr (KS == 1) {
        if (!strided) return launch_few<T, KS, 1, 2, WAVES>(p, q, x, w, bias, y, stream, plan);
    }
    return launch_few<T, KS, 2, 1, WAVES>(p, q, x, w, bias, y, stream, plan);
}

template <class T, int KS>
static int run_few(const ConvProblem& p, const void* x, const void* w, const void* bias, void* y, hipStream_t stream, uint32_t* plan, bool& few3_asked) {
    constexpr int64_t TAPS = KS * KS;
    const uint64_t pixels = static_cast<uint64_t>(p.N) * p.HO * p.WO;
    if (pixels == 0 || p.O == 0 || p.C == 0 || p.C % 32 != 0) return TANNIC_UNSUPPORTED_DTYPE;
    // the weights of a lane's eight channels are one run of memory
    if (TAPS > 1 && (p.ws[3] != 1 || p.ws[2] != KS)) return TANNIC_UNSUPPORTED_DTYPE;
    if (p.ws[1] != TAPS || p.ws[0] < 0) return TANNIC_UNSUPPORTED_DTYPE;
    for (int d = 0; d < 4; ++d)
        if (p.xs[d] < 0) return TANNIC_UNSUPPORTED_DTYPE;
    // byte offsets into the signal are 31-bit (an extent of one may have any stride: it is not counted)
    const uint64_t extent[4] = {p.N, p.C, p.H, p.W};
    uint64_t last = 0;
    for (int d = 0; d < 4; ++d) {
        if (extent[d] > 1 && static_cast<uint64_t>(p.xs[d]) >= (1ull << 30)) return TANNIC_UNSUPPORTED_DTYPE;
        if (extent[d] > 1) last += (extent[d] - 1) * static_cast<uint64_t>(p.xs[d]);
        if (last >= (1ull << 30)) return TANNIC_UNSUPPORTED_DTYPE;
    }
    if (pixels >= (1ull << 24)) return TANNIC_UNSUPPORTED_DTYPE;
    const bool work = few_work(p, pixels);
    if constexpr (KS == 3) {
        // (from 256 output channels on also beyond the line: few3's own rule then says where it ends)
        few3_asked = work || p.O >= 256;
        const int rc = few3_asked ? conv2d_few3(p, dtype_code<T>(), x, w, bias, y, stream, plan) : TANNIC_UNSUPPORTED_DTYPE;
        if (rc != TANNIC_UNSUPPORTED_DTYPE) return rc;
    }
    if constexpr (KS == 1) {
        const int rc = !work ? TANNIC_UNSUPPORTED_DTYPE : conv2d_few1(p, dtype_code<T>(), true, x, w, bias, y, stream, plan);
        if (rc != TANNIC_UNSUPPORTED_DTYPE) return rc;
    }
    if (!work) return TANNIC_UNSUPPORTED_DTYPE;
    FewPlan q{};
    q.pixels = static_cast<uint32_t>(pixels);
    q.units = p.C / 32;
    q.records = static_cast<uint32_t>((last + 1) * sizeof(T));
    q.div_hw = FastDiv(p.HO * p.WO);
    q.div_wo = FastDiv(p.WO);
    const uint64_t tiles = static_cast<uint64_t>((p.O + 15) / 16) * ((pixels + 15) / 16);
    if (q.units >= 16) return few_shape<T, KS, 16>(p, q, tiles, x, w, bias, y, stream, plan);
    if (q.units >= 8) return few_shape<T, KS, 8>(p, q, tiles, x, w, bias, y, stream, plan);
    if (q.units >= 4) return few_shape<T, KS, 4>(p, q, tiles, x, w, bias, y, stream, plan);
    return few_shape<T, KS, 2>(p, q, tiles, x, w, bias, y, stream, plan);
}

static int choose_few(const ConvProblem& p, int dtype, const void* x, const void* w, const void* bias, void* y, hipStream_t stream, uint32_t* plan, bool& few3_asked) {
    few3_asked = false;
    if (p.KH != p.KW) return TANNIC_UNSUPPORTED_DTYPE;
    if (dtype == TANNIC_FLOAT16 && p.KH == 1) return run_few<f16, 1>(p, x, w, bias, y, stream, plan, few3_asked);
    if (dtype == TANNIC_FLOAT16 && p.KH == 3) return run_few<f16, 3>(p, x, w, bias, y, stream, plan, few3_asked);
    if (dtype == TANNIC_BFLOAT16 && p.KH == 1) return run_few<bf16, 1>(p, x, w, bias, y, stream, plan, few3_asked);
    if (dtype == TANNIC_BFLOAT16 && p.KH == 3) return run_few<bf16, 3>(p, x, w, bias, y, stream, plan, few3_asked);
    return TANNIC_UNSUPPORTED_DTYPE;
}

int conv2d_few(const ConvProblem& p, int dtype, const void* x, const void* w, const void* bias, void* y, hipStream_t stream, bool& few3_asked) {
    return choose_few(p, dtype, x, w, bias, y, stream, nullptr, few3_asked);
}

// (the addresses are asked for their alignment: the staged kernels do not take every one)
bool conv2d_few_plan(const ConvProblem& p, int dtype, const void* x, const void* w, uint32_t out[kConvPlanValues], bool& few3_asked) {
    return choose_few(p, dtype, x, w, nullptr, nullptr, nullptr, out, few3_asked) == TANNIC_SUCCESS;
}

}  // namespace th
