// Problem description shared by the convolution kernels.
#pragma once

#include "common.hpp"

namespace th {

// NCHW signal, OIHW kernel, cross-correlation with zero padding
// (src/cpu/conv2d.cpp:17-64).  Strides are element strides of each operand.
struct ConvProblem {
    uint32_t N, C, H, W;       // signal
    uint32_t O, KH, KW;        // kernel: O x C x KH x KW
    uint32_t HO, WO;           // output spatial size
    uint32_t pad_h, pad_w, stride_h, stride_w;
    int64_t xs[4], ws[4], ys[4];
    int64_t bs;                // element stride of the bias (the CPU path reads it as 1, src/cpu/conv2d.cpp:86)
    bool has_bias;
};

// The plan of the kernel that would take a problem, for tannic_hip_conv2d_plan: which of the kernels below, then its parameters and
// the parts of its plan that say where a tile's windows lie (named in include/tannic_hip.h).
constexpr int kConvPlanValues = 20;
// true where the kernel takes the problem (conv2d_split, conv2d_f32, conv2d_few, conv2d_batch3 and, through the tiles over images,
// conv2d_pointwise launch what these report)
bool conv2d_split_plan(const ConvProblem& p, int dtype, const void* x, const void* w, uint32_t out[kConvPlanValues]);
bool conv2d_pointwise_plan(const ConvProblem& p, int dtype, const void* x, const void* w, uint32_t out[kConvPlanValues]);
bool conv2d_batch3_plan(const ConvProblem& p, int dtype, const void* x, const void* w, uint32_t out[kConvPlanValues]);
bool conv2d_f32_plan(const ConvProblem& p, int dtype, const void* x, const void* w, uint32_t out[kConvPlanValues]);
bool conv2d_few_plan(const ConvProblem& p, int dtype, const void* x, const void* w, uint32_t out[kConvPlanValues], bool& few3_asked);

// Each returns TANNIC_UNSUPPORTED_DTYPE when the problem does not meet its
// conditions, so that the caller can try the next, more general kernel.
// 16-bit 1x1 and 3x3 over few output pixels; few3_asked: whether conv2d_few3 has been asked, and has refused if this returns UNSUPPORTED_DTYPE
int conv2d_few(const ConvProblem& p, int dtype, const void* x, const void* w, const void* bias, void* y, hipStream_t stream, bool& few3_asked);
// 16-bit 3x3 from 64 channels and 32 output channels on, few output pixels, the weights and the signal staged in LDS (what conv2d_few asks first, and
// what conv2d_batch3 leaves); `plan`: only asked which tiles it would take
int conv2d_few3(const ConvProblem& p, int dtype, const void* x, const void* w, const void* bias, void* y, hipStream_t stream, uint32_t* plan = nullptr);
// 16-bit 1x1, stride 1, the same way; `few`: below conv2d_few's line
int conv2d_few1(const ConvProblem& p, int dtype, bool few, const void* x, const void* w, const void* bias, void* y, hipStream_t stream, uint32_t* plan = nullptr);
bool conv2d_k1_takes(const ConvProblem& p, int dtype, const void* x, const void* w, const void* y);
int conv2d_k1(const ConvProblem& p, int dtype, const void* x, const void* w, const void* bias, void* y, hipStream_t stream);
int conv2d_pointwise(const ConvProblem& p, int dtype, const void* x, const void* w, const void* bias, void* y, hipStream_t stream);
int conv2d_stem(const ConvProblem& p, int dtype, const void* x, const void* w, const void* bias, void* y, hipStream_t stream);
int conv2d_k3(const ConvProblem& p, int dtype, const void* x, const void* w, const void* bias, void* y, hipStream_t stream);
int conv2d_resident(const ConvProblem& p, int dtype, const void* x, const void* w, const void* bias, void* y, hipStream_t stream);
int conv2d_patch(const ConvProblem& p, int dtype, const void* x, const void* w, const void* bias, void* y, hipStream_t stream);
// fp32 1x1 (from 100 channels on, 140 under fewer than 128 output channels) and 3x3 (from 32) on the 16-bit matrix pipe, every value as three bfloat16 values
int conv2d_split(const ConvProblem& p, int dtype, const void* x, const void* w, const void* bias, void* y, hipStream_t stream);
// the blocks of conv2d_k3 for a 16-bit 3x3 problem (none where it does not take it), how many of them the chip runs at once, whether rows are no
// whole aligned vectors
struct K3Load {
    uint64_t blocks;
    uint32_t at_once;
    bool flat;
};
K3Load conv2d_k3_load(const ConvProblem& p, const void* x, const void* w);
// 16-bit 3x3, a batch of small maps under many channels, over the flattened batch
int conv2d_batch3(const ConvProblem& p, int dtype, const void* x, const void* w, const void* bias, void* y, hipStream_t stream);
// the time (us) that conv2d_f32 is expected to take; negative where it does not take the problem
double conv2d_f32_expected(const ConvProblem& p, int dtype, const void* x, const void* w);
int conv2d_f32(const ConvProblem& p, int dtype, const void* x, const void* w, const void* bias, void* y, hipStream_t stream);
int conv2d_gather32(const ConvProblem& p, int dtype, const void* x, const void* w, const void* bias, void* y, hipStream_t stream);
int conv2d_unfold(const ConvProblem& p, int dtype, const void* x, const void* w, const void* bias, void* y, hipStream_t stream);
// few output pixels per image under many channels (fp16, bf16, fp32): the whole batch unfolded side by side, one product
int conv2d_unfold_batch(const ConvProblem& p, int dtype, const void* x, const void* w, const void* bias, void* y, hipStream_t stream);
int conv2d_unfold_batch_any(const ConvProblem& p, int dtype, const void* x, const void* w, const void* bias, void* y, hipStream_t stream);
int conv2d_mfma(const ConvProblem& p, int dtype, const void* x, const void* w, const void* bias, void* y, hipStream_t stream);

}  // namespace th
