// Host-side launch interface of the block convolution (sbnet_conv.hip).
#pragma once

#include <hip/hip_runtime_api.h>
#include <stddef.h>
#include <stdint.h>

namespace sbnet {

// Inference batch norm followed by ReLU; gamma == nullptr: none.
struct BnArgs {
    const float *gamma, *beta, *mean, *var;
    float eps;
};

// The batch norm and ReLU between a convolution and the one in front of it, as a training step's forward pass left them:
// z [rows, C] in front, act [rows, C] behind, the batch's mean and 1 / sqrt(variance + eps).  sums[(slot * C + c) * 2 ...]:
// GRAD_SLOTS partial pairs per channel that add up to (sum g, sum g * xhat), in double and added to atomically, one slot
// per XCD; g is the gradient behind the ReLU's mask, xhat = (z - mean) * inv.
constexpr int GRAD_SLOTS = 8;
struct NormGradArgs {
    const float *z, *act, *mean, *inv, *gamma;
    double* sums;
};

struct ConvArgs {
    // input: an image [N,H,W,C] read at block (n, bh, bw) = idx[3 * i ...] from pixel (oh + bh * U, ow + bw * V) on,
    // or, with idx == nullptr, a block stack: N blocks of H x W pixels
    const float* a;
    const int16_t* idx;
    int N, H, W, C;
    int U, V, oh, ow;
    int M;                    // listed blocks
    const int32_t* countDev;  // optional device-resident count, M is then the list's capacity
    // kernel [kh, kw, C, K], stride 1, VALID on each block
    const float* w;
    int K, kh, kw;
    int Ro, So;               // output pixels per block
    BnArgs pre, post;         // on the input's values, on the result's
    // output: pixels (bh * oU + r, bw * oV + s) of an image [oN,oH,oW,K], assigned or added to, or (oidx == nullptr) a
    // block stack [M,Ro,So,K]
    float* y;
    const int16_t* oidx;
    int oN, oH, oW, oU, oV;
    int add;
    NormGradArgs norm;        // launch_block_conv_grad only
};

// Whether the kernel takes the sizes (32-bit byte offsets, LDS).
bool conv_fits(const ConvArgs& c);
hipError_t launch_block_conv(const ConvArgs& c, hipStream_t stream);

// c and, on its result, the 1x1 convolution `next` (whose input is not looked at) in one launch; `done` is false, and nothing
// launched, where that does not apply: c must be larger than 1x1, with 16 input channels or more, 128 output channels or
// fewer and all channels multiples of four.
hipError_t launch_block_conv_next(const ConvArgs& c, const ConvArgs& next, hipStream_t stream, bool& done);

// Gradient of a convolution's input on block stacks, masked by the ReLU in front of it: a is the gradient of the output
// [M,H,W,C], w [K,kh,kw,C] the convolution's kernel, y [M,Ro,So,K] the result (Ro = H + kh - 1, So = W + kw - 1); adds to
// norm.sums.  Channels multiples of four, pointers 16-byte aligned (conv_grad_fits).
bool conv_grad_fits(const ConvArgs& c);
hipError_t launch_block_conv_grad(const ConvArgs& c, hipStream_t stream);

// Backward of the batch norm: g [rows, C], behind the mask, becomes the gradient of z in place; dgamma, dbeta (nullptr: not
// asked for).
hipError_t launch_norm_grad(float* g, const NormGradArgs& norm, uint32_t rows, int C, float* dgamma, float* dbeta,
                            hipStream_t stream);

// Gradients of up to three kernels at once: dw [kh,kw,C,K] = sum over all output pixels of act^T * dz.
struct WgradArgs {
    const float* act;         // [M,R,S,C]
    const float* dz;          // [M,R-kh+1,S-kw+1,K]
    int M, R, S, C, K, kh, kw;
    float* dw;
};
size_t wgrad_workspace_bytes(const WgradArgs* w, int count);
hipError_t launch_wgrad(const WgradArgs* w, int count, void* workspace, hipStream_t stream);

// A ReLU in place; x 16-byte aligned.
hipError_t launch_relu(float* x, size_t count, hipStream_t stream);

// Up to three kernels [kh,kw,C,K] (dims: four each) to [K,C,kh,kw] in one launch.
hipError_t launch_kernels(const float* const* from, const int32_t* dims, float* const* to, int count, hipStream_t stream);

// Up to ten matrix transposes [M][A][B] -> [M][B][A] in one launch (block stacks from planar to NHWC and back), which clears
// zeroCount floats besides.
struct TransposeArgs {
    const float* from;
    float* to;
    uint32_t M, A, B;
};
hipError_t launch_transposes(const TransposeArgs* t, int count, hipStream_t stream, float* zeros = nullptr, uint32_t zeroCount = 0);

}  // namespace sbnet
