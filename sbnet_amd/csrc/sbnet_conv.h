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
};

// Whether the kernel takes the sizes (32-bit byte offsets, LDS).
bool conv_fits(const ConvArgs& c);
hipError_t launch_block_conv(const ConvArgs& c, hipStream_t stream);

}  // namespace sbnet
