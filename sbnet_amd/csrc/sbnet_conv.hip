// Convolution over the active blocks on the fp32 matrix cores of gfx950: gather, the batch norm and ReLU in front
// of a convolution, the convolution itself, and the paste or add of its result, without a block stack in between.
//
// Replaces, for the layers of sparse_conv.py in inference, the chain sparse_gather -> batch norm -> ReLU -> library
// convolution (-> batch norm -> ReLU -> ...) -> sparse_scatter (sbnet_tensorflow/benchmark/sparse_conv_lib.py:536-587,
// 677-723, 751-824).
#include "sbnet_device.h"
#include "sbnet_conv.h"

namespace sbnet {

// ---------------------------------------------------------------------------------------------
// k_block_conv: out[p, n] = sum over k = (tap, c) of in[p + tap, c] * w[k, n]
// ---------------------------------------------------------------------------------------------
//
// Rows p are the output pixels of all listed blocks, one after the other; k runs over the kernel's taps and the input
// channels of each, in the memory order of w [kh, kw, C, K], so w is the right-hand matrix as it stands and channel
// counts need no padding to a tap.  The input is an NHWC image read at the blocks' positions (pixels outside it are
// zeros, as sparse_gather has them) or a block stack [M, R, S, C].
//
// A wave computes 16 pixels x 16*FN channels with v_mfma_f32_16x16x4_f32 (full fp32 products and sums: the precision
// of the convolution it replaces).  Channels are the rows of the matrix instruction and pixels its columns, so that a
// lane ends with four consecutive channels of one pixel: 16-byte stores into NHWC memory.  Both operands go from memory
// straight to registers: with the instruction's k index spread as (lane / 16) * 4 + step, a lane's four pixel values
// are one 16-byte load, and 4 lanes read the 64 bytes of a pixel that 16 k need.  The fp32 matrix rate is low enough
// that the caches feed it (with FN = 2 a wave multiplies for 256 cycles per 16 k, for which it reads 1 KB of pixels and
// 2 KB of weights: 48 bytes a cycle for the four waves of a CU), and without LDS
// tiles there are no barriers: the problems are small (a few thousand pixels) and their time is a chain of latencies.
// Large products run at 80-95 TFLOP/s (of 153), with single-float loads at 35-40; from where the library is faster at
// them is a rule of the caller (sbnet_torch.cpp).
// CONV_DEPTH sets of operands are in flight per wave.
//
// Measured (MI355X, kernel trace): 85 blocks of 17x17x48, 3x3 to 48 channels (19 000 pixels, 0.8 GFLOP; 5.2 us at the
// rate of a large fp32 product): 15.7 us; 20.5 us with an exit inside a round of the loop and places found by division, 27 us
// while the loads of a step sat behind branches; the library convolution took 21 us behind 5 us of layout copies, and up
// to 800 us the first time a block count occurred.  A bottleneck block of 200 17x17x96 blocks: 33 us in three launches
// against about 300 us in 17 (31 us in two with NEXT, below).
//
// WK > 1: the WK waves of a workgroup split k among them and add up through LDS.  For launches whose tiles alone would
// leave most of the 1024 SIMDs idle.
//
// Batch norm of the input (pre) applies to values after the load, out-of-image zeros included, with mean, scale and shift
// read once per workgroup into LDS; batch norm of the result (post), for the convolution that follows, at the end.

typedef float acc_t __attribute__((ext_vector_type(4)));

constexpr int CONV_DEPTH = 2;   // operand sets in flight per wave (3: 1-8 % slower, 4: 2-10 %)
constexpr uint32_t W_OOB = 0x40000000u;   // beyond any kernel (conv_fits), alone and added to itself

// Kernels of one tap; of several, each at least the 16 k of a step long; of several shorter ones.
enum ConvTaps { TAPS_ONE = 0, TAPS_WIDE = 1, TAPS_NARROW = 2 };

struct ConvKernelArgs {
    ConvArgs c;
    FastDiv dC, dKw, dP, dSo;
    uint32_t kTot, kSteps;      // taps * C, ceil(kTot / 16)
    uint32_t rows, P;           // output pixels in all, per block
    uint32_t tilesP, tilesN;
    uint32_t aBytes, wBytes, yBytes;
    const float* w2;            // NEXT: the second kernel [K, K2]
    int K2;
    uint32_t w2Bytes;
};

__device__ __forceinline__ float relu_keep_nan(float v) { return v < 0.f ? 0.f : v; }

// An inference batch norm, y = (x - mean) * scale + beta, of channel c.  The mean is taken off first: folded into the shift
// it costs accuracy in proportion to |mean| / sigma (relative error 3e-7 at 10, 3e-5 at 1000; 5e-8 this way).
__device__ __forceinline__ void bn_read(const BnArgs& bn, uint32_t c, float& mean, float& scale, float& beta)
{
    mean = bn.mean[c];
    scale = bn.gamma[c] * (1.f / sqrtf(bn.var[c] + bn.eps));
    beta = bn.beta[c];
}

// Channels of the input's batch norm in LDS: the last four, past the end, make zeros of the zeros that k past the end reads
// (any channel's own could make an infinity, which the zero weights turn into NaN).
__host__ __device__ constexpr uint32_t pre_channels(int C) { return (((uint32_t)C + 3u) & ~3u) + 4u; }

// GRAD: the gradient of a convolution's input.  The same product with the kernel turned around, w [K, kh, kw, C] (n, then
// k: a lane's four k are one 16-byte load of w, too); the epilogue masks the result where the ReLU did and adds up what
// the batch norm's gradient needs, in fp32 over 16 pixels and in double from there on.
//
// NEXT: a 1x1 convolution on top, on the workgroup's own pixels, before anything is written: the result of the first is
// laid out as the matrix instructions want their input (a lane holds channels 16 * i + 4 * quad + 0..3 of its pixel, the
// four k of step i) and stays in registers.  All its channels are in one tile.
// Saves a launch, the stack in between and the second kernel's start: the 3x3 and the last 1x1 of a bottleneck on 200
// 17x17x96 blocks, 24 channels in between, take 20.1 us; 22.5 us one after the other (MI355X, kernel trace).
template <int FN, int WK, int VEC, bool PRE, int TAPS, bool GRAD, bool NEXT>
__global__ __launch_bounds__(256) void k_block_conv(ConvKernelArgs a)
{
    constexpr int WAVES = 4, WP = WAVES / WK;
    constexpr int TP = 16 * WP, TN = 16 * FN;
    extern __shared__ float lds[];
    const uint32_t cPad = PRE ? pre_channels(a.c.C) : 0u;
    float *const preMean = lds, *const preScale = lds + cPad, *const preBeta = lds + 2 * cPad;
    float *const postMean = lds + 3 * cPad, *const postScale = postMean + TN;   // (GRAD: mean and 1 / sigma)
    float* const postBeta = postMean + 2 * TN;                            // not GRAD
    double* const sums = reinterpret_cast<double*>(postMean + 2 * TN);    // [WP][TN][2], GRAD only
    float* const red = postMean + (GRAD ? 2 + 4 * WP : 3) * TN;           // [WP][WK][FN][64] x 4, WK > 1 only

    // Eight consecutive workgroups go to eight XCDs.  Each XCD takes one range of the pixels, so that its L2 fetches the
    // rows that neighbouring tiles share once; the tiles that differ in channels only follow each other.  (Tiles dealt to
    // the XCDs in turn fetch 3.3 times the image's part for a 3x3 kernel.  us a bottleneck: 250 blocks of 9x9x128 21.5 / 18.4,
    // 25 of 20x20x192 22.2 / 19.6, 60 of 22x22x128 27.6 / 25.4; single convolutions as before.)
    uint32_t rows = a.rows;
    if (a.c.countDev) rows = min(rows, (uint32_t)max(*a.c.countDev, 0) * a.P);
    const uint32_t tiles = (rows + TP - 1) / TP, perXcd = (tiles + 7u) >> 3;
    const uint32_t g = blockIdx.x >> 3;
    const uint32_t tn = g % a.tilesN, inXcd = g / a.tilesN, tp = (blockIdx.x & 7u) * perXcd + inXcd;
    if (inXcd >= perXcd || tp >= tiles) return;   // (the whole workgroup)

    const uint32_t tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, quad = lane >> 4;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6)), wk = wave % WK, wp = wave / WK;
    const uint32_t n0 = tn * TN;
    const bool post = a.c.post.gamma != nullptr;

    // The wave's pixels: one per lane, the same for the four quads.
    int h0, w0;
    uint32_t base;   // byte offset of channel 0 of the pixel under tap (0, 0)
    {
        const uint32_t row = tp * TP + wp * 16 + l16;
        bool ok = row < rows;
        const uint32_t ib = fdiv(ok ? row : 0u, a.dP), p = (ok ? row : 0u) - ib * a.P;
        const uint32_t r = fdiv(p, a.dSo), s = p - r * (uint32_t)a.c.So;
        int n = (int)ib;
        h0 = (int)r;
        w0 = (int)s;
        if (a.c.idx) {
            const int16_t* t = a.c.idx + (size_t)ib * 3;
            n = t[0];
            h0 += a.c.oh + t[1] * a.c.U;
            w0 += a.c.ow + t[2] * a.c.V;
            ok = ok && (unsigned)n < (unsigned)a.c.N;
        }
        base = (((uint32_t)n * (uint32_t)a.c.H + (uint32_t)h0) * (uint32_t)a.c.W + (uint32_t)w0) * (uint32_t)a.c.C * 4u;
        if (!ok) h0 = -0x40000000;   // outside the image under every tap
    }

    // Where the lane's pixel goes (the list is read here, not behind the products).
    bool outOk = tp * TP + wp * 16 + l16 < rows;
    uint32_t outPix = tp * TP + wp * 16 + l16;
    if (!GRAD && a.c.oidx) {
        const uint32_t row = outOk ? outPix : 0u, ib = fdiv(row, a.dP), p = row - ib * a.P;
        const uint32_t r = fdiv(p, a.dSo), s = p - r * (uint32_t)a.c.So;
        const int16_t* t = a.c.oidx + (size_t)ib * 3;
        const int on = t[0], oh = t[1] * a.c.oU + (int)r, ow = t[2] * a.c.oV + (int)s;
        outOk = outOk && (unsigned)on < (unsigned)a.c.oN && (unsigned)oh < (unsigned)a.c.oH && (unsigned)ow < (unsigned)a.c.oW;
        outPix = ((uint32_t)on * (uint32_t)a.c.oH + (uint32_t)oh) * (uint32_t)a.c.oW + (uint32_t)ow;
    }

    const rsrc_t ra = make_rsrc(a.c.a, a.aBytes);
    const uint32_t per = (a.kSteps + WK - 1) / WK;
    const uint32_t sBeg = wk * per, sEnd = min(sBeg + per, a.kSteps);
    const uint32_t K = (uint32_t)a.c.K, C = (uint32_t)a.c.C;

    // Where the lane's k of the next step to load is: pixel, channel and byte offset, moved on by 16 k a step.  Found by
    // division once: divisions and products per step cost more cycles than the matrix instructions.  Within a row of taps
    // the input lies in the order of k (backwards in GRAD, tap by tap).
    constexpr int DIR = GRAD ? -1 : 1, LANE_K = VEC == 4 ? 1 : 4;   // (four k share a tap, or each has its own)
    struct Place {
        uint32_t k, c, off;
        int h, w;
    } at[LANE_K];
#pragma unroll
    for (int j = 0; j < LANE_K; ++j) {
        Place& t = at[j];
        t.k = sBeg * 16u + quad * 4u + j;
        const uint32_t tap = TAPS ? fdiv(t.k, a.dC) : 0u;
        const int dr = TAPS ? (int)fdiv(tap, a.dKw) : 0, ds = (int)tap - dr * a.c.kw;
        t.c = t.k - tap * C;
        t.h = h0 + DIR * dr;
        t.w = w0 + (TAPS ? DIR * ds : 0);
        t.off = base + (TAPS ? (uint32_t)(DIR * (dr * a.c.W + ds)) * C * 4u : 0u) + t.c * 4u;
    }
    const int wEnd = w0 + DIR * a.c.kw;
    const uint32_t tapStep = GRAD ? 0u - 2u * C * 4u : 0u;   // besides the 64 bytes of a step
    const uint32_t rowStep = (uint32_t)(DIR * (a.c.W - a.c.kw)) * C * 4u;
    const int wraps = TAPS == TAPS_NARROW ? (int)((15u + C) / C) : TAPS ? 1 : 0;   // taps a step can pass
    const bool pixelOk = (unsigned)h0 < (unsigned)a.c.H && (unsigned)w0 < (unsigned)a.c.W;   // (of a single tap)

    // Weights: the lane's offset inside the 16 k of a step; the step is in the descriptor.  Columns past the last channel
    // read something or other for results that are not stored.
    uint32_t wOff[GRAD ? FN : 4];
    if constexpr (GRAD) {
#pragma unroll
        for (int f = 0; f < FN; ++f) wOff[f] = n0 + f * 16 + l16 < K ? ((n0 + f * 16 + l16) * a.kTot + quad * 4u) * 4u : W_OOB;
    } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) wOff[j] = ((quad * 4u + j) * K + n0 + l16) * 4u;
    }

    struct Operands {
        acc_t px;
        float wv[FN][4];
        uint32_t c[PRE ? LANE_K : 1];   // input channel of the lane's k (its first, where four share a tap)
    };

    // Loads of a step: out-of-range k, channels, rows and pixels get an offset outside the descriptor and read as 0; steps
    // past the wave's last get empty descriptors.  All by selects: written with && the compiler branches around each load
    // and waits inside the branch.
    auto load = [&](uint32_t step, Operands& o) {
        const bool run = step < sEnd;   // (wave-uniform)
        const uint32_t first = step * 16u * (GRAD ? 1u : K) * 4u;
        const rsrc_t rw = make_rsrc(reinterpret_cast<const char*>(a.c.w) + (run ? first : 0u), run ? a.wBytes - first : 0u);
#pragma unroll
        for (int j = 0; j < LANE_K; ++j) {
            Place& t = at[j];
            uint32_t bad = (uint32_t)(t.k >= a.kTot) | (uint32_t)!run;
            if constexpr (GRAD) {
#pragma unroll
                for (int f = 0; f < FN; ++f) {
                    const f4 v = buf_load<4>(rw, wOff[f] | (0u - (uint32_t)(t.k >= a.kTot)));
#pragma unroll
                    for (int i = 0; i < 4; ++i) o.wv[f][i] = v[i];
                }
            }
            if constexpr (PRE) o.c[j] = TAPS ? (t.k >= a.kTot ? cPad - 4u : t.c) : min(t.c, cPad - 4u);
            if constexpr (TAPS) bad |= (uint32_t)((unsigned)t.h >= (unsigned)a.c.H) | (uint32_t)((unsigned)t.w >= (unsigned)a.c.W);
            else bad |= (uint32_t)!pixelOk;
            const uint32_t off = t.off | (0u - bad);
            if constexpr (VEC == 4) o.px = buf_load<4>(ra, off);
            else o.px[j] = buf_load<1>(ra, off);
            t.k += 16u;
            t.c += 16u;
            t.off += 64u;
            for (int i = 0; i < wraps; ++i) {
                const bool next = t.c >= C;
                t.c -= next ? C : 0u;
                t.w += next ? DIR : 0;
                if constexpr (GRAD) t.off += next ? tapStep : 0u;
                const bool turn = t.w == wEnd;
                t.w = turn ? w0 : t.w;
                t.h += turn ? DIR : 0;
                t.off += turn ? rowStep : 0u;
            }
        }
        if constexpr (!GRAD) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int f = 0; f < FN; ++f) o.wv[f][j] = buf_load<1>(rw, wOff[j] + f * 64u);
        }
    };

    acc_t acc[FN];
#pragma unroll
    for (int i = 0; i < FN; ++i) acc[i] = (acc_t)(0.f);

    Operands ops[CONV_DEPTH];
#pragma unroll
    for (int d = 0; d < CONV_DEPTH; ++d) {
        load(sBeg + d, ops[d]);
        // (in this order: shuffled, the waits of the loop would be for the set that was loaded last)
        __builtin_amdgcn_sched_barrier(0);
    }

    if (PRE) {
        for (uint32_t c = tid; c < C; c += 64 * WAVES) bn_read(a.c.pre, c, preMean[c], preScale[c], preBeta[c]);
        if (tid < cPad - C) preMean[C + tid] = preScale[C + tid] = preBeta[C + tid] = 0.f;
    }
    if constexpr (GRAD) {
        for (uint32_t i = tid; i < (uint32_t)TN; i += 64 * WAVES) {
            const uint32_t n = min(n0 + i, K - 1);
            postMean[i] = a.c.norm.mean[n];
            postScale[i] = a.c.norm.inv[n];
        }
    } else if (post) {
        for (uint32_t i = tid; i < (uint32_t)TN; i += 64 * WAVES)
            if (n0 + i < K) bn_read(a.c.post, n0 + i, postMean[i], postScale[i], postBeta[i]);
    }
    if (PRE || GRAD || post) lds_barrier();

    auto multiply = [&](Operands& o) {
        if constexpr (PRE) {
            acc_t mean, sc, beta;
            if constexpr (VEC == 4) {
                mean = lds_read4(preMean + o.c[0]);
                sc = lds_read4(preScale + o.c[0]);
                beta = lds_read4(preBeta + o.c[0]);
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    mean[j] = preMean[o.c[j]];
                    sc[j] = preScale[o.c[j]];
                    beta[j] = preBeta[o.c[j]];
                }
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) o.px[j] = relu_keep_nan((o.px[j] - mean[j]) * sc[j] + beta[j]);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int i = 0; i < FN; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(o.wv[i][j], o.px[j], acc[i], 0, 0, 0);
    };
    // Whole rounds without a way out, then what is left.  With an exit inside a round the compiler waits for all loads at
    // the head of the loop, or moves a round's loads to its end: either way nothing stays in flight.
    uint32_t step = sBeg;
    for (; step + CONV_DEPTH <= sEnd; step += CONV_DEPTH) {
#pragma unroll
        for (int d = 0; d < CONV_DEPTH; ++d) {
            multiply(ops[d]);
            load(step + d + CONV_DEPTH, ops[d]);   // past the wave's last step: all out of range, no traffic
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int d = 0; d < CONV_DEPTH - 1; ++d)
        if (step + d < sEnd) multiply(ops[d]);   // (wave-uniform)

    const rsrc_t ry = make_rsrc(a.c.y, a.yBytes);
    // Four channels from n on of the lane's pixel.
    auto emit = [&](uint32_t n, uint32_t channels, acc_t v) {
        const uint32_t off = (outPix * channels + n) * 4u;
        if constexpr (VEC == 4) {
            const uint32_t o = outOk && n < channels ? off : BUF_OOB;   // channels are a multiple of 4 here
            if (!NEXT && a.c.add) v += buf_load<4>(ry, o);
            buf_store<0>(ry, o, (f4)v);
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t o = outOk && n + j < channels ? off + 4u * j : BUF_OOB;
                float t = v[j];
                if (a.c.add) t += buf_load<1>(ry, o);
                buf_store<0>(ry, o, t);
            }
        }
    };
    auto finish = [&](int i, acc_t v) {
        const uint32_t nl = i * 16 + quad * 4, n = n0 + nl;
        if constexpr (GRAD) {
            const uint32_t row = tp * TP + wp * 16 + l16;
            const uint32_t o = row < rows && n < K ? (row * K + n) * 4u : BUF_OOB;
            const acc_t z = (acc_t)buf_load<4>(make_rsrc(a.c.norm.z, a.yBytes), o);
            const acc_t act = (acc_t)buf_load<4>(make_rsrc(a.c.norm.act, a.yBytes), o);   // (0 past the end: masked)
            const acc_t xhat = (z - (acc_t)lds_read4(postMean + nl)) * (acc_t)lds_read4(postScale + nl);
            acc_t s1, s2;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                s1[j] = act[j] <= 0.f ? 0.f : v[j];
                s2[j] = s1[j] * xhat[j];
            }
            buf_store<0>(ry, o, (f4)s1);
#pragma unroll
            for (int off = 1; off < 16; off <<= 1)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    s1[j] += __shfl_xor(s1[j], off);
                    s2[j] += __shfl_xor(s2[j], off);
                }
            if (l16 == 0)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    sums[(wp * TN + nl + j) * 2] = s1[j];
                    sums[(wp * TN + nl + j) * 2 + 1] = s2[j];
                }
            return;
        }
        if (post) {
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = relu_keep_nan((v[j] - postMean[nl + j]) * postScale[nl + j] + postBeta[nl + j]);
        }
        emit(n, K, v);
    };

    if constexpr (NEXT) {
        auto between = [&](int i, acc_t v) {   // (columns past the last channel hold something or other: cleared)
            const uint32_t nl = i * 16 + quad * 4;
            const acc_t mean = lds_read4(postMean + nl), sc = lds_read4(postScale + nl), beta = lds_read4(postBeta + nl);
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = nl < K ? (post ? relu_keep_nan((v[j] - mean[j]) * sc[j] + beta[j]) : v[j]) : 0.f;
            return v;
        };
#pragma unroll
        for (int i = 0; i < FN; ++i) acc[i] = between(i, acc[i]);
        const uint32_t K2 = (uint32_t)a.K2;
        const rsrc_t rw2 = make_rsrc(a.w2, a.w2Bytes);
        constexpr int FO = 4;
        for (uint32_t t0 = 0; t0 < K2; t0 += 16u * FO) {
            float wv[2][4][FO];
            auto fetch = [&](int i) {   // (rows past the last channel read as zeros)
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int f = 0; f < FO; ++f)
                        wv[i & 1][j][f] = buf_load<1>(rw2, ((i * 16u + quad * 4u + j) * K2 + t0 + l16) * 4u + f * 64u);
            };
            acc_t out[FO], y[FO];   // (y: what the result is added to, loaded ahead of the products)
#pragma unroll
            for (int f = 0; f < FO; ++f) {
                const uint32_t n = t0 + f * 16u + quad * 4u;
                out[f] = (acc_t)(0.f);
                y[f] = buf_load<4>(ry, a.c.add && outOk && n < K2 ? (outPix * K2 + n) * 4u : BUF_OOB);
            }
            fetch(0);
#pragma unroll
            for (int i = 0; i < FN; ++i) {
                if (i + 1 < FN) fetch(i + 1);
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int f = 0; f < FO; ++f)
                        out[f] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[i & 1][j][f], acc[i][j], out[f], 0, 0, 0);
            }
#pragma unroll
            for (int f = 0; f < FO; ++f) emit(t0 + f * 16u + quad * 4u, K2, out[f] + y[f]);
        }
    } else if constexpr (WK == 1) {
#pragma unroll
        for (int i = 0; i < FN; ++i) finish(i, acc[i]);
    } else {
#pragma unroll
        for (int i = 0; i < FN; ++i) *reinterpret_cast<acc_t*>(red + (((wp * WK + wk) * FN + i) * 64 + lane) * 4) = acc[i];
        lds_barrier();
#pragma unroll
        for (int i = 0; i < FN; ++i) {
            if (i % WK != (int)wk) continue;   // (wave-uniform)
            acc_t v = (acc_t)(0.f);
#pragma unroll
            for (int k = 0; k < WK; ++k) v += (acc_t)lds_read4(red + (((wp * WK + k) * FN + i) * 64 + lane) * 4);
            finish(i, v);
        }
    }

    if constexpr (GRAD) {
        lds_barrier();
        // one atomic per channel, sum and workgroup; consecutive threads to consecutive doubles
        for (uint32_t i = tid; i < 2u * TN; i += 64 * WAVES) {
            double s = 0.0;
#pragma unroll
            for (int k = 0; k < WP; ++k) s += sums[k * TN * 2 + i];
            if (n0 + (i >> 1) < K)
                unsafeAtomicAdd(a.c.norm.sums + ((size_t)(blockIdx.x & (GRAD_SLOTS - 1)) * K + n0) * 2 + i, s);
        }
    }
}

template <int FN, int WK, int VEC, bool PRE, int TAPS, bool GRAD = false, bool NEXT = false>
static hipError_t launch_conv_as(ConvKernelArgs& a, hipStream_t stream)
{
    constexpr int WAVES = 4, TP = 16 * (WAVES / WK), TN = 16 * FN;
    a.tilesP = (a.rows + TP - 1) / TP;
    a.tilesN = ((uint32_t)a.c.K + TN - 1) / TN;
    const uint64_t grid = (uint64_t)((a.tilesP + 7) / 8 * 8) * a.tilesN;
    const size_t lds = sizeof(float) * ((a.c.pre.gamma ? 3 * (size_t)pre_channels(a.c.C) : 0) + (GRAD ? 2 + 4 * (WAVES / WK) : 3) * TN + (WK > 1 ? (size_t)WAVES * FN * 256 : 0));
    if (grid >= (1ull << 31) || lds > 64 * 1024) return hipErrorInvalidConfiguration;
    hipLaunchKernelGGL((k_block_conv<FN, WK, VEC, PRE, TAPS, GRAD, NEXT>), dim3((unsigned)grid), dim3(64 * WAVES), lds, stream, a);
    return hipGetLastError();
}

template <int FN, int WK, int VEC, bool PRE, bool GRAD>
static hipError_t launch_conv_taps(ConvKernelArgs& a, hipStream_t stream)
{
    if (a.c.kh * a.c.kw == 1) return launch_conv_as<FN, WK, VEC, PRE, TAPS_ONE, GRAD>(a, stream);
    if (a.c.C >= 16) return launch_conv_as<FN, WK, VEC, PRE, TAPS_WIDE, GRAD>(a, stream);
    return launch_conv_as<FN, WK, VEC, PRE, TAPS_NARROW, GRAD>(a, stream);
}

template <int FN, int WK, int VEC>
static hipError_t launch_conv_one(ConvKernelArgs& a, hipStream_t stream)
{
    return a.c.pre.gamma ? launch_conv_taps<FN, WK, VEC, true, false>(a, stream) : launch_conv_taps<FN, WK, VEC, false, false>(a, stream);
}

bool conv_fits(const ConvArgs& c)
{
    // 32-bit byte offsets in the input, the weights and the output; the batch norm of the input's channels in LDS
    const uint64_t most = 1ull << 30;
    const uint64_t a = (uint64_t)c.N * c.H * c.W * c.C, w = (uint64_t)c.kh * c.kw * c.C * c.K;
    const uint64_t rows = (uint64_t)c.M * c.Ro * c.So;
    const uint64_t y = (c.oidx ? (uint64_t)c.oN * c.oH * c.oW : rows) * c.K;
    return a < most && w < (1ull << 28) && y < most && rows < (1ull << 28) && c.C <= 4096 && c.Ro > 0 && c.So > 0;
}

static bool make_conv_args(const ConvArgs& c, ConvKernelArgs& a)
{
    a.c = c;
    a.dC = make_fastdiv((uint32_t)c.C);
    a.dKw = make_fastdiv((uint32_t)c.kw);
    a.P = (uint32_t)(c.Ro * c.So);
    a.dP = make_fastdiv(a.P);
    a.dSo = make_fastdiv((uint32_t)c.So);
    a.kTot = (uint32_t)(c.kh * c.kw * c.C);
    a.kSteps = (a.kTot + 15) / 16;
    a.rows = (uint32_t)c.M * a.P;
    a.aBytes = (uint32_t)((uint64_t)c.N * c.H * c.W * c.C * 4);
    a.wBytes = a.kTot * (uint32_t)c.K * 4u;
    a.yBytes = (uint32_t)((c.oidx ? (uint64_t)c.oN * c.oH * c.oW : (uint64_t)a.rows) * c.K * 4);
    const uintptr_t bits = reinterpret_cast<uintptr_t>(c.a) | reinterpret_cast<uintptr_t>(c.y);
    return c.C % 4 == 0 && c.K % 4 == 0 && (bits & 15) == 0;   // 16-byte accesses on both sides
}

// fn: fragments of 16 channels per wave; wk: waves that split k.
static void conv_tile(const ConvKernelArgs& a, bool vec, int& fn, int& wk)
{
    // Narrow wave tiles (16 pixels x 32 channels; 48 where that leaves no channel over, 16 where there are no more) and as
    // many waves per tile as it takes to occupy the SIMDs: a launch of fewer than about 1500 waves is four times shorter
    // with k split four ways than its occupancy would suggest, and one with few steps per wave has nothing to split.
    // Tiles of 64 channels are no faster (us for 32 / 64: 2350 pixels, k 1152, 128 channels 13.5 / 14.9; 3850, 512, 128:
    // 12.4 / 11.7; 2350, 128, 512: 8.7 / 9.0), of 16 slower (17.6; 16.4; 10.1), for all that splits.
    const uint32_t nFrag = ((uint32_t)a.c.K + 15) / 16;
    fn = nFrag == 1 ? 1 : (vec && nFrag % 3 == 0 && nFrag % 2 == 1 ? 3 : 2);
    const uint64_t waves = (uint64_t)((a.rows + 15) / 16) * ((nFrag + fn - 1) / fn);
    wk = a.kSteps < 8 ? 1 : (waves < 1536 ? 4 : (waves < 3072 && a.kSteps >= 16 ? 2 : 1));
}

hipError_t launch_block_conv(const ConvArgs& c, hipStream_t stream)
{
    if (c.M <= 0) return hipSuccess;
    if (!conv_fits(c)) return hipErrorInvalidValue;
    ConvKernelArgs a;
    const bool vec = make_conv_args(c, a);
    int fn, wk;
    conv_tile(a, vec, fn, wk);
    if (!vec) {
        if (fn == 1) return wk > 1 ? launch_conv_one<1, 4, 1>(a, stream) : launch_conv_one<1, 1, 1>(a, stream);
        return wk > 1 ? launch_conv_one<2, 4, 1>(a, stream) : launch_conv_one<2, 1, 1>(a, stream);
    }
    switch (fn * 8 + wk) {
    case 8 + 1: return launch_conv_one<1, 1, 4>(a, stream);
    case 8 + 2: return launch_conv_one<1, 2, 4>(a, stream);
    case 8 + 4: return launch_conv_one<1, 4, 4>(a, stream);
    case 16 + 1: return launch_conv_one<2, 1, 4>(a, stream);
    case 16 + 2: return launch_conv_one<2, 2, 4>(a, stream);
    case 16 + 4: return launch_conv_one<2, 4, 4>(a, stream);
    case 24 + 1: return launch_conv_one<3, 1, 4>(a, stream);
    case 24 + 2: return launch_conv_one<3, 2, 4>(a, stream);
    default: return launch_conv_one<3, 4, 4>(a, stream);
    }
}

hipError_t launch_block_conv_next(const ConvArgs& c, const ConvArgs& next, hipStream_t stream, bool& done)
{
    done = false;
    if (c.M <= 0 || c.pre.gamma || next.pre.gamma || next.post.gamma || next.kh != 1 || next.kw != 1 || c.kh * c.kw == 1 ||
        c.C < 16 || c.K > 128 || next.C != c.K || next.K % 4 != 0 || !conv_fits(c) || !conv_fits(next))
        return hipSuccess;
    ConvArgs both = c;   // input and kernel of the first, output of the second
    both.y = next.y;
    both.oidx = next.oidx;
    both.oN = next.oN; both.oH = next.oH; both.oW = next.oW; both.oU = next.oU; both.oV = next.oV;
    both.add = next.add;
    ConvKernelArgs a;
    if (!make_conv_args(both, a)) return hipSuccess;
    a.yBytes = (uint32_t)((next.oidx ? (uint64_t)next.oN * next.oH * next.oW : (uint64_t)a.rows) * next.K * 4);
    a.w2 = next.w;
    a.K2 = next.K;
    a.w2Bytes = (uint32_t)(next.C * next.K * 4);
    // A wave per 16 pixels and all channels: with fewer of them than SIMDs to fill, two launches that split further are
    // faster.  us a block, in one launch / in two, by the channels in between and at 993, 2025, 6807 waves: 24: 19.7 / 21.1,
    // 26.2 / 27.6, 50.7 / 55.4; 48: 31.5 / 31.4, 41.0 / 45.1, 103 / 116; 64: 44.1 / 44.5, 62.4 / 74.2, 170 / 215; 128: 128 / 125,
    // 191 / 230, 623 / 813; and at 307: 15.1 / 14.3, 23.3 / 19.0, 33.0 / 24.6, 104 / 50.  (16 channels gain at any size.)
    if ((a.rows + 15) / 16 < 1536) return hipSuccess;
    done = true;
    switch ((c.K + 15) / 16) {
    case 1: return launch_conv_as<1, 1, 4, false, TAPS_WIDE, false, true>(a, stream);
    case 2: return launch_conv_as<2, 1, 4, false, TAPS_WIDE, false, true>(a, stream);
    case 3: return launch_conv_as<3, 1, 4, false, TAPS_WIDE, false, true>(a, stream);
    case 4: return launch_conv_as<4, 1, 4, false, TAPS_WIDE, false, true>(a, stream);
    case 5:
    case 6: return launch_conv_as<6, 1, 4, false, TAPS_WIDE, false, true>(a, stream);
    default: return launch_conv_as<8, 1, 4, false, TAPS_WIDE, false, true>(a, stream);
    }
}

bool conv_grad_fits(const ConvArgs& c)
{
    const uintptr_t bits = reinterpret_cast<uintptr_t>(c.a) | reinterpret_cast<uintptr_t>(c.y) | reinterpret_cast<uintptr_t>(c.w) |
                           reinterpret_cast<uintptr_t>(c.norm.z) | reinterpret_cast<uintptr_t>(c.norm.act);
    return conv_fits(c) && c.M > 0 && c.C % 4 == 0 && c.K % 4 == 0 && (bits & 15) == 0 && !c.idx && !c.oidx && !c.countDev &&
           c.Ro == c.H + c.kh - 1 && c.So == c.W + c.kw - 1;
}

hipError_t launch_block_conv_grad(const ConvArgs& c, hipStream_t stream)
{
    if (!conv_grad_fits(c)) return hipErrorInvalidValue;
    ConvKernelArgs a;
    if (!make_conv_args(c, a)) return hipErrorInvalidValue;
    int fn, wk;
    conv_tile(a, true, fn, wk);
    switch (fn * 8 + wk) {
    case 8 + 1: return launch_conv_taps<1, 1, 4, false, true>(a, stream);
    case 8 + 2: return launch_conv_taps<1, 2, 4, false, true>(a, stream);
    case 8 + 4: return launch_conv_taps<1, 4, 4, false, true>(a, stream);
    case 16 + 1: return launch_conv_taps<2, 1, 4, false, true>(a, stream);
    case 16 + 2: return launch_conv_taps<2, 2, 4, false, true>(a, stream);
    case 16 + 4: return launch_conv_taps<2, 4, 4, false, true>(a, stream);
    case 24 + 1: return launch_conv_taps<3, 1, 4, false, true>(a, stream);
    case 24 + 2: return launch_conv_taps<3, 2, 4, false, true>(a, stream);
    default: return launch_conv_taps<3, 4, 4, false, true>(a, stream);
    }
}

}  // namespace sbnet
