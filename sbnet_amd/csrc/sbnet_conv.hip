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
// A wave computes 16*FP pixels x 16*FN channels with v_mfma_f32_16x16x4_f32 (full fp32 products and sums: the precision
// of the convolution it replaces).  Channels are the rows of the matrix instruction and pixels its columns, so that a
// lane ends with four consecutive channels of one pixel: 16-byte stores into NHWC memory.  Both operands go from memory
// straight to registers: with the instruction's k index spread as (lane / 16) * 4 + step, a lane's four pixel values
// are one 16-byte load, and 4 lanes read the 64 bytes of a pixel that 16 k need.  The fp32 matrix rate is low enough
// (a 2x2 wave tile multiplies for 512 cycles per 16 k, for which it reads 4 KB) that L1 feeds it, and without LDS
// tiles there are no barriers: the problems are small (a few thousand pixels) and their time is a chain of latencies.
// CONV_DEPTH sets of operands are in flight per wave.
//
// Measured (MI355X, kernel trace): 85 blocks of 17x17x48, 3x3 to 48 channels (19 000 pixels, 0.8 GFLOP; 5.2 us at the
// rate of a large fp32 product): 19 us, 27 us while the loads of a step sat behind branches; the library convolution
// took 21 us behind 5 us of layout copies, and up to 800 us the first time a block count occurred.  A bottleneck block of
// 200 17x17x96 blocks: 39 us in three launches against about 300 us in 17.
//
// WK > 1: the WK waves of a workgroup split k among them and add up through LDS.  For launches whose tiles alone would
// leave most of the 1024 SIMDs idle.
//
// Batch norm of the input (pre) applies to values after the load, out-of-image zeros included, with scale and shift
// computed once per workgroup into LDS; batch norm of the result (post), for the convolution that follows, at the end.

typedef float acc_t __attribute__((ext_vector_type(4)));

constexpr int CONV_DEPTH = 3;   // operand sets in flight per wave
constexpr uint32_t W_OOB = 0x40000000u;   // beyond any kernel (conv_fits), alone and added to itself

struct ConvKernelArgs {
    ConvArgs c;
    FastDiv dC, dKw, dP, dSo;
    uint32_t kTot, kSteps;      // taps * C, ceil(kTot / 16)
    uint32_t rows, P;           // output pixels in all, per block
    uint32_t tilesP, tilesN;
    uint32_t aBytes, wBytes, yBytes;
};

__device__ __forceinline__ float relu_keep_nan(float v) { return v < 0.f ? 0.f : v; }

// scale and shift of an inference batch norm, y = x * scale + shift
__device__ __forceinline__ void bn_fold(const BnArgs& bn, uint32_t c, float& scale, float& shift)
{
    scale = bn.gamma[c] * (1.f / sqrtf(bn.var[c] + bn.eps));
    shift = bn.beta[c] - bn.mean[c] * scale;
}

// GRAD: the gradient of a convolution's input.  The same product with the kernel turned around, w [K, kh, kw, C] (n, then
// k: a lane's four k are one 16-byte load of w, too); the epilogue masks the result where the ReLU did and adds up what
// the batch norm's gradient needs, in fp32 over 16 pixels and in double from there on.
template <int FP, int FN, int WK, int VEC, bool PRE, bool TAPS, bool GRAD>
__global__ __launch_bounds__(WK > 4 ? 64 * WK : 256) void k_block_conv(ConvKernelArgs a)
{
    constexpr int WAVES = WK > 4 ? WK : 4, WP = WAVES / WK;
    constexpr int TP = 16 * FP * WP, TN = 16 * FN;
    extern __shared__ float lds[];
    const uint32_t cPad = PRE ? ((uint32_t)a.c.C + 3u) & ~3u : 0u;
    float* const preScale = lds;
    float* const preShift = lds + cPad;
    float* const postScale = lds + 2 * cPad;
    float* const postShift = postScale + TN;
    double* const sums = reinterpret_cast<double*>(postScale + 2 * TN);   // [WP * FP][TN][2], GRAD only
    float* const red = postScale + (GRAD ? 2 + 4 * WP * FP : 2) * TN;     // [WP][WK][FP * FN][64] x 4, WK > 1 only

    // Eight consecutive workgroups go to eight XCDs; the tiles of one pixel range that differ in channels only follow
    // each other on one XCD, whose L2 then holds the pixels once.
    const uint32_t g = blockIdx.x >> 3;
    const uint32_t tn = g % a.tilesN, tp = (g / a.tilesN) * 8u + (blockIdx.x & 7u);
    uint32_t rows = a.rows;
    if (a.c.countDev) rows = min(rows, (uint32_t)max(*a.c.countDev, 0) * a.P);
    if (tp * TP >= rows) return;   // (the whole workgroup)

    const uint32_t tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, quad = lane >> 4;
    const uint32_t wave = tid >> 6, wk = wave % WK, wp = wave / WK;
    const uint32_t n0 = tn * TN;
    const bool post = a.c.post.gamma != nullptr;

    // The wave's pixels: one per lane and fragment, the same for the four quads.
    int h[FP], w[FP];
    uint32_t base[FP];   // byte offset of channel 0 of the pixel under tap (0, 0)
#pragma unroll
    for (int f = 0; f < FP; ++f) {
        const uint32_t row = tp * TP + (wp * FP + f) * 16 + l16;
        bool ok = row < rows;
        const uint32_t ib = fdiv(ok ? row : 0u, a.dP), p = (ok ? row : 0u) - ib * a.P;
        const uint32_t r = fdiv(p, a.dSo), s = p - r * (uint32_t)a.c.So;
        int n = (int)ib;
        h[f] = (int)r;
        w[f] = (int)s;
        if (a.c.idx) {
            const int16_t* t = a.c.idx + (size_t)ib * 3;
            n = t[0];
            h[f] += a.c.oh + t[1] * a.c.U;
            w[f] += a.c.ow + t[2] * a.c.V;
            ok = ok && (unsigned)n < (unsigned)a.c.N;
        }
        base[f] = (((uint32_t)n * (uint32_t)a.c.H + (uint32_t)h[f]) * (uint32_t)a.c.W + (uint32_t)w[f]) * (uint32_t)a.c.C * 4u;
        if (!ok) h[f] = -0x40000000;   // outside the image under every tap
    }

    const rsrc_t ra = make_rsrc(a.c.a, a.aBytes), rw = make_rsrc(a.c.w, a.wBytes);
    const uint32_t per = (a.kSteps + WK - 1) / WK;
    const uint32_t sBeg = wk * per, sEnd = min(sBeg + per, a.kSteps);
    const uint32_t kEnd = min(sEnd * 16u, a.kTot);
    const uint32_t K = (uint32_t)a.c.K;
    uint32_t wCol[FN];
#pragma unroll
    for (int f = 0; f < FN; ++f) {
        const uint32_t n = n0 + f * 16 + l16;
        wCol[f] = n < K ? n * (GRAD ? a.kTot : 1u) * 4u : W_OOB;
    }

    struct Operands {
        acc_t px[FP];
        float wv[FN][4];
        uint32_t c[VEC == 4 ? 1 : 4];   // input channel of the lane's k (its first, where four share a tap)
    };

    // Loads of a step: out-of-range k, channels, rows and pixels get an offset outside the descriptor and read as 0.
    // All by selects: written with && the compiler branches around each load and waits inside the branch.
    auto load = [&](uint32_t step, Operands& o) {
        const uint32_t k = step * 16u + quad * 4u;
#pragma unroll
        for (int j = 0; j < (VEC == 4 ? 1 : 4); ++j) {
            const uint32_t kj = k + j;
            uint32_t c = kj;
            int dr = 0, ds = 0;
            if constexpr (TAPS) {
                const uint32_t tap = fdiv(kj, a.dC);
                c = kj - tap * (uint32_t)a.c.C;
                dr = (int)fdiv(tap, a.dKw);
                ds = (int)tap - dr * a.c.kw;
            } else {
                c = min(c, (uint32_t)a.c.C - (VEC == 4 ? 4u : 1u));   // (a channel to look scale and shift up for, past the end)
            }
            o.c[j] = c;
            if constexpr (GRAD) {
                const uint32_t row = kj < kEnd ? kj * 4u : W_OOB;
#pragma unroll
                for (int f = 0; f < FN; ++f) {
                    const f4 t = buf_load<4>(rw, row + wCol[f]);
#pragma unroll
                    for (int i = 0; i < 4; ++i) o.wv[f][i] = t[i];
                }
                dr = -dr;   // (the output pixel that this tap took the input pixel to)
                ds = -ds;
            }
            const uint32_t toff = (((uint32_t)dr * (uint32_t)a.c.W + (uint32_t)ds) * (uint32_t)a.c.C + c) * 4u;
#pragma unroll
            for (int f = 0; f < FP; ++f) {
                const uint32_t bad = (uint32_t)((unsigned)(h[f] + dr) >= (unsigned)a.c.H) |
                                     (uint32_t)((unsigned)(w[f] + ds) >= (unsigned)a.c.W) | (uint32_t)(kj >= kEnd);
                const uint32_t off = (base[f] + toff) | (0u - bad);
                if constexpr (VEC == 4) o.px[f] = buf_load<4>(ra, off);
                else o.px[f][j] = buf_load<1>(ra, off);
            }
        }
        if constexpr (!GRAD) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t row = (k + j < kEnd) ? (k + j) * K * 4u : W_OOB;
#pragma unroll
                for (int f = 0; f < FN; ++f) o.wv[f][j] = buf_load<1>(rw, row + wCol[f]);
            }
        }
    };

    acc_t acc[FN][FP];
#pragma unroll
    for (int i = 0; i < FN; ++i)
#pragma unroll
        for (int f = 0; f < FP; ++f) acc[i][f] = (acc_t)(0.f);

    Operands ops[CONV_DEPTH];
#pragma unroll
    for (int d = 0; d < CONV_DEPTH; ++d) load(sBeg + d, ops[d]);

    if (PRE)
        for (uint32_t c = tid; c < (uint32_t)a.c.C; c += 64 * WAVES) bn_fold(a.c.pre, c, preScale[c], preShift[c]);
    if constexpr (GRAD) {   // mean and 1 / sigma
        for (uint32_t i = tid; i < (uint32_t)TN; i += 64 * WAVES) {
            const uint32_t n = min(n0 + i, K - 1);
            postScale[i] = a.c.norm.mean[n];
            postShift[i] = a.c.norm.inv[n];
        }
    } else if (post) {
        for (uint32_t i = tid; i < (uint32_t)TN; i += 64 * WAVES)
            if (n0 + i < K) bn_fold(a.c.post, n0 + i, postScale[i], postShift[i]);
    }
    if (PRE || GRAD || post) lds_barrier();

    for (uint32_t step = sBeg; step < sEnd; step += CONV_DEPTH) {
#pragma unroll
        for (int d = 0; d < CONV_DEPTH; ++d) {
            if (d && step + d >= sEnd) break;   // (wave-uniform; a round of multiplying zeros would cost as much as a full one)
            Operands& o = ops[d];
            if constexpr (PRE) {
                acc_t sc, sh;
                if constexpr (VEC == 4) {
                    sc = lds_read4(preScale + o.c[0]);
                    sh = lds_read4(preShift + o.c[0]);
                } else {
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        sc[j] = preScale[o.c[j]];
                        sh[j] = preShift[o.c[j]];
                    }
                }
#pragma unroll
                for (int f = 0; f < FP; ++f)
#pragma unroll
                    for (int j = 0; j < 4; ++j) o.px[f][j] = relu_keep_nan(o.px[f][j] * sc[j] + sh[j]);
            }
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int i = 0; i < FN; ++i)
#pragma unroll
                    for (int f = 0; f < FP; ++f)
                        acc[i][f] = __builtin_amdgcn_mfma_f32_16x16x4f32(o.wv[i][j], o.px[f][j], acc[i][f], 0, 0, 0);
            load(step + d + CONV_DEPTH, o);   // past the wave's last step: all out of range, no traffic
        }
    }

    const rsrc_t ry = make_rsrc(a.c.y, a.yBytes);
    auto finish = [&](int i, int f, acc_t v) {
        const uint32_t nl = i * 16 + quad * 4, n = n0 + nl;
        if constexpr (GRAD) {
            const uint32_t group = wp * FP + f, row = tp * TP + group * 16 + l16;
            const uint32_t o = row < rows && n < K ? (row * K + n) * 4u : BUF_OOB;
            const acc_t z = (acc_t)buf_load<4>(make_rsrc(a.c.norm.z, a.yBytes), o);
            const acc_t act = (acc_t)buf_load<4>(make_rsrc(a.c.norm.act, a.yBytes), o);   // (0 past the end: masked)
            const acc_t xhat = (z - (acc_t)lds_read4(postScale + nl)) * (acc_t)lds_read4(postShift + nl);
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
                    sums[(group * TN + nl + j) * 2] = s1[j];
                    sums[(group * TN + nl + j) * 2 + 1] = s2[j];
                }
            return;
        }
        if (post) {
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = relu_keep_nan(v[j] * postScale[nl + j] + postShift[nl + j]);
        }
        const uint32_t row = tp * TP + (wp * FP + f) * 16 + l16;
        bool ok = row < rows;
        uint32_t pix = row;
        if (a.c.oidx) {
            const uint32_t ib = fdiv(ok ? row : 0u, a.dP), p = (ok ? row : 0u) - ib * a.P;
            const uint32_t r = fdiv(p, a.dSo), s = p - r * (uint32_t)a.c.So;
            const int16_t* t = a.c.oidx + (size_t)ib * 3;
            const int on = t[0], oh = t[1] * a.c.oU + (int)r, ow = t[2] * a.c.oV + (int)s;
            ok = ok && (unsigned)on < (unsigned)a.c.oN && (unsigned)oh < (unsigned)a.c.oH && (unsigned)ow < (unsigned)a.c.oW;
            pix = ((uint32_t)on * (uint32_t)a.c.oH + (uint32_t)oh) * (uint32_t)a.c.oW + (uint32_t)ow;
        }
        const uint32_t off = (pix * K + n) * 4u;
        if constexpr (VEC == 4) {
            const uint32_t o = ok && n < K ? off : BUF_OOB;   // K is a multiple of 4 here
            if (a.c.add) v += buf_load<4>(ry, o);
            buf_store<0>(ry, o, (f4)v);
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t o = ok && n + j < K ? off + 4u * j : BUF_OOB;
                float t = v[j];
                if (a.c.add) t += buf_load<1>(ry, o);
                buf_store<0>(ry, o, t);
            }
        }
    };

    if constexpr (WK == 1) {
#pragma unroll
        for (int i = 0; i < FN; ++i)
#pragma unroll
            for (int f = 0; f < FP; ++f) finish(i, f, acc[i][f]);
    } else {
#pragma unroll
        for (int i = 0; i < FN; ++i)
#pragma unroll
            for (int f = 0; f < FP; ++f)
                *reinterpret_cast<acc_t*>(red + (((wp * WK + wk) * (FP * FN) + i * FP + f) * 64 + lane) * 4) = acc[i][f];
        lds_barrier();
#pragma unroll
        for (int q = 0; q < FP * FN; ++q) {
            if (q % WK != (int)wk) continue;   // (wave-uniform)
            acc_t v = (acc_t)(0.f);
#pragma unroll
            for (int k = 0; k < WK; ++k)
                v += (acc_t)lds_read4(red + (((wp * WK + k) * (FP * FN) + q) * 64 + lane) * 4);
            finish(q / FP, q % FP, v);
        }
    }

    if constexpr (GRAD) {
        lds_barrier();
        // one atomic per channel, sum and workgroup; consecutive threads to consecutive doubles
        for (uint32_t i = tid; i < 2u * TN; i += 64 * WAVES) {
            double s = 0.0;
#pragma unroll
            for (int k = 0; k < WP * FP; ++k) s += sums[k * TN * 2 + i];
            if (n0 + (i >> 1) < K)
                unsafeAtomicAdd(a.c.norm.sums + ((size_t)(blockIdx.x & (GRAD_SLOTS - 1)) * K + n0) * 2 + i, s);
        }
    }
}

template <int FP, int FN, int WK, int VEC, bool PRE, bool TAPS, bool GRAD = false>
static hipError_t launch_conv_as(ConvKernelArgs& a, hipStream_t stream)
{
    constexpr int WAVES = WK > 4 ? WK : 4, TP = 16 * FP * (WAVES / WK), TN = 16 * FN;
    a.tilesP = (a.rows + TP - 1) / TP;
    a.tilesN = ((uint32_t)a.c.K + TN - 1) / TN;
    const uint64_t grid = (uint64_t)((a.tilesP + 7) / 8 * 8) * a.tilesN;
    const size_t lds = sizeof(float) * ((a.c.pre.gamma ? 2 * (((size_t)a.c.C + 3) & ~(size_t)3) : 0) + (GRAD ? 2 + 4 * FP * (WAVES / WK) : 2) * TN + (WK > 1 ? (size_t)WAVES * FP * FN * 256 : 0));
    if (grid >= (1ull << 31) || lds > 64 * 1024) return hipErrorInvalidConfiguration;
    hipLaunchKernelGGL((k_block_conv<FP, FN, WK, VEC, PRE, TAPS, GRAD>), dim3((unsigned)grid), dim3(64 * WAVES), lds, stream, a);
    return hipGetLastError();
}

template <int FP, int FN, int WK, int VEC>
static hipError_t launch_conv_one(ConvKernelArgs& a, hipStream_t stream)
{
    const bool taps = a.c.kh * a.c.kw > 1;
    if (a.c.pre.gamma) return taps ? launch_conv_as<FP, FN, WK, VEC, true, true>(a, stream) : launch_conv_as<FP, FN, WK, VEC, true, false>(a, stream);
    return taps ? launch_conv_as<FP, FN, WK, VEC, false, true>(a, stream) : launch_conv_as<FP, FN, WK, VEC, false, false>(a, stream);
}

bool conv_fits(const ConvArgs& c)
{
    // 32-bit byte offsets in the input, the weights and the output; scale and shift of the input's channels in LDS
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
    // Wider tiles read less and wait more: 32x32 is 10-40 % slower on all but the narrowest and largest problems (us for
    // 16x32 / 32x32, best split: 2450 pixels, k 1152, 128 channels 16.4 / 19.0; 4860, 576, 64: 10.3 / 12.0; 45 000, 216, 24:
    // 13.2 / 12.6; 38 400, 600, 24: 24.7 / 22.7).
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
        if (fn == 1) return wk > 1 ? launch_conv_one<1, 1, 4, 1>(a, stream) : launch_conv_one<1, 1, 1, 1>(a, stream);
        return wk > 1 ? launch_conv_one<1, 2, 4, 1>(a, stream) : launch_conv_one<1, 2, 1, 1>(a, stream);
    }
    switch (fn * 8 + wk) {
    case 8 + 1: return launch_conv_one<1, 1, 1, 4>(a, stream);
    case 8 + 2: return launch_conv_one<1, 1, 2, 4>(a, stream);
    case 8 + 4: return launch_conv_one<1, 1, 4, 4>(a, stream);
    case 16 + 1: return launch_conv_one<1, 2, 1, 4>(a, stream);
    case 16 + 2: return launch_conv_one<1, 2, 2, 4>(a, stream);
    case 16 + 4: return launch_conv_one<1, 2, 4, 4>(a, stream);
    case 24 + 1: return launch_conv_one<1, 3, 1, 4>(a, stream);
    case 24 + 2: return launch_conv_one<1, 3, 2, 4>(a, stream);
    default: return launch_conv_one<1, 3, 4, 4>(a, stream);
    }
}

template <int FN, int WK>
static hipError_t launch_conv_grad_one(ConvKernelArgs& a, hipStream_t stream)
{
    if (a.c.kh * a.c.kw > 1) return launch_conv_as<1, FN, WK, 4, false, true, true>(a, stream);
    return launch_conv_as<1, FN, WK, 4, false, false, true>(a, stream);
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
    case 8 + 1: return launch_conv_grad_one<1, 1>(a, stream);
    case 8 + 2: return launch_conv_grad_one<1, 2>(a, stream);
    case 8 + 4: return launch_conv_grad_one<1, 4>(a, stream);
    case 16 + 1: return launch_conv_grad_one<2, 1>(a, stream);
    case 16 + 2: return launch_conv_grad_one<2, 2>(a, stream);
    case 16 + 4: return launch_conv_grad_one<2, 4>(a, stream);
    case 24 + 1: return launch_conv_grad_one<3, 1>(a, stream);
    case 24 + 2: return launch_conv_grad_one<3, 2>(a, stream);
    default: return launch_conv_grad_one<3, 4>(a, stream);
    }
}

}  // namespace sbnet
