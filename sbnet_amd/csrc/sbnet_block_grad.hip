// The gradient of a bottleneck's residual function beside its convolutions (sbnet_conv.hip): the backward of the batch
// norms, the gradients of the kernels, and block stacks from planar to NHWC and back.
//
// Replaces the library's backward passes behind the reference's layer functions (sbnet_tensorflow/benchmark/
// sparse_conv_lib.py:590-723 under tf.gradients).
#include "sbnet_conv.h"
#include "sbnet_device.h"

namespace sbnet {

typedef float acc_t __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------------------------------------
// k_norm_grad: dz = gamma / sigma * (g - mean(g) - xhat * mean(g * xhat)), xhat = (z - mean) / sigma
// ---------------------------------------------------------------------------------------------
//
// Four channels per thread, `cols` threads side by side, `tall` rows at a time; a workgroup takes as many rows as leave
// about 512 workgroups.  Two tensors in, one out, once each.  The channels' coefficients are worked out once per
// workgroup, a channel a thread (four of them in every thread, 32 loads ahead of the first row, took 22.9 us for the three
// launches of a step on 85 blocks of 11x11, 256-64-64 channels; 15.2 this way).

struct ChannelArgs {
    uint32_t rows, C;
    uint32_t cols, tall, rowsPerWg;
};

static ChannelArgs channel_args(uint32_t rows, int C, dim3& grid)
{
    ChannelArgs a;
    a.rows = rows;
    a.C = (uint32_t)C;
    a.cols = min((uint32_t)C / 4u, 64u);
    a.tall = 256u / a.cols;
    const uint32_t chunks = (a.C / 4u + a.cols - 1) / a.cols;
    const uint32_t steps = ((uint64_t)rows * chunks + a.tall * 512ull - 1) / (a.tall * 512ull);
    a.rowsPerWg = a.tall * max(steps, 4u);
    grid = dim3((rows + a.rowsPerWg - 1) / a.rowsPerWg, chunks);
    return a;
}

__global__ __launch_bounds__(256) void k_norm_grad(float* __restrict__ g, NormGradArgs norm, ChannelArgs a,
                                                   float* __restrict__ dgamma, float* __restrict__ dbeta)
{
    __shared__ __attribute__((aligned(16))) float coef[4][256];   // mean, scale and the two means, of the workgroup's channels
    const uint32_t tid = threadIdx.x, ty = tid / a.cols, tx = tid - ty * a.cols;
    const uint32_t first = blockIdx.y * a.cols * 4u, mine = first + tid;
    if (tid < a.cols * 4u && mine < a.C) {
        double s1 = 0.0, s2 = 0.0;
#pragma unroll
        for (int i = 0; i < GRAD_SLOTS; ++i) {
            const double2 t = *reinterpret_cast<const double2*>(norm.sums + ((size_t)i * a.C + mine) * 2);
            s1 += t.x;
            s2 += t.y;
        }
        const float inv = norm.inv[mine];
        coef[0][tid] = norm.mean[mine];
        coef[1][tid] = inv * norm.gamma[mine];
        coef[2][tid] = (float)(s1 / a.rows);
        coef[3][tid] = (float)(s2 / a.rows * inv);
        if (blockIdx.x == 0) {
            if (dgamma) dgamma[mine] = (float)s2;
            if (dbeta) dbeta[mine] = (float)s1;
        }
    }
    lds_barrier();
    const uint32_t c = first + tx * 4u;
    if (ty >= a.tall || c >= a.C) return;
    const f4 mean = lds_read4(coef[0] + tx * 4u), scale = lds_read4(coef[1] + tx * 4u), c1 = lds_read4(coef[2] + tx * 4u),
             c2 = lds_read4(coef[3] + tx * 4u);
    const float* const z = norm.z;
    const uint32_t end = min((blockIdx.x + 1) * a.rowsPerWg, a.rows);
#pragma unroll 4
    for (uint32_t r = blockIdx.x * a.rowsPerWg + ty; r < end; r += a.tall) {
        const size_t at = (size_t)r * a.C + c;
        const f4 x = *reinterpret_cast<const f4*>(z + at);
        f4 v = *reinterpret_cast<const f4*>(g + at);
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = scale[j] * (v[j] - c1[j] - (x[j] - mean[j]) * c2[j]);
        *reinterpret_cast<f4*>(g + at) = v;
    }
}

hipError_t launch_norm_grad(float* g, const NormGradArgs& norm, uint32_t rows, int C, float* dgamma, float* dbeta,
                            hipStream_t stream)
{
    dim3 grid;
    const ChannelArgs a = channel_args(rows, C, grid);
    hipLaunchKernelGGL(k_norm_grad, grid, dim3(256), 0, stream, g, norm, a, dgamma, dbeta);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------
// k_transposes: [M][A][B] -> [M][B][A], several tensors in one launch
// ---------------------------------------------------------------------------------------------
//
// 64 x 32 tiles through LDS (a row more than a multiple of the banks apart), one dword per lane and access: 128 bytes in a
// row on both sides, whatever B is (a block's pixel count, mostly odd).

constexpr uint32_t TR_A = 64, TR_B = 32;

struct TransposeProblem {
    TransposeArgs t;
    uint32_t tilesB, tiles, firstWg;
};

// Besides, `zeros` are cleared, 256 a workgroup behind those of the transposes: the sums that the launches behind add to.
struct TransposeKernelArgs {
    TransposeProblem p[10];
    int count;
    float* zeros;
    uint32_t zeroCount, firstZeroWg;
};

__global__ __launch_bounds__(256) void k_transposes(TransposeKernelArgs k)
{
    __shared__ float tile[TR_A * (TR_B + 1)];
    if (blockIdx.x >= k.firstZeroWg) {
        const uint32_t z = (blockIdx.x - k.firstZeroWg) * 256u + threadIdx.x;
        if (z < k.zeroCount) k.zeros[z] = 0.f;
        return;
    }
    int i = 0;
    while (i + 1 < k.count && blockIdx.x >= k.p[i + 1].firstWg) ++i;
    const TransposeProblem& q = k.p[i];
    const uint32_t A = q.t.A, B = q.t.B;
    const uint32_t local = blockIdx.x - q.firstWg, m = local / q.tiles, rest = local - m * q.tiles;
    const uint32_t ta = rest / q.tilesB, a0 = ta * TR_A, b0 = (rest - ta * q.tilesB) * TR_B;
    const float* __restrict__ from = q.t.from + (size_t)m * A * B;
    float* __restrict__ to = q.t.to + (size_t)m * A * B;
    const uint32_t tid = threadIdx.x;
    float v[TR_A * TR_B / 256];
#pragma unroll
    for (uint32_t j = 0; j < TR_A * TR_B / 256; ++j) {
        const uint32_t r = a0 + (tid >> 5) + 8 * j, c = b0 + (tid & 31);
        v[j] = r < A && c < B ? from[(size_t)r * B + c] : 0.f;
    }
#pragma unroll
    for (uint32_t j = 0; j < TR_A * TR_B / 256; ++j) tile[((tid >> 5) + 8 * j) * (TR_B + 1) + (tid & 31)] = v[j];
    lds_barrier();
#pragma unroll
    for (uint32_t j = 0; j < TR_A * TR_B / 256; ++j) {
        const uint32_t r = (tid >> 6) + 4 * j, c = tid & 63;
        if (b0 + r < B && a0 + c < A) to[(size_t)(b0 + r) * A + a0 + c] = tile[c * (TR_B + 1) + r];
    }
}

hipError_t launch_transposes(const TransposeArgs* t, int count, hipStream_t stream, float* zeros, uint32_t zeroCount)
{
    if (count < 1 || count > 10) return hipErrorInvalidValue;
    TransposeKernelArgs k;
    uint64_t wgs = 0;
    for (int i = 0; i < count; ++i) {
        TransposeProblem& q = k.p[i];
        q.t = t[i];
        q.tilesB = (t[i].B + TR_B - 1) / TR_B;
        q.tiles = (t[i].A + TR_A - 1) / TR_A * q.tilesB;
        q.firstWg = (uint32_t)wgs;
        wgs += (uint64_t)t[i].M * q.tiles;
    }
    k.zeros = zeros;
    k.zeroCount = zeroCount;
    k.firstZeroWg = (uint32_t)wgs;
    wgs += (zeroCount + 255u) / 256u;
    if (wgs >= (1ull << 31)) return hipErrorInvalidConfiguration;
    k.count = count;
    hipLaunchKernelGGL(k_transposes, dim3((unsigned)wgs), dim3(256), 0, stream, k);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------
// k_relu: a ReLU in place, NaN kept and zeros positive, as the library's has them
// ---------------------------------------------------------------------------------------------
//
// The library's takes 7 us of host time a call, this one 3.

__device__ __forceinline__ float relu_of_library(float v) { return v != v ? v : fmaxf(v, 0.f); }

constexpr uint32_t RELU_UNR = 4;

__global__ __launch_bounds__(256) void k_relu(float* __restrict__ x, size_t n4, uint32_t rest)
{
    const size_t at = (size_t)blockIdx.x * (256u * RELU_UNR) + threadIdx.x;
    f4* const v4 = reinterpret_cast<f4*>(x);
    f4 v[RELU_UNR];
#pragma unroll
    for (uint32_t u = 0; u < RELU_UNR; ++u) {
        v[u] = (f4)(0.f);
        if (at + 256u * u < n4) v[u] = v4[at + 256u * u];
    }
#pragma unroll
    for (uint32_t u = 0; u < RELU_UNR; ++u) {
#pragma unroll
        for (int j = 0; j < 4; ++j) v[u][j] = relu_of_library(v[u][j]);
        if (at + 256u * u < n4) v4[at + 256u * u] = v[u];
    }
    if (blockIdx.x == 0 && threadIdx.x < rest) x[n4 * 4 + threadIdx.x] = relu_of_library(x[n4 * 4 + threadIdx.x]);
}

hipError_t launch_relu(float* x, size_t count, hipStream_t stream)
{
    const size_t n4 = count / 4, wgs = (n4 + 256u * RELU_UNR - 1) / (256u * RELU_UNR);
    if (count == 0) return hipSuccess;
    if (wgs >= (1ull << 31)) return hipErrorInvalidConfiguration;
    hipLaunchKernelGGL(k_relu, dim3(wgs ? (unsigned)wgs : 1u), dim3(256), 0, stream, x, n4, (uint32_t)(count - n4 * 4));
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------
// k_kernels: [taps][C][K] -> [K][C][taps], the three kernels of a residual function in one launch
// ---------------------------------------------------------------------------------------------
//
// In the order of the results; what is read lies K floats apart, in the caches: the kernels are small.  (Three copies of
// permuted views through the library: 11 us on the GPU and 24 in the host for 256-64-64-256 channels; 4 and 5 this way.)

struct KernelsProblem {
    const float* from;
    float* to;
    uint32_t count, K, C, taps, firstWg;
    FastDiv dRow, dTaps;   // by C * taps, by taps
};

struct KernelsArgs {
    KernelsProblem p[3];
    int count;
};

constexpr uint32_t KERNELS_UNR = 4;

__global__ __launch_bounds__(256) void k_kernels(KernelsArgs a)
{
    int i = 0;
    while (i + 1 < a.count && blockIdx.x >= a.p[i + 1].firstWg) ++i;
    const KernelsProblem& q = a.p[i];
    const uint32_t o0 = (blockIdx.x - q.firstWg) * (256u * KERNELS_UNR) + threadIdx.x;
    float v[KERNELS_UNR];
#pragma unroll
    for (uint32_t u = 0; u < KERNELS_UNR; ++u) {
        const uint32_t o = min(o0 + 256u * u, q.count - 1u);
        const uint32_t k = fdiv(o, q.dRow), r = o - k * (q.C * q.taps), c = fdiv(r, q.dTaps), t = r - c * q.taps;
        v[u] = q.from[(size_t)(t * q.C + c) * q.K + k];
    }
#pragma unroll
    for (uint32_t u = 0; u < KERNELS_UNR; ++u)
        if (o0 + 256u * u < q.count) q.to[o0 + 256u * u] = v[u];
}

hipError_t launch_kernels(const float* const* from, const int32_t* dims, float* const* to, int count, hipStream_t stream)
{
    if (count < 1 || count > 3) return hipErrorInvalidValue;
    KernelsArgs a;
    uint64_t wgs = 0;
    for (int i = 0; i < count; ++i) {
        const int32_t* d = dims + 4 * i;
        const uint64_t n = (uint64_t)d[0] * d[1] * d[2] * d[3];
        if (n == 0 || n >= (1ull << 30)) return hipErrorInvalidValue;
        KernelsProblem& q = a.p[i];
        q.from = from[i];
        q.to = to[i];
        q.count = (uint32_t)n;
        q.taps = (uint32_t)(d[0] * d[1]);
        q.C = (uint32_t)d[2];
        q.K = (uint32_t)d[3];
        q.firstWg = (uint32_t)wgs;
        q.dRow = make_fastdiv(q.C * q.taps);
        q.dTaps = make_fastdiv(q.taps);
        wgs += (n + 256u * KERNELS_UNR - 1) / (256u * KERNELS_UNR);
    }
    a.count = count;
    hipLaunchKernelGGL(k_kernels, dim3((unsigned)wgs), dim3(256), 0, stream, a);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------
// k_wgrad: dw[m, n] = sum over output pixels p of act[p + tap, c] * dz[p, n], m = (tap, c)
// ---------------------------------------------------------------------------------------------
//
// The sum runs over thousands of pixels and the result is small, so the pixels are what is split: a workgroup takes one
// 64 x 64 (or 64 x 32) tile of one kernel's gradient over one range of pixels, its four waves every fourth quadruple of
// pixels, and writes a partial tile that k_wgrad_sum adds to the others.  All three kernels of a bottleneck share the
// launch: alone, each would leave part of the chip idle.
//
// v_mfma_f32_16x16x4_f32 with the four quads of a wave on four pixels: a lane's 16-byte load of four consecutive channels
// of its pixel feeds four fragments (fragment i has rows 4 * l + i), so 4 pixels x 64 x 64 products cost two 16-byte loads
// and 16 matrix instructions per lane, straight from memory.
//
// Measured (MI355X, kernel trace; 256-64-64-256 channels on about 85 active 11x11 blocks of [1,100,175,256]): 18.5 us for the
// three products and 5.2 for the sum of the partial tiles, where the library took 77 us and six transposes of its operands
// (23 us).  The whole gradient: 105 us in 12 launches; 190 us in 27 with the library's passes.

struct WgradProblem {
    WgradArgs w;
    FastDiv dP, dSo, dC, dKw;
    uint32_t rows, P, So, mTot;
    uint32_t tilesM, tiles, rowsPerSplit, splits;
    uint32_t aBytes, dzBytes;
    uint32_t firstWg;      // of the launch
    uint32_t firstSum;     // 16-byte pieces of the results before this one
    int jb;                // output channels per lane: 4 or 2
    float* part;           // [splits][tiles][4 * jb][64] x 4
};

struct WgradKernelArgs {
    WgradProblem p[3];
    int count;
    uint32_t sums;
};

constexpr int WG_DEPTH = 4;   // pixel quadruples in flight per wave

template <int JB, bool TAPS>
__device__ __forceinline__ void wgrad_tile(const WgradProblem& q, uint32_t local, float* lds)
{
    const uint32_t tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, quad = lane >> 4, wave = tid >> 6;
    const uint32_t split = local / q.tiles, tile = local - split * q.tiles;
    const uint32_t tn = tile / q.tilesM, tm = tile - tn * q.tilesM;
    const uint32_t C = (uint32_t)q.w.C, K = (uint32_t)q.w.K;

    const uint32_t m = tm * 64u + l16 * 4u;
    const bool mOk = m < q.mTot;
    const uint32_t tap = TAPS ? fdiv(mOk ? m : 0u, q.dC) : 0u, c = (mOk ? m : 0u) - tap * C;
    const uint32_t dr = TAPS ? fdiv(tap, q.dKw) : 0u, ds = tap - dr * (uint32_t)q.w.kw;
    const uint32_t aOff = mOk ? (TAPS ? (dr * (uint32_t)q.w.S + ds) * C + c : c) * 4u : 0u;
    const uint32_t n = tn * (16u * JB) + l16 * JB;
    const bool nOk = n < K;
    const rsrc_t ra = make_rsrc(q.w.act, q.aBytes), rd = make_rsrc(q.w.dz, q.dzBytes);

    const uint32_t beg = split * q.rowsPerSplit, end = min(beg + q.rowsPerSplit, q.rows);
    struct Operands {
        acc_t v;
        float d[JB];
    };
    // Rows past the range read zeros on both sides.
    auto load = [&](uint32_t row, Operands& o) {
        const bool ok = row < end;
        uint32_t pix = row;
        if constexpr (TAPS) {
            const uint32_t ib = fdiv(ok ? row : 0u, q.dP), p = (ok ? row : 0u) - ib * q.P;
            const uint32_t r = fdiv(p, q.dSo), s = p - r * q.So;
            pix = (ib * (uint32_t)q.w.R + r) * (uint32_t)q.w.S + s;
        }
        o.v = (acc_t)buf_load<4>(ra, ok && mOk ? pix * C * 4u + aOff : BUF_OOB);
        const uint32_t od = ok && nOk ? (row * K + n) * 4u : BUF_OOB;
        if constexpr (JB == 4) {
            const f4 t = buf_load<4>(rd, od);
#pragma unroll
            for (int j = 0; j < 4; ++j) o.d[j] = t[j];
        } else {
            const f2 t = buf_load<2>(rd, od);
            o.d[0] = t[0];
            o.d[1] = t[1];
        }
    };

    acc_t acc[4][JB];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < JB; ++j) acc[i][j] = (acc_t)(0.f);
    Operands ops[WG_DEPTH];
    uint32_t row = beg + wave * 4u + quad;
#pragma unroll
    for (int d = 0; d < WG_DEPTH; ++d) load(row + d * 16u, ops[d]);
    for (uint32_t first = beg + wave * 4u; first < end; first += WG_DEPTH * 16u) {
#pragma unroll
        for (int d = 0; d < WG_DEPTH; ++d) {
            Operands& o = ops[d];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < JB; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(o.v[i], o.d[j], acc[i][j], 0, 0, 0);
            load(row + (WG_DEPTH + d) * 16u, o);
        }
        row += WG_DEPTH * 16u;
    }

#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < JB; ++j)
            *reinterpret_cast<acc_t*>(lds + ((wave * (4 * JB) + i * JB + j) * 64 + lane) * 4) = acc[i][j];
    lds_barrier();
    float* const out = q.part + (size_t)local * (4 * JB * 256);
#pragma unroll
    for (int f = 0; f < JB; ++f) {
        const uint32_t frag = f * 4 + wave;
        acc_t v = (acc_t)(0.f);
#pragma unroll
        for (int k = 0; k < 4; ++k) v += (acc_t)lds_read4(lds + ((k * (4 * JB) + frag) * 64 + lane) * 4);
        *reinterpret_cast<acc_t*>(out + (frag * 64 + lane) * 4) = v;
    }
}

__global__ __launch_bounds__(256) void k_wgrad(WgradKernelArgs a)
{
    extern __shared__ float lds[];
    int i = 0;
    while (i + 1 < a.count && blockIdx.x >= a.p[i + 1].firstWg) ++i;
    const WgradProblem& q = a.p[i];
    const uint32_t local = blockIdx.x - q.firstWg;
    const bool taps = q.w.kh * q.w.kw > 1;
    if (q.jb == 4) {
        if (taps) wgrad_tile<4, true>(q, local, lds);
        else wgrad_tile<4, false>(q, local, lds);
    } else {
        if (taps) wgrad_tile<2, true>(q, local, lds);
        else wgrad_tile<2, false>(q, local, lds);
    }
}

// Adds the partial tiles, in double, and writes the gradients.  The results are few and the splits many: a workgroup takes
// 64 pieces of 16 bytes, its waves every eighth split of them.  (A thread for all splits of a piece: 17.6 us for 642 partial
// tiles of 16 KB, from 68 workgroups that wait for one round of loads after the other; 5.2 this way.)
constexpr int SUM_WAVES = 8;

__global__ __launch_bounds__(64 * SUM_WAVES) void k_wgrad_sum(WgradKernelArgs a)
{
    __shared__ double part[SUM_WAVES][4][64];
    const uint32_t wave = threadIdx.x >> 6;
    const uint32_t id = blockIdx.x * 64u + (threadIdx.x & 63u);   // (a.sums is a multiple of 64)
    int k = 0;
    while (k + 1 < a.count && id >= a.p[k + 1].firstSum) ++k;
    const WgradProblem& q = a.p[k];
    const uint32_t local = id - q.firstSum, frags = 4u * (uint32_t)q.jb;
    const uint32_t lane = local & 63, l16 = lane & 15, quad = lane >> 4;
    const uint32_t tile = (local >> 6) / frags, frag = (local >> 6) - tile * frags;
    const uint32_t tn = tile / q.tilesM, tm = tile - tn * q.tilesM;
    const float* p = q.part + (size_t)local * 4;
    const size_t step = (size_t)q.tiles * frags * 256;
    double s[4] = {};
#pragma unroll 8
    for (uint32_t i = wave; i < q.splits; i += SUM_WAVES) {
        const f4 v = *reinterpret_cast<const f4*>(p + i * step);
#pragma unroll
        for (int j = 0; j < 4; ++j) s[j] += (double)v[j];
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) part[wave][r][lane] = s[r];
    lds_barrier();
    if (wave >= 4u) return;   // (wave r has the r-th float of each piece)
    double sum = 0.0;
#pragma unroll
    for (int w = 0; w < SUM_WAVES; ++w) sum += part[w][wave][lane];
    const uint32_t i = frag / (uint32_t)q.jb, j = frag - i * (uint32_t)q.jb;
    const uint32_t n = (tn * 16u + l16) * (uint32_t)q.jb + j, m = tm * 64u + (quad * 4u + wave) * 4u + i;
    if (n < (uint32_t)q.w.K && m < q.mTot) q.w.dw[(size_t)m * q.w.K + n] = (float)sum;
}

// About 640 workgroups in all, each of at least 64 pixels, the pixels' ranges of all problems equally long.
static void wgrad_plan(const WgradArgs* w, int count, WgradKernelArgs& a)
{
    uint64_t cost = 0;
    for (int i = 0; i < count; ++i) {
        WgradProblem& q = a.p[i];
        q.w = w[i];
        q.P = (uint32_t)((w[i].R - w[i].kh + 1) * (w[i].S - w[i].kw + 1));
        q.So = (uint32_t)(w[i].S - w[i].kw + 1);
        q.rows = (uint32_t)w[i].M * q.P;
        q.mTot = (uint32_t)(w[i].kh * w[i].kw * w[i].C);
        q.jb = w[i].K > 32 ? 4 : 2;
        q.tilesM = (q.mTot + 63) / 64;
        q.tiles = q.tilesM * (((uint32_t)w[i].K + 16 * q.jb - 1) / (16 * q.jb));
        cost += (uint64_t)q.rows * q.tiles;
    }
    uint64_t per = (cost + 639) / 640;
    per = per < 64 ? 64 : (per + 15) / 16 * 16;
    uint32_t wg = 0, sum = 0;
    for (int i = 0; i < count; ++i) {
        WgradProblem& q = a.p[i];
        q.rowsPerSplit = (uint32_t)per;
        q.splits = (uint32_t)((q.rows + per - 1) / per);
        q.firstWg = wg;
        q.firstSum = sum;
        wg += q.splits * q.tiles;
        sum += q.tiles * 4 * q.jb * 64;
    }
    a.count = count;
    a.sums = sum;
}

size_t wgrad_workspace_bytes(const WgradArgs* w, int count)
{
    WgradKernelArgs a;
    wgrad_plan(w, count, a);
    size_t total = 0;
    for (int i = 0; i < count; ++i) total += (size_t)a.p[i].splits * a.p[i].tiles * (4 * a.p[i].jb * 256) * sizeof(float);
    return total;
}

hipError_t launch_wgrad(const WgradArgs* w, int count, void* workspace, hipStream_t stream)
{
    if (count < 1 || count > 3) return hipErrorInvalidValue;
    WgradKernelArgs a;
    wgrad_plan(w, count, a);
    float* part = static_cast<float*>(workspace);
    for (int i = 0; i < count; ++i) {
        WgradProblem& q = a.p[i];
        q.dP = make_fastdiv(q.P);
        q.dSo = make_fastdiv(q.So);
        q.dC = make_fastdiv((uint32_t)w[i].C);
        q.dKw = make_fastdiv((uint32_t)w[i].kw);
        q.aBytes = (uint32_t)((uint64_t)w[i].M * w[i].R * w[i].S * w[i].C * 4);
        q.dzBytes = (uint32_t)((uint64_t)q.rows * w[i].K * 4);
        q.part = part;
        part += (size_t)q.splits * q.tiles * (4 * q.jb * 256);
    }
    const WgradProblem& last = a.p[count - 1];
    const uint32_t wgs = last.firstWg + last.splits * last.tiles;
    hipLaunchKernelGGL(k_wgrad, dim3(wgs), dim3(256), 65536, stream, a);
    hipLaunchKernelGGL(k_wgrad_sum, dim3(a.sums / 64), dim3(64 * SUM_WAVES), 0, stream, a);
    return hipGetLastError();
}

}  // namespace sbnet
