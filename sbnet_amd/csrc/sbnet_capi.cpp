// C ABI of libsbnet_amd.so (declared in include/sbnet_amd.h): argument validation that mirrors
// the reference ops' OP_REQUIRES checks, then the kernel launches of sbnet_reduce_mask.hip, sbnet_gather.hip and sbnet_scatter.hip.
//
// Reference behaviour reproduced here (sbnet_tensorflow/sbnet_ops/):
//   reduce_mask.cc:132-138, 141-220   parameter shape check, host-visible count, zero-count fix-up
//   sparse_gather.cc:164-175, 190-207 rank / parameter checks, count taken from the host
//   sparse_gather.cc:307-346          parameter checks, add/atomic/overlap rule, rank check,
//                                     in place (Var) versus copy-then-scatter
#include "../../include/sbnet_amd.h"

#include <hip/hip_runtime_api.h>
#include <sched.h>

#include <algorithm>
#include <mutex>
#include <vector>

#include "sbnet_conv.h"
#include "sbnet_launch.h"

namespace {

thread_local int g_lastHipError = 0;
thread_local int t_forceGeneric = 0;  // test hook, see sbnet_test_force_generic

int hip_fail(hipError_t e)
{
    g_lastHipError = (int)e;
    return SBNET_EHIP;
}

#define SBNET_HIP(call)                                  \
    do {                                                 \
        hipError_t e_ = (call);                          \
        if (e_ != hipSuccess) return hip_fail(e_);       \
    } while (0)

bool pair_ok(const int32_t* p, int len) { return p != nullptr && len == 2; }

// The host-visible count of reduce_mask (reduce_mask.cc:198-204: a HostMemory output filled by a blocking
// cudaMemcpy).  Instead of a device-to-host copy and a stream synchronisation (about 17 us of a 113 us
// pipeline step), the kernel that knows the count stores it, tagged with a sequence number, into one word
// of pinned host memory and the calling thread polls that word.  One word per thread and device, allocated
// on first use and kept until the process ends.
constexpr int MAX_SIGNAL_DEVICES = 64;
struct HostSignal {
    unsigned long long* host = nullptr;  // pinned, device-visible (same address on both sides)
    uint32_t seq = 0;
    bool failed = false;                 // allocation refused once: do not try again
};

// Words are handed out per thread and device; a thread that ends returns its words to a free list, so the
// number of words is bounded by the largest number of threads alive at once, and sbnet_shutdown() frees
// them.  Nothing is freed from a static destructor: the HIP runtime may already be gone by then.
std::mutex g_signalMutex;
std::vector<unsigned long long*> g_signalFree[MAX_SIGNAL_DEVICES];
std::vector<unsigned long long*> g_signalAll;

struct ThreadSignals {
    HostSignal dev[MAX_SIGNAL_DEVICES];
    ~ThreadSignals()
    {
        std::lock_guard<std::mutex> lock(g_signalMutex);
        for (int d = 0; d < MAX_SIGNAL_DEVICES; ++d)
            if (dev[d].host) g_signalFree[d].push_back(dev[d].host);
    }
};
thread_local ThreadSignals t_signal;

HostSignal* host_signal()
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_SIGNAL_DEVICES) return nullptr;
    HostSignal& s = t_signal.dev[dev];
    if (!s.host && !s.failed) {
        std::lock_guard<std::mutex> lock(g_signalMutex);
        if (!g_signalFree[dev].empty()) {
            s.host = g_signalFree[dev].back();
            g_signalFree[dev].pop_back();
            // the word keeps the last tag its previous owner saw: continue from there, never reuse a tag
            s.seq = (uint32_t)(__atomic_load_n(s.host, __ATOMIC_ACQUIRE) >> 32);
        } else {
            void* p = nullptr;
            if (hipHostMalloc(&p, 64, hipHostMallocMapped | hipHostMallocPortable) != hipSuccess || !p) {
                (void)hipGetLastError();
                s.failed = true;
            } else {
                s.host = static_cast<unsigned long long*>(p);
                *s.host = 0;
                g_signalAll.push_back(s.host);
            }
        }
    }
    return s.host ? &s : nullptr;
}

inline void cpu_relax()
{
#if defined(__x86_64__) || defined(__i386__)
    __builtin_ia32_pause();
#endif
}

// Reads of the word before the stream is asked.  The question is no mere look: the runtime answers it by enqueueing a
// barrier packet behind the kernels, which costs host time and holds up the launch that follows the count.  Asked every 256
// reads, one came into nearly every wait: a step of mask, gather and scatter on a [1,64,64,16] map took 38.9 us,
// 31.4 without it, on [3,301,203,15] 46.6 and 31.5.  After 2^14 reads, most of them behind a yield, some milliseconds have passed.
constexpr uint32_t SPINS_PER_QUERY = 1u << 14;

// Waits until the word carries `seq` and returns the count; gives up (false) as soon as the stream has
// drained without the word arriving or reports an error, so the wait always ends with the stream.
bool poll_host_signal(const HostSignal& s, uint32_t seq, hipStream_t stream, int32_t* count, hipError_t* err)
{
    *err = hipSuccess;
    // Back-off: the count normally arrives within a few microseconds, so the first reads only pause the core;
    // behind a long queue the thread yields between reads instead of burning its core.
    for (uint32_t spins = 1;; ++spins) {
        const unsigned long long v = __atomic_load_n(s.host, __ATOMIC_ACQUIRE);
        if ((uint32_t)(v >> 32) == seq) {
            *count = (int32_t)(uint32_t)v;
            return true;
        }
        if (spins < 4096u) cpu_relax();
        else sched_yield();
        if ((spins & (SPINS_PER_QUERY - 1u)) == 0) {
            const hipError_t q = hipStreamQuery(stream);
            if (q == hipErrorNotReady) {
                (void)hipGetLastError();
                continue;
            }
            if (q != hipSuccess) {
                *err = q;
                return false;
            }
            // the stream is idle: the store has been issued; look once more, then leave it to a copy
            const unsigned long long w = __atomic_load_n(s.host, __ATOMIC_ACQUIRE);
            if ((uint32_t)(w >> 32) == seq) {
                *count = (int32_t)(uint32_t)w;
                return true;
            }
            return false;
        }
    }
}

// Limits the reference leaves unchecked.  Indices are int16 triples, so n, bh and bw must fit.
bool geom_ok(int N, int H, int W, int C, const int32_t* bsize, const int32_t* bstride)
{
    return N > 0 && H > 0 && W > 0 && C > 0 && bsize[0] > 0 && bsize[1] > 0 && bstride[0] > 0 &&
           bstride[1] > 0 && (int64_t)N * H * W * C < (1ll << 40);
}

sbnet::Geom make_geom(int N, int H, int W, int C, const int32_t* bsize, const int32_t* bstride,
                      const int32_t* boffset)
{
    sbnet::Geom g;
    g.N = N; g.H = H; g.W = W; g.C = C;
    g.R = bsize[0]; g.S = bsize[1];
    g.U = bstride[0]; g.V = bstride[1];
    g.oh = boffset[0]; g.ow = boffset[1];
    g.countDev = nullptr;
    g.forceGeneric = t_forceGeneric;
    return g;
}

bool dims_fit_int(const int64_t* d)
{
    for (int i = 0; i < 4; ++i)
        if (d[i] < 0 || d[i] > 0x7fffffffll) return false;
    return true;
}

int reduce_mask_impl(const float* mask, int N, int H, int W, const int32_t* bcount,
                     const int32_t* bsize, const int32_t* bstride, const int32_t* boffset, float tol,
                     int avgpool, bool fixup, int16_t* idx, int32_t* countHost, int32_t* countDev,
                     void* workspace, size_t workspaceBytes, hipStream_t stream)
{
    if (!mask || !idx || (!countHost && !countDev)) return SBNET_EINVAL_ARG;
    if (!geom_ok(N, H, W, 1, bsize, bstride)) return SBNET_EINVAL_ARG;
    if (bcount[0] <= 0 || bcount[1] <= 0) return SBNET_EINVAL_ARG;
    // (n, bh, bw) are stored as int16
    if (N > 32768 || bcount[0] > 32768 || bcount[1] > 32768) return SBNET_EINVAL_ARG;
    const int64_t T = (int64_t)N * bcount[0] * bcount[1];
    if (T >= (1ll << 31)) return SBNET_EINVAL_ARG;
    // block origins and ends must stay inside int arithmetic
    const int64_t hEnd = (int64_t)boffset[0] + (int64_t)bstride[0] * (bcount[0] - 1) + bsize[0];
    const int64_t wEnd = (int64_t)boffset[1] + (int64_t)bstride[1] * (bcount[1] - 1) + bsize[1];
    if (hEnd > 0x7fffffffll || wEnd > 0x7fffffffll || (int64_t)bsize[0] * bsize[1] > 0x7fffffffll)
        return SBNET_EINVAL_ARG;

    const size_t need = sbnet::reduce_mask_workspace_bytes(T);
    void* ws = workspace;
    bool ownWs = false;
    if (ws && (workspaceBytes < need || (reinterpret_cast<uintptr_t>(ws) & 15))) return SBNET_EINVAL_ARG;
    // Neither a host-visible count (nothing runs during capture) nor a scratch buffer of the library's own
    // (allocating and freeing it synchronises) can be had while the stream is being captured: refuse before
    // anything is allocated or enqueued, so the capture stays valid.
    bool capturing = false;
    if (countHost || !ws) {
        hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
        if (hipStreamIsCapturing(stream, &cap) != hipSuccess) (void)hipGetLastError();  // (cannot be asked: not capturing)
        else capturing = cap != hipStreamCaptureStatusNone;
        if (capturing) return hip_fail(hipErrorStreamCaptureUnsupported);
    }
    if (!ws) {
        SBNET_HIP(hipMalloc(&ws, need));
        ownWs = true;
    }
    const sbnet::Geom g = make_geom(N, H, W, 1, bsize, bstride, boffset);
    HostSignal* sig = nullptr;
    uint32_t seq = 0;
    if (countHost) {
        sig = host_signal();
        if (sig) {
            seq = ++sig->seq;
            if (seq == 0) seq = ++sig->seq;  // 0 is the word's initial tag
        }
    }
    hipError_t e = sbnet::launch_reduce_mask(mask, g, bcount[0], bcount[1], tol, avgpool != 0, fixup, idx,
                                             countDev, ws, stream, sig ? sig->host : nullptr, seq);
    bool haveCount = false;
    if (e == hipSuccess && sig) haveCount = poll_host_signal(*sig, seq, stream, countHost, &e);
    if (e == hipSuccess && countHost && !haveCount) {
        // the count sits in countDev, or in the workspace
        const int32_t* src = countDev ? countDev : sbnet::reduce_mask_count_slot(ws, T);
        e = hipMemcpyAsync(countHost, src, sizeof(int32_t), hipMemcpyDeviceToHost, stream);
        if (e == hipSuccess) e = hipStreamSynchronize(stream);
    }
    if (ownWs) {
        hipError_t e2 = hipStreamSynchronize(stream);
        hipError_t e3 = hipFree(ws);
        if (e == hipSuccess) e = e2 != hipSuccess ? e2 : e3;
    }
    if (e != hipSuccess) return hip_fail(e);
    return SBNET_OK;
}

int gather_impl(const float* x, int N, int H, int W, int C, float* y, const int32_t* bsize, const int32_t* bstride,
                const int32_t* boffset, int numActive, const int32_t* countDev, const int16_t* idx, int transpose,
                hipStream_t stream)
{
    if (numActive < 0) return SBNET_EINVAL_ARG;
    if (numActive > 0 && (!x || !y || !idx)) return SBNET_EINVAL_ARG;
    if (!geom_ok(N, H, W, C, bsize, bstride)) return SBNET_EINVAL_ARG;
    sbnet::Geom g = make_geom(N, H, W, C, bsize, bstride, boffset);
    g.countDev = countDev;
    SBNET_HIP(sbnet::launch_gather(x, y, idx, numActive, g, transpose != 0, stream));
    return SBNET_OK;
}

int scatter_impl(const float* x, int32_t numActive, const int32_t* countDev, const int16_t* idx, float* out,
                 const int64_t* dims, const int32_t* bsize, const int32_t* bstride,
                 const int32_t* boffset, int add, int atomic, int transpose, void* workspace,
                 size_t workspaceBytes, hipStream_t stream)
{
    if (numActive < 0) return SBNET_EINVAL_ARG;
    if (numActive > 0 && (!x || !idx)) return SBNET_EINVAL_ARG;
    if (!out || !dims_fit_int(dims)) return SBNET_EINVAL_ARG;
    if (!geom_ok((int)dims[0], (int)dims[1], (int)dims[2], (int)dims[3], bsize, bstride))
        return SBNET_EINVAL_ARG;
    sbnet::Geom g = make_geom((int)dims[0], (int)dims[1], (int)dims[2], (int)dims[3], bsize, bstride, boffset);
    g.countDev = countDev;
    const sbnet::ScatterMode mode =
        !add ? sbnet::SCATTER_ASSIGN : (atomic ? sbnet::SCATTER_ATOMIC : sbnet::SCATTER_ADD);
    if (mode == sbnet::SCATTER_ATOMIC && workspace) {
        // with scratch an "atomic" add needs no atomics: the owner-computes kernel where it applies (NHWC stack,
        // at most 2x2 blocks per pixel; exact sequential order), else passes of plain adds over non-overlapping
        // classes of blocks
        bool done = false;
        if (!transpose)
            SBNET_HIP(sbnet::launch_scatter_pull(x, out, idx, numActive, g, workspace, workspaceBytes, stream, done));
        if (done) return SBNET_OK;
        SBNET_HIP(sbnet::launch_scatter_colored(x, out, idx, numActive, g, transpose != 0, workspace, workspaceBytes,
                                                stream, done));
        if (done) return SBNET_OK;
    }
    if (mode == sbnet::SCATTER_ASSIGN) {
        // overlapping plain writes land in the CPU functor's order (the block listed last wins): decided inside the
        // planar kernel where that applies, else with scratch (nothing is done here without scratch then)
        bool done = false;
        SBNET_HIP(sbnet::launch_scatter_owned(x, out, idx, numActive, g, transpose != 0, workspace, workspaceBytes,
                                              stream, done));
        if (done) return SBNET_OK;
    }
    SBNET_HIP(sbnet::launch_scatter(x, out, idx, numActive, g, transpose != 0, mode, stream));
    return SBNET_OK;
}

// Library-managed scratch for callers without an allocator at hand (sbnet_scratch_acquire): one grow-only buffer
// per (device, stream).  Work on one stream runs in order, so consecutive calls on that stream may share it.
struct ScratchSlot {
    int dev;
    hipStream_t stream;
    void* ptr;
    size_t bytes;
};
std::mutex g_scratchMutex;
std::vector<ScratchSlot> g_scratch;
// Buffers that a slot has outgrown.  A caller may still hold such a pointer (it asked before another thread's
// larger request on the same stream) and work that uses it may still be queued, so nothing is freed before
// sbnet_shutdown.
std::vector<ScratchSlot> g_scratchRetired;

}  // namespace

extern "C" {

const char* sbnet_version(void) { return "sbnet_amd 0.1 (gfx950)"; }

int sbnet_last_hip_error(void) { return g_lastHipError; }

const char* sbnet_status_string(int status)
{
    switch (status) {
    case SBNET_OK: return "OK";
    case SBNET_EINVAL_PARAM_SHAPE:
        return "InvalidArgument: dynamic_b<count, size, stride, offset> should be one-dimensional with shape[0] == 2.";
    case SBNET_EINVAL_RANK: return "InvalidArgument: x / ybase must be rank 4";
    case SBNET_EINVAL_OVERLAP:
        return "InvalidArgument: Only non-overlapping blocks are supported with add=True, atomic=False";
    case SBNET_EINVAL_ARG: return "InvalidArgument: null pointer, size out of range or workspace too small";
    case SBNET_EHIP: return "HIP runtime error (see sbnet_last_hip_error)";
    case SBNET_ETOOBIG:
        return "InvalidArgument: more blocks than the library's own scratch holds (sbnet_reduce_mask_static_max_indices); "
               "use sbnet_reduce_mask with a workspace";
    default: return "unknown sbnet status";
    }
}

int64_t sbnet_reduce_mask_max_indices(int N, const int32_t* bcount, int bcount_len)
{
    if (!pair_ok(bcount, bcount_len) || N < 0 || bcount[0] < 0 || bcount[1] < 0) return -1;
    return (int64_t)N * bcount[0] * bcount[1];
}

size_t sbnet_reduce_mask_workspace_bytes(int N, const int32_t* bcount, int bcount_len)
{
    const int64_t T = sbnet_reduce_mask_max_indices(N, bcount, bcount_len);
    if (T < 0) return 0;
    return sbnet::reduce_mask_workspace_bytes(T);
}

int sbnet_reduce_mask(const float* mask, int N, int H, int W, const int32_t* bcount, int bcount_len,
                      const int32_t* bsize, int bsize_len, const int32_t* bstride, int bstride_len,
                      const int32_t* boffset, int boffset_len, float tol, int avgpool,
                      int16_t* active_block_indices, int32_t* bin_counts_host,
                      int32_t* bin_counts_device, void* workspace, size_t workspace_bytes, void* stream)
{
    if (!pair_ok(bcount, bcount_len) || !pair_ok(bsize, bsize_len) || !pair_ok(bstride, bstride_len) ||
        !pair_ok(boffset, boffset_len))
        return SBNET_EINVAL_PARAM_SHAPE;
    return reduce_mask_impl(mask, N, H, W, bcount, bsize, bstride, boffset, tol, avgpool, true,
                            active_block_indices, bin_counts_host, bin_counts_device, workspace,
                            workspace_bytes, static_cast<hipStream_t>(stream));
}

int sbnet_reduce_mask_static(const float* mask, int N, int H, int W, const int32_t* bcount, int bcount_len,
                             const int32_t* bsize, int bsize_len, const int32_t* bstride, int bstride_len,
                             const int32_t* boffset, int boffset_len, float tol, int avgpool,
                             int16_t* active_block_indices, int32_t* bin_counts_device, void* stream)
{
    if (!pair_ok(bcount, bcount_len) || !pair_ok(bsize, bsize_len) || !pair_ok(bstride, bstride_len) ||
        !pair_ok(boffset, boffset_len))
        return SBNET_EINVAL_PARAM_SHAPE;
    if (!bin_counts_device) return SBNET_EINVAL_ARG;
    // what sbnet_reduce_mask rejects as an argument error is one here too; SBNET_ETOOBIG is for valid sizes only
    if (N <= 0 || bcount[0] <= 0 || bcount[1] <= 0 || N > 32768 || bcount[0] > 32768 || bcount[1] > 32768)
        return SBNET_EINVAL_ARG;
    const int64_t T = (int64_t)N * bcount[0] * bcount[1];
    if (T >= (1ll << 31)) return SBNET_EINVAL_ARG;
    if (sbnet::reduce_mask_workspace_bytes(T) > sbnet::STATIC_SCRATCH_BYTES) return SBNET_ETOOBIG;
    void* ws = nullptr;
    SBNET_HIP(sbnet::static_scratch(&ws));
    return reduce_mask_impl(mask, N, H, W, bcount, bsize, bstride, boffset, tol, avgpool, true, active_block_indices,
                            nullptr, bin_counts_device, ws, sbnet::STATIC_SCRATCH_BYTES,
                            static_cast<hipStream_t>(stream));
}

int64_t sbnet_reduce_mask_static_max_indices(void)
{
    // the largest T with reduce_mask_workspace_bytes(T) <= STATIC_SCRATCH_BYTES
    int64_t lo = 0, hi = (int64_t)sbnet::STATIC_SCRATCH_BYTES;
    while (lo < hi) {
        const int64_t mid = (lo + hi + 1) / 2;
        if (sbnet::reduce_mask_workspace_bytes(mid) <= sbnet::STATIC_SCRATCH_BYTES) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

int sbnet_reduce_mask_functor(const float* mask, int N, int H, int W, float threshold, int bOffsH0,
                              int bOffsW0, int bSzH, int bSzW, int bStrH, int bStrW, int bCntH,
                              int bCntW, unsigned int numBins, unsigned int binSize,
                              int16_t* activeBlockIndices, int32_t* binCounts, int avgPool,
                              void* workspace, size_t workspace_bytes, void* stream)
{
    (void)binSize;
    if (numBins != 1 || !binCounts) return SBNET_EINVAL_ARG;  // reduce_mask.cc:69 asserts numBins == 1
    const int32_t bcount[2] = {bCntH, bCntW}, bsize[2] = {bSzH, bSzW}, bstride[2] = {bStrH, bStrW},
                  boffset[2] = {bOffsH0, bOffsW0};
    return reduce_mask_impl(mask, N, H, W, bcount, bsize, bstride, boffset, threshold, avgPool, false,
                            activeBlockIndices, nullptr, binCounts, workspace, workspace_bytes,
                            static_cast<hipStream_t>(stream));
}

int sbnet_sparse_gather(const float* x, const int64_t* x_dims, int x_rank, int32_t num_active,
                        const int16_t* active_block_indices, const int32_t* bsize, int bsize_len,
                        const int32_t* bstride, int bstride_len, const int32_t* boffset,
                        int boffset_len, int transpose, float* y, void* stream)
{
    if (x_rank != 4) return SBNET_EINVAL_RANK;  // sparse_gather.cc:164
    if (!pair_ok(bsize, bsize_len) || !pair_ok(bstride, bstride_len) || !pair_ok(boffset, boffset_len))
        return SBNET_EINVAL_PARAM_SHAPE;  // sparse_gather.cc:169-175
    if (!x_dims || !dims_fit_int(x_dims)) return SBNET_EINVAL_ARG;
    return sbnet_sparse_gather_functor(x, (int)x_dims[0], (int)x_dims[1], (int)x_dims[2], (int)x_dims[3], y,
                                       boffset[0], boffset[1], bsize[0], bsize[1], bstride[0], bstride[1],
                                       num_active, active_block_indices, transpose, stream);
}

int sbnet_sparse_gather_functor(const float* x, int N, int H, int W, int C, float* y, int bOffsH0,
                                int bOffsW0, int bSzH, int bSzW, int bStrH, int bStrW, int numActive,
                                const int16_t* activeBlockIndices, int transpose, void* stream)
{
    const int32_t bsize[2] = {bSzH, bSzW}, bstride[2] = {bStrH, bStrW}, boffset[2] = {bOffsH0, bOffsW0};
    return gather_impl(x, N, H, W, C, y, bsize, bstride, boffset, numActive, nullptr, activeBlockIndices, transpose,
                       static_cast<hipStream_t>(stream));
}

int sbnet_sparse_gather_device_count(const float* x, const int64_t* x_dims, int x_rank,
                                     const int32_t* bin_counts_device, int32_t max_active,
                                     const int16_t* active_block_indices, const int32_t* bsize, int bsize_len,
                                     const int32_t* bstride, int bstride_len, const int32_t* boffset,
                                     int boffset_len, int transpose, float* y, void* stream)
{
    if (x_rank != 4) return SBNET_EINVAL_RANK;
    if (!pair_ok(bsize, bsize_len) || !pair_ok(bstride, bstride_len) || !pair_ok(boffset, boffset_len))
        return SBNET_EINVAL_PARAM_SHAPE;
    if (!x_dims || !dims_fit_int(x_dims) || !bin_counts_device) return SBNET_EINVAL_ARG;
    return gather_impl(x, (int)x_dims[0], (int)x_dims[1], (int)x_dims[2], (int)x_dims[3], y, bsize, bstride, boffset,
                       max_active, bin_counts_device, active_block_indices, transpose,
                       static_cast<hipStream_t>(stream));
}

size_t sbnet_sparse_scatter_workspace_bytes(int32_t num_active, const int64_t* ybase_dims, int ybase_rank,
                                            const int32_t* bsize, int bsize_len, const int32_t* bstride,
                                            int bstride_len, const int32_t* boffset, int boffset_len)
{
    if (ybase_rank != 4 || !ybase_dims || !dims_fit_int(ybase_dims) || num_active <= 0) return 0;
    if (!pair_ok(bsize, bsize_len) || !pair_ok(bstride, bstride_len) || !pair_ok(boffset, boffset_len)) return 0;
    if (!geom_ok((int)ybase_dims[0], (int)ybase_dims[1], (int)ybase_dims[2], (int)ybase_dims[3], bsize, bstride))
        return 0;
    const sbnet::Geom g = make_geom((int)ybase_dims[0], (int)ybase_dims[1], (int)ybase_dims[2], (int)ybase_dims[3],
                                    bsize, bstride, boffset);
    const size_t pull = sbnet::scatter_pull_workspace_bytes(g, num_active);
    const size_t color = sbnet::scatter_color_workspace_bytes(g, num_active);
    const size_t cover = sbnet::scatter_cover_workspace_bytes(g, num_active);
    const size_t owner = sbnet::scatter_owner_workspace_bytes(g, num_active);
    size_t m = pull > color ? pull : color;
    if (cover > m) m = cover;
    return owner > m ? owner : m;
}

static int scatter_op(const float* x, int32_t num_active, const int32_t* bin_counts_device,
                      const int16_t* active_block_indices, const float* ybase, const int64_t* ybase_dims,
                      int ybase_rank, const int32_t* bsize, int bsize_len, const int32_t* bstride, int bstride_len,
                      const int32_t* boffset, int boffset_len, int add, int atomic, int transpose, float* y,
                      void* workspace, size_t workspace_bytes, void* stream)
{
    // order of checks as in sparse_gather.cc:307-327
    if (!pair_ok(bsize, bsize_len) || !pair_ok(bstride, bstride_len) || !pair_ok(boffset, boffset_len))
        return SBNET_EINVAL_PARAM_SHAPE;
    if (!atomic && add && !(bstride[0] >= bsize[0] && bstride[1] >= bsize[1])) return SBNET_EINVAL_OVERLAP;
    if (ybase_rank != 4) return SBNET_EINVAL_RANK;
    if (!ybase || !y || !ybase_dims || !dims_fit_int(ybase_dims)) return SBNET_EINVAL_ARG;
    const size_t count = (size_t)ybase_dims[0] * ybase_dims[1] * ybase_dims[2] * ybase_dims[3];
    {
        const uintptr_t a = reinterpret_cast<uintptr_t>(ybase), b = reinterpret_cast<uintptr_t>(y);
        const uintptr_t bytes = count * sizeof(float);
        if (a < b + bytes && b < a + bytes) return SBNET_EINVAL_ARG;
    }
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (!geom_ok((int)ybase_dims[0], (int)ybase_dims[1], (int)ybase_dims[2], (int)ybase_dims[3], bsize, bstride))
        return SBNET_EINVAL_ARG;
    // With scratch for one flag byte per pixel the output is built in one pass over its bytes: uncovered pixels
    // are copied, covered ones written by the scatter (which reads ybase where it adds).
    if (num_active > 0 && x && active_block_indices && !(add && atomic)) {
        sbnet::Geom g = make_geom((int)ybase_dims[0], (int)ybase_dims[1], (int)ybase_dims[2], (int)ybase_dims[3], bsize,
                                  bstride, boffset);
        g.countDev = bin_counts_device;
        bool done = false;
        SBNET_HIP(sbnet::launch_scatter_over_base(x, ybase, y, active_block_indices, num_active, g, transpose != 0,
                                                  add ? sbnet::SCATTER_ADD : sbnet::SCATTER_ASSIGN, workspace,
                                                  workspace_bytes, s, done));
        if (done) return SBNET_OK;
    }
    SBNET_HIP(sbnet::launch_copy(y, ybase, count, s));  // sparse_gather.cc:338-346, no stream sync
    return scatter_impl(x, num_active, bin_counts_device, active_block_indices, y, ybase_dims, bsize, bstride, boffset,
                        add, atomic, transpose, workspace, workspace_bytes, s);
}

int sbnet_sparse_scatter(const float* x, int32_t num_active, const int16_t* active_block_indices,
                         const float* ybase, const int64_t* ybase_dims, int ybase_rank,
                         const int32_t* bsize, int bsize_len, const int32_t* bstride, int bstride_len,
                         const int32_t* boffset, int boffset_len, int add, int atomic, int transpose,
                         float* y, void* workspace, size_t workspace_bytes, void* stream)
{
    return scatter_op(x, num_active, nullptr, active_block_indices, ybase, ybase_dims, ybase_rank, bsize, bsize_len,
                      bstride, bstride_len, boffset, boffset_len, add, atomic, transpose, y, workspace,
                      workspace_bytes, stream);
}

int sbnet_sparse_scatter_device_count(const float* x, const int32_t* bin_counts_device, int32_t max_active,
                                      const int16_t* active_block_indices, const float* ybase,
                                      const int64_t* ybase_dims, int ybase_rank, const int32_t* bsize, int bsize_len,
                                      const int32_t* bstride, int bstride_len, const int32_t* boffset,
                                      int boffset_len, int add, int atomic, int transpose, float* y,
                                      void* workspace, size_t workspace_bytes, void* stream)
{
    if (!bin_counts_device) return SBNET_EINVAL_ARG;
    return scatter_op(x, max_active, bin_counts_device, active_block_indices, ybase, ybase_dims, ybase_rank, bsize,
                      bsize_len, bstride, bstride_len, boffset, boffset_len, add, atomic, transpose, y, workspace,
                      workspace_bytes, stream);
}

static int scatter_var_op(const float* x, int32_t num_active, const int32_t* bin_counts_device,
                          const int16_t* active_block_indices, float* ybase, const int64_t* ybase_dims,
                          int ybase_rank, const int32_t* bsize, int bsize_len, const int32_t* bstride,
                          int bstride_len, const int32_t* boffset, int boffset_len, int add, int atomic,
                          int transpose, void* workspace, size_t workspace_bytes, void* stream)
{
    if (!pair_ok(bsize, bsize_len) || !pair_ok(bstride, bstride_len) || !pair_ok(boffset, boffset_len))
        return SBNET_EINVAL_PARAM_SHAPE;
    if (!atomic && add && !(bstride[0] >= bsize[0] && bstride[1] >= bsize[1])) return SBNET_EINVAL_OVERLAP;
    if (ybase_rank != 4) return SBNET_EINVAL_RANK;
    if (!ybase || !ybase_dims) return SBNET_EINVAL_ARG;
    return scatter_impl(x, num_active, bin_counts_device, active_block_indices, ybase, ybase_dims, bsize, bstride,
                        boffset, add, atomic, transpose, workspace, workspace_bytes, static_cast<hipStream_t>(stream));
}

int sbnet_sparse_scatter_var(const float* x, int32_t num_active, const int16_t* active_block_indices,
                             float* ybase, const int64_t* ybase_dims, int ybase_rank,
                             const int32_t* bsize, int bsize_len, const int32_t* bstride,
                             int bstride_len, const int32_t* boffset, int boffset_len, int add,
                             int atomic, int transpose, void* workspace, size_t workspace_bytes,
                             void* stream)
{
    return scatter_var_op(x, num_active, nullptr, active_block_indices, ybase, ybase_dims, ybase_rank, bsize,
                          bsize_len, bstride, bstride_len, boffset, boffset_len, add, atomic, transpose, workspace,
                          workspace_bytes, stream);
}

int sbnet_sparse_scatter_var_device_count(const float* x, const int32_t* bin_counts_device, int32_t max_active,
                                          const int16_t* active_block_indices, float* ybase,
                                          const int64_t* ybase_dims, int ybase_rank, const int32_t* bsize,
                                          int bsize_len, const int32_t* bstride, int bstride_len,
                                          const int32_t* boffset, int boffset_len, int add, int atomic,
                                          int transpose, void* workspace, size_t workspace_bytes, void* stream)
{
    if (!bin_counts_device) return SBNET_EINVAL_ARG;
    return scatter_var_op(x, max_active, bin_counts_device, active_block_indices, ybase, ybase_dims, ybase_rank,
                          bsize, bsize_len, bstride, bstride_len, boffset, boffset_len, add, atomic, transpose,
                          workspace, workspace_bytes, stream);
}

int sbnet_sparse_gather_grad(const float* dy, int32_t num_active, const int16_t* active_block_indices, float* dx,
                             const int64_t* x_dims, int x_rank, const int32_t* bsize, int bsize_len,
                             const int32_t* bstride, int bstride_len, const int32_t* boffset, int boffset_len,
                             int transpose, void* workspace, size_t workspace_bytes, void* stream)
{
    if (x_rank != 4) return SBNET_EINVAL_RANK;
    if (!pair_ok(bsize, bsize_len) || !pair_ok(bstride, bstride_len) || !pair_ok(boffset, boffset_len))
        return SBNET_EINVAL_PARAM_SHAPE;
    if (!dx || !x_dims || !dims_fit_int(x_dims) || num_active < 0) return SBNET_EINVAL_ARG;
    if (num_active > 0 && (!dy || !active_block_indices)) return SBNET_EINVAL_ARG;
    if (!geom_ok((int)x_dims[0], (int)x_dims[1], (int)x_dims[2], (int)x_dims[3], bsize, bstride)) return SBNET_EINVAL_ARG;
    const sbnet::Geom g = make_geom((int)x_dims[0], (int)x_dims[1], (int)x_dims[2], (int)x_dims[3], bsize, bstride, boffset);
    hipStream_t s = static_cast<hipStream_t>(stream);
    bool done = false;
    SBNET_HIP(sbnet::launch_scatter_onto_zeros(dy, dx, active_block_indices, num_active, g, transpose != 0, workspace,
                                               workspace_bytes, s, done));
    if (done) return SBNET_OK;
    SBNET_HIP(sbnet::launch_scatter_colored(dy, dx, active_block_indices, num_active, g, transpose != 0, workspace,
                                            workspace_bytes, s, done, true));
    if (done) return SBNET_OK;
    // no scratch, or a geometry the passes do not take: zeros everywhere, then the atomic scatter-add
    SBNET_HIP(sbnet::launch_zero(dx, (size_t)x_dims[0] * x_dims[1] * x_dims[2] * x_dims[3], s));
    return scatter_impl(dy, num_active, nullptr, active_block_indices, dx, x_dims, bsize, bstride, boffset, 1, 1, transpose,
                        workspace, workspace_bytes, s);
}

static bool aligned16(const void* p) { return p && (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

size_t sbnet_sparse_scatter_base_grad_workspace_bytes(int32_t num_active, const int64_t* dims, const int32_t* bsize,
                                                      const int32_t* bstride, const int32_t* boffset)
{
    if (num_active <= 0 || !dims || !dims_fit_int(dims) || !bsize || !bstride || !boffset ||
        !geom_ok((int)dims[0], (int)dims[1], (int)dims[2], (int)dims[3], bsize, bstride))
        return 0;
    return sbnet::scatter_base_grad_workspace_bytes(
        make_geom((int)dims[0], (int)dims[1], (int)dims[2], (int)dims[3], bsize, bstride, boffset), num_active);
}

int sbnet_sparse_scatter_base_grad(const float* dy, int32_t num_active, const int16_t* active_block_indices, float* dbase,
                                   const int64_t* dims, const int32_t* bsize, const int32_t* bstride, const int32_t* boffset,
                                   void* workspace, size_t workspace_bytes, void* stream)
{
    const size_t need = sbnet_sparse_scatter_base_grad_workspace_bytes(num_active, dims, bsize, bstride, boffset);
    if (!need || !active_block_indices || !workspace || workspace_bytes < need || !aligned16(dy) || !aligned16(dbase))
        return SBNET_EINVAL_ARG;
    const sbnet::Geom g = make_geom((int)dims[0], (int)dims[1], (int)dims[2], (int)dims[3], bsize, bstride, boffset);
    bool done = false;
    SBNET_HIP(sbnet::launch_scatter_base_grad(dy, dbase, active_block_indices, num_active, g, workspace, workspace_bytes,
                                              static_cast<hipStream_t>(stream), done));
    return done ? SBNET_OK : SBNET_EINVAL_ARG;
}

// The input side of a block convolution: checks, and the geometry of [N,H,W,C] read at the listed blocks.
static int conv_input(const float* x, const int64_t* x_dims, int32_t num_active, const int32_t* bin_counts_device,
                      const int16_t* active_block_indices, const int32_t* bsize, const int32_t* bstride,
                      const int32_t* boffset, sbnet::ConvArgs& c)
{
    if (!x || !x_dims || !active_block_indices || !bsize || !bstride || !boffset || num_active < 0 || !dims_fit_int(x_dims))
        return SBNET_EINVAL_ARG;
    if (!geom_ok((int)x_dims[0], (int)x_dims[1], (int)x_dims[2], (int)x_dims[3], bsize, bstride)) return SBNET_EINVAL_ARG;
    c = sbnet::ConvArgs();
    c.a = x;
    c.idx = active_block_indices;
    c.N = (int)x_dims[0]; c.H = (int)x_dims[1]; c.W = (int)x_dims[2]; c.C = (int)x_dims[3];
    c.U = bstride[0]; c.V = bstride[1]; c.oh = boffset[0]; c.ow = boffset[1];
    c.M = num_active;
    c.countDev = bin_counts_device;
    return SBNET_OK;
}

// The kernel side: w [kh,kw,C,K] on blocks of R x S pixels, false where they do not fit together.
static bool conv_kernel(sbnet::ConvArgs& c, const float* w, const int32_t* w_dims, int R, int S)
{
    if (!w || w_dims[0] <= 0 || w_dims[1] <= 0 || w_dims[2] != c.C || w_dims[3] <= 0) return false;
    c.w = w;
    c.kh = w_dims[0]; c.kw = w_dims[1]; c.K = w_dims[3];
    c.Ro = R - c.kh + 1; c.So = S - c.kw + 1;
    return c.Ro > 0 && c.So > 0;
}

int sbnet_block_conv(const float* x, const int64_t* x_dims, int32_t num_active, const int32_t* bin_counts_device,
                     const int16_t* active_block_indices, const int32_t* bsize, const int32_t* bstride,
                     const int32_t* boffset, const float* w, const int32_t* w_dims, float* q, void* stream)
{
    sbnet::ConvArgs c;
    const int st = conv_input(x, x_dims, num_active, bin_counts_device, active_block_indices, bsize, bstride, boffset, c);
    if (st != SBNET_OK) return st;
    if (!q || !w_dims || !conv_kernel(c, w, w_dims, bsize[0], bsize[1]) || !sbnet::conv_fits(c)) return SBNET_EINVAL_ARG;
    c.y = q;
    SBNET_HIP(sbnet::launch_block_conv(c, static_cast<hipStream_t>(stream)));
    return SBNET_OK;
}

// The three convolutions of a bottleneck; the result of each is the block stack the next one reads.
static int bottleneck_args(sbnet::ConvArgs (&c)[3], const float* const* weights, const int32_t* w_dims,
                           const float* const* batch_norms, float eps, const int32_t* bsize)
{
    int R = bsize[0], S = bsize[1];
    sbnet::BnArgs bn[3];
    for (int i = 0; i < 3; ++i) {
        const float* const* b = batch_norms + 4 * i;
        if (i > 0 && (!b[0] || !b[1] || !b[2] || !b[3])) return SBNET_EINVAL_ARG;
        if (i == 0 && b[0] && (!b[1] || !b[2] || !b[3])) return SBNET_EINVAL_ARG;
        bn[i] = sbnet::BnArgs{b[0], b[1], b[2], b[3], eps};
    }
    for (int i = 0; i < 3; ++i) {
        if (i > 0) {
            c[i] = sbnet::ConvArgs();
            c[i].N = c[i].M = c[0].M;
            c[i].H = R; c[i].W = S; c[i].C = c[i - 1].K;
            c[i].countDev = c[0].countDev;
        }
        if (!conv_kernel(c[i], weights[i], w_dims + 4 * i, R, S)) return SBNET_EINVAL_ARG;
        R = c[i].Ro; S = c[i].So;
        c[i].post = i < 2 ? bn[i + 1] : sbnet::BnArgs();
    }
    c[0].pre = bn[0];
    for (int i = 0; i < 3; ++i)
        if (!sbnet::conv_fits(c[i])) return SBNET_EINVAL_ARG;
    return SBNET_OK;
}

size_t sbnet_block_bottleneck_workspace_bytes(int32_t num_active, const int32_t* bsize, const int32_t* w_dims)
{
    if (num_active <= 0 || !bsize || !w_dims) return 0;
    size_t total = 0;
    int64_t R = bsize[0], S = bsize[1];
    for (int i = 0; i < 2; ++i) {
        R -= w_dims[4 * i] - 1;
        S -= w_dims[4 * i + 1] - 1;
        if (R <= 0 || S <= 0 || w_dims[4 * i + 3] <= 0) return 0;
        total += ((size_t)num_active * R * S * w_dims[4 * i + 3] * sizeof(float) + 255) & ~(size_t)255;
    }
    return total;
}

int sbnet_block_bottleneck(const float* x, const int64_t* x_dims, int32_t num_active, const int32_t* bin_counts_device,
                           const int16_t* active_block_indices, const int32_t* bsize, const int32_t* bstride,
                           const int32_t* boffset, const float* const* weights, const int32_t* w_dims,
                           const float* const* batch_norms, float bn_eps, float* q, float* y,
                           const int32_t* out_bstride, void* workspace, size_t workspace_bytes, void* stream)
{
    sbnet::ConvArgs c[3];
    const int st = conv_input(x, x_dims, num_active, bin_counts_device, active_block_indices, bsize, bstride, boffset, c[0]);
    if (st != SBNET_OK) return st;
    if (!weights || !w_dims || !batch_norms || (q != nullptr) == (y != nullptr)) return SBNET_EINVAL_ARG;
    if (num_active == 0) return SBNET_OK;
    const int st2 = bottleneck_args(c, weights, w_dims, batch_norms, bn_eps, bsize);
    if (st2 != SBNET_OK) return st2;
    const size_t need = sbnet_block_bottleneck_workspace_bytes(num_active, bsize, w_dims);
    if (!workspace || workspace_bytes < need || (reinterpret_cast<uintptr_t>(workspace) & 15)) return SBNET_EINVAL_ARG;
    float* const h1 = static_cast<float*>(workspace);
    float* const h2 = h1 + (((size_t)num_active * c[0].Ro * c[0].So * c[0].K * sizeof(float) + 255) & ~(size_t)255) / sizeof(float);
    c[0].y = h1;
    c[1].a = h1;
    c[1].y = h2;
    c[2].a = h2;
    if (y) {
        // added at the blocks' positions: their results must not meet, and the image has the last kernel's channels
        if (!out_bstride || out_bstride[0] < c[2].Ro || out_bstride[1] < c[2].So || c[2].K != c[0].C) return SBNET_EINVAL_ARG;
        c[2].y = y;
        c[2].oidx = active_block_indices;
        c[2].oN = c[0].N; c[2].oH = c[0].H; c[2].oW = c[0].W;
        c[2].oU = out_bstride[0]; c[2].oV = out_bstride[1];
        c[2].add = 1;
        if (!sbnet::conv_fits(c[2])) return SBNET_EINVAL_ARG;
    } else {
        c[2].y = q;
    }
    hipStream_t s = static_cast<hipStream_t>(stream);
    SBNET_HIP(sbnet::launch_block_conv(c[0], s));
    bool done = false;
    SBNET_HIP(sbnet::launch_block_conv_next(c[1], c[2], s, done));
    for (int i = 1; i < 3 && !done; ++i) SBNET_HIP(sbnet::launch_block_conv(c[i], s));
    return SBNET_OK;
}

// The gradients of a bottleneck's three convolutions as launch_block_conv_grad takes them (c[i]: from the gradient of
// result i to that of its input), the kernels' gradients, and where what lies between them is in the scratch.
struct BottleneckGrad {
    sbnet::ConvArgs c[3];
    sbnet::WgradArgs w[3];
    size_t sums[3], sumBytes;                 // of the batch norms
    size_t z[3], act[3], kernel[3], dz[4];    // NHWC stacks (dz[3]: dq), kernels [C,kh,kw,K]
    size_t part, total;
};

static bool bottleneck_grad_plan(int32_t num_blocks, const int32_t* bsize, const int32_t* w_dims, BottleneckGrad& b)
{
    if (num_blocks <= 0 || !bsize || !w_dims || bsize[0] <= 0 || bsize[1] <= 0) return false;
    auto take = [](size_t& at, uint64_t bytes) {
        const size_t here = at;
        at += (size_t)((bytes + 255) & ~(uint64_t)255);
        return here;
    };
    int R = bsize[0], S = bsize[1];
    size_t at = 0;
    for (int i = 0; i < 3; ++i) {
        const int32_t* d = w_dims + 4 * i;
        if (d[0] <= 0 || d[1] <= 0 || d[2] <= 0 || d[3] <= 0 || d[0] > R || d[1] > S || (i && d[2] != w_dims[4 * i - 1])) return false;
        sbnet::ConvArgs& c = b.c[i];
        c = sbnet::ConvArgs();
        c.N = c.M = num_blocks;
        c.kh = d[0]; c.kw = d[1]; c.K = d[2]; c.C = d[3];
        c.Ro = R; c.So = S;
        c.H = R -= d[0] - 1;
        c.W = S -= d[1] - 1;
        if (!sbnet::conv_grad_fits(c) || (int64_t)num_blocks * c.Ro * c.So < 2) return false;
        sbnet::WgradArgs& w = b.w[i];
        w = sbnet::WgradArgs();
        w.M = num_blocks; w.R = c.Ro; w.S = c.So; w.C = c.K; w.K = c.C; w.kh = c.kh; w.kw = c.kw;
        b.sums[i] = take(at, sizeof(double) * sbnet::GRAD_SLOTS * 2 * c.K);
    }
    b.sumBytes = at;
    for (int i = 0; i < 3; ++i) {
        const sbnet::ConvArgs& c = b.c[i];
        const uint64_t stack = sizeof(float) * (uint64_t)num_blocks * c.Ro * c.So * c.K;
        b.z[i] = take(at, stack);
        b.act[i] = take(at, stack);
        b.dz[i] = take(at, stack);
        b.kernel[i] = take(at, sizeof(float) * (uint64_t)c.K * c.kh * c.kw * c.C);
    }
    b.dz[3] = take(at, sizeof(float) * (uint64_t)num_blocks * R * S * b.c[2].C);
    // (the pixels are split by how many kernels there are to do: the most that any of them together need)
    size_t part = 0;
    for (int s = 1; s < 8; ++s) {
        sbnet::WgradArgs w[3];
        int n = 0;
        for (int i = 0; i < 3; ++i)
            if (s >> i & 1) w[n++] = b.w[i];
        part = std::max(part, sbnet::wgrad_workspace_bytes(w, n));
    }
    b.part = take(at, part);
    b.total = at;
    return true;
}

size_t sbnet_bottleneck_grad_workspace_bytes(int32_t num_blocks, const int32_t* bsize, const int32_t* w_dims)
{
    BottleneckGrad b;
    return bottleneck_grad_plan(num_blocks, bsize, w_dims, b) ? b.total : 0;
}

int sbnet_bottleneck_grad(const float* dq, int32_t num_blocks, const int32_t* bsize, const float* const* z,
                          const float* const* act, const float* const* mean, const float* const* inv,
                          const float* const* gamma, const float* const* weights, const int32_t* w_dims, float* dp,
                          float* const* dw, float* const* dgamma, float* const* dbeta, void* workspace,
                          size_t workspace_bytes, void* stream)
{
    BottleneckGrad b;
    if (!dq || !z || !act || !mean || !inv || !gamma || !weights || !dw || !dgamma || !dbeta || !workspace ||
        (reinterpret_cast<uintptr_t>(workspace) & 15) || !bottleneck_grad_plan(num_blocks, bsize, w_dims, b) ||
        workspace_bytes < b.total)
        return SBNET_EINVAL_ARG;
    for (int i = 0; i < 3; ++i)
        if (!z[i] || !act[i] || !mean[i] || !inv[i] || !gamma[i] || !weights[i] || (reinterpret_cast<uintptr_t>(dw[i]) & 15))
            return SBNET_EINVAL_ARG;
    // how far down the gradient has to go: whether batch norm i or anything in front of it has one that is asked for
    bool needs[3], any = dp != nullptr;
    for (int i = 0; i < 3; ++i) {
        needs[i] = any = any || dgamma[i] || dbeta[i];
        any = any || dw[i];
    }
    if (!any) return SBNET_OK;
    hipStream_t s = static_cast<hipStream_t>(stream);
    uint8_t* const ws = static_cast<uint8_t*>(workspace);
    auto at = [&](size_t offset) { return reinterpret_cast<float*>(ws + offset); };

    sbnet::TransposeArgs t[10];
    int n = 0;
    for (int i = 0; i < 3; ++i) {
        const sbnet::ConvArgs& c = b.c[i];
        const uint32_t M = (uint32_t)num_blocks, C = (uint32_t)c.K, P = (uint32_t)(c.Ro * c.So);
        if (needs[i]) t[n++] = sbnet::TransposeArgs{z[i], at(b.z[i]), M, C, P};
        if (needs[i] || dw[i]) t[n++] = sbnet::TransposeArgs{act[i], at(b.act[i]), M, C, P};
        if (needs[i]) t[n++] = sbnet::TransposeArgs{weights[i], at(b.kernel[i]), 1, (uint32_t)c.C, C * (uint32_t)(c.kh * c.kw)};
    }
    t[n++] = sbnet::TransposeArgs{dq, at(b.dz[3]), (uint32_t)num_blocks, (uint32_t)b.c[2].C, (uint32_t)(b.c[2].H * b.c[2].W)};
    SBNET_HIP(sbnet::launch_transposes(t, n, s, at(0), needs[2] ? (uint32_t)(b.sumBytes / sizeof(float)) : 0u));
    for (int i = 2; i >= 0 && needs[i]; --i) {
        sbnet::ConvArgs& c = b.c[i];
        c.a = at(b.dz[i + 1]);
        c.w = at(b.kernel[i]);
        c.y = at(b.dz[i]);
        c.norm = sbnet::NormGradArgs{at(b.z[i]), at(b.act[i]), mean[i], inv[i], gamma[i], reinterpret_cast<double*>(ws + b.sums[i])};
        SBNET_HIP(sbnet::launch_block_conv_grad(c, s));
        SBNET_HIP(sbnet::launch_norm_grad(at(b.dz[i]), c.norm, (uint32_t)(c.M * c.Ro * c.So), c.K, dgamma[i], dbeta[i], s));
    }
    sbnet::WgradArgs w[3];
    int kernels = 0;
    for (int i = 0; i < 3; ++i) {
        if (!dw[i]) continue;
        b.w[i].act = at(b.act[i]);
        b.w[i].dz = at(b.dz[i + 1]);
        b.w[i].dw = dw[i];
        w[kernels++] = b.w[i];
    }
    if (kernels) SBNET_HIP(sbnet::launch_wgrad(w, kernels, ws + b.part, s));
    if (!dp) return SBNET_OK;
    t[0] = sbnet::TransposeArgs{at(b.dz[0]), dp, (uint32_t)num_blocks, (uint32_t)(b.c[0].Ro * b.c[0].So), (uint32_t)b.c[0].K};
    SBNET_HIP(sbnet::launch_transposes(t, 1, s));
    return SBNET_OK;
}

int sbnet_relu(float* x, int64_t count, void* stream)
{
    if (count < 0 || (count > 0 && (!x || (reinterpret_cast<uintptr_t>(x) & 15)))) return SBNET_EINVAL_ARG;
    SBNET_HIP(sbnet::launch_relu(x, (size_t)count, static_cast<hipStream_t>(stream)));
    return SBNET_OK;
}

int sbnet_kernels_oihw(const float* const* weights, const int32_t* w_dims, float* const* out, int count, void* stream)
{
    if (!weights || !w_dims || !out || count < 1 || count > 3) return SBNET_EINVAL_ARG;
    for (int i = 0; i < count; ++i) {
        const int32_t* d = w_dims + 4 * i;
        if (!weights[i] || !out[i] || d[0] <= 0 || d[1] <= 0 || d[2] <= 0 || d[3] <= 0 ||
            (int64_t)d[0] * d[1] >= (1ll << 30) || (int64_t)d[0] * d[1] * d[2] >= (1ll << 30) ||
            (int64_t)d[0] * d[1] * d[2] * d[3] >= (1ll << 30))
            return SBNET_EINVAL_ARG;
    }
    SBNET_HIP(sbnet::launch_kernels(weights, w_dims, out, count, static_cast<hipStream_t>(stream)));
    return SBNET_OK;
}

int sbnet_sparse_scatter_functor(const float* x, int N, int H, int W, int C, float* y, int bOffsH0,
                                 int bOffsW0, int bSzH, int bSzW, int bStrH, int bStrW, int numActive,
                                 const int16_t* activeBlockIndices, int add, int transpose, int atomic,
                                 void* stream)
{
    return sbnet_sparse_scatter_functor_ws(x, N, H, W, C, y, bOffsH0, bOffsW0, bSzH, bSzW, bStrH, bStrW, numActive,
                                           activeBlockIndices, add, transpose, atomic, nullptr, 0, stream);
}

int sbnet_sparse_scatter_functor_ws(const float* x, int N, int H, int W, int C, float* y, int bOffsH0,
                                    int bOffsW0, int bSzH, int bSzW, int bStrH, int bStrW, int numActive,
                                    const int16_t* activeBlockIndices, int add, int transpose, int atomic,
                                    void* workspace, size_t workspace_bytes, void* stream)
{
    const int32_t bsize[2] = {bSzH, bSzW}, bstride[2] = {bStrH, bStrW}, boffset[2] = {bOffsH0, bOffsW0};
    const int64_t dims[4] = {N, H, W, C};
    return scatter_impl(x, numActive, nullptr, activeBlockIndices, y, dims, bsize, bstride, boffset, add, atomic,
                        transpose, workspace, workspace_bytes, static_cast<hipStream_t>(stream));
}

void* sbnet_scratch_acquire(size_t bytes, void* stream)
{
    if (bytes == 0) return nullptr;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
    }
    hipStream_t s = static_cast<hipStream_t>(stream);
    std::lock_guard<std::mutex> lock(g_scratchMutex);
    ScratchSlot* slot = nullptr;
    for (ScratchSlot& c : g_scratch)
        if (c.dev == dev && c.stream == s) slot = &c;
    if (slot && slot->bytes >= bytes) return slot->ptr;
    // growing allocates, which a stream under capture must not do
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &cap) != hipSuccess) {
        (void)hipGetLastError();  // a stream that cannot be asked is not being captured
        cap = hipStreamCaptureStatusNone;
    }
    if (cap != hipStreamCaptureStatusNone) return nullptr;
    size_t want = (size_t)1 << 20;
    while (want < bytes) want <<= 1;
    void* p = nullptr;
    if (hipMalloc(&p, want) != hipSuccess || !p) {
        (void)hipGetLastError();
        return nullptr;
    }
    if (slot) {
        g_scratchRetired.push_back(*slot);  // may still be handed out or in use by queued work: kept until shutdown
        slot->ptr = p;
        slot->bytes = want;
    } else {
        g_scratch.push_back(ScratchSlot{dev, s, p, want});
    }
    return p;
}

int sbnet_shutdown(void)
{
    hipError_t first = hipSuccess;
    {
        std::lock_guard<std::mutex> lock(g_scratchMutex);
        for (std::vector<ScratchSlot>* list : {&g_scratch, &g_scratchRetired}) {
            for (ScratchSlot& c : *list) {
                int cur = 0;
                (void)hipGetDevice(&cur);
                (void)hipSetDevice(c.dev);
                hipError_t e = hipFree(c.ptr);  // waits for the device
                (void)hipSetDevice(cur);
                if (e != hipSuccess && first == hipSuccess) first = e;
            }
            list->clear();
        }
    }
    {
        // only the words no thread holds; a live thread keeps its own until it ends
        std::lock_guard<std::mutex> lock(g_signalMutex);
        for (int d = 0; d < MAX_SIGNAL_DEVICES; ++d) {
            for (unsigned long long* w : g_signalFree[d]) {
                hipError_t e = hipHostFree(w);
                if (e != hipSuccess && first == hipSuccess) first = e;
                for (size_t i = 0; i < g_signalAll.size(); ++i)
                    if (g_signalAll[i] == w) {
                        g_signalAll[i] = g_signalAll.back();
                        g_signalAll.pop_back();
                        break;
                    }
            }
            g_signalFree[d].clear();
        }
    }
    if (first != hipSuccess) return hip_fail(first);
    return SBNET_OK;
}

// Test hook, not part of the public header: while on (per calling thread), gather and scatter never take a
// kernel instance compiled for one block shape, so the tests cover the run-time-geometry kernels on the
// benchmark shapes as well.  Returns the previous setting.
int sbnet_test_force_generic(int on)
{
    const int prev = t_forceGeneric;
    t_forceGeneric = on ? 1 : 0;
    return prev;
}

// Test hook, not part of the public header: the tile the planar kernels would choose (no device work, so the
// choice can be checked on a machine without a GPU).  out must hold 11 int32; see sbnet::tile_choice.
int sbnet_test_tile_choice(int kind, int N, int H, int W, int C, int R, int S, int U, int V, int num_active, int vec,
                           int y_aligned_to, int32_t* out)
{
    const int32_t bsize[2] = {R, S}, bstride[2] = {U, V}, boffset[2] = {0, 0};
    if (!out || !geom_ok(N, H, W, C, bsize, bstride)) return -1;
    return sbnet::tile_choice(kind, make_geom(N, H, W, C, bsize, bstride, boffset), num_active, vec, y_aligned_to, out);
}

// Test hook, not part of the public header: the copying scatter's route.  dims, geometry: four and six ints (bsize, bstride,
// boffset); out must hold 5 int32; see sbnet::scatter_route.
int sbnet_test_scatter_route(const int32_t* dims, const int32_t* geometry, int num_active, int transpose, int add, int y_aligned_to,
                             int32_t* out)
{
    if (!dims || !geometry || !out || num_active <= 0 || !geom_ok(dims[0], dims[1], dims[2], dims[3], geometry, geometry + 2)) return -1;
    sbnet::scatter_route(make_geom(dims[0], dims[1], dims[2], dims[3], geometry, geometry + 2, geometry + 4), num_active, transpose != 0,
                         add != 0, y_aligned_to, out);
    return 0;
}

int sbnet_copy_tensor(float* dst, const float* src, size_t count, void* stream)
{
    if (count && (!dst || !src)) return SBNET_EINVAL_ARG;
    SBNET_HIP(sbnet::launch_copy(dst, src, count, static_cast<hipStream_t>(stream)));
    return SBNET_OK;
}

int sbnet_timer_start(void* stream, int64_t* start_event)
{
    if (!start_event) return SBNET_EINVAL_ARG;
    hipEvent_t ev;
    SBNET_HIP(hipEventCreate(&ev));
    hipError_t e = hipEventRecord(ev, static_cast<hipStream_t>(stream));
    if (e != hipSuccess) {
        (void)hipEventDestroy(ev);
        return hip_fail(e);
    }
    *start_event = (int64_t)reinterpret_cast<intptr_t>(ev);
    return SBNET_OK;
}

int sbnet_timer_end(int64_t start_event, void* stream, float* dt_ms)
{
    if (!start_event || !dt_ms) return SBNET_EINVAL_ARG;
    hipEvent_t start = reinterpret_cast<hipEvent_t>((intptr_t)start_event);
    hipEvent_t end;
    SBNET_HIP(hipEventCreate(&end));
    hipError_t e = hipEventRecord(end, static_cast<hipStream_t>(stream));
    if (e == hipSuccess) e = hipEventSynchronize(end);
    if (e == hipSuccess) e = hipEventElapsedTime(dt_ms, start, end);
    (void)hipEventDestroy(end);
    (void)hipEventDestroy(start);
    if (e != hipSuccess) return hip_fail(e);
    return SBNET_OK;
}

}  // extern "C"
