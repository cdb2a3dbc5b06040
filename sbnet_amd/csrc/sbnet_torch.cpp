// The op wrappers' common case in native code (Python module sbnet_amd._native): plain arguments in, one C-ABI call, the
// result out.  Everything else (parameters that are no pair of ints, tensors that need a copy or a cast, sizes and types
// that are an error) is left to the Python wrappers of ops.py, which these functions tell by returning None before
// anything has been allocated or enqueued.
//
// A call through ctypes costs 25-35 us of host time for argument conversion, two numpy round trips per parameter pair,
// the device context manager and the call itself: the three ops of a step took 114 us from Python on a [1,64,64,16] map
// whose kernels take 13.  Through this module the step takes 27 us (26-28 from box to box).
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/autocast_mode.h>
#include <ATen/core/grad_mode.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>

#include <map>
#include <mutex>
#include <utility>

#include "../../include/sbnet_amd.h"

namespace {

PyObject* g_check = nullptr;      // ops._check: raises the exception of a status
PyObject* g_by_layers = nullptr;  // sparse_conv._residual_by_layers: a residual function's gradients through its layers
PyObject* g_gather_gradient = nullptr;    // autograd.gather_gradient, autograd.scatter_gradients: the gradients by the general
PyObject* g_scatter_gradients = nullptr;  // wrappers

struct Pair {
    int32_t v[2];
};

bool int_of(PyObject* o, int32_t* out)
{
    if (!PyLong_CheckExact(o)) return false;
    int overflow = 0;
    const long v = PyLong_AsLongAndOverflow(o, &overflow);
    if (overflow || v < INT32_MIN || v > INT32_MAX) return false;
    *out = (int32_t)v;
    return true;
}

// A list or tuple of exactly two ints.
bool pair_of(PyObject* o, Pair& p)
{
    if (PyList_CheckExact(o))
        return PyList_GET_SIZE(o) == 2 && int_of(PyList_GET_ITEM(o, 0), &p.v[0]) && int_of(PyList_GET_ITEM(o, 1), &p.v[1]);
    if (PyTuple_CheckExact(o))
        return PyTuple_GET_SIZE(o) == 2 && int_of(PyTuple_GET_ITEM(o, 0), &p.v[0]) && int_of(PyTuple_GET_ITEM(o, 1), &p.v[1]);
    return false;
}

bool has_memory(const at::Tensor& t, at::ScalarType type)
{
    return t.defined() && t.scalar_type() == type && t.layout() == at::kStrided && t.has_storage() &&
           (t.numel() == 0 || t.const_data_ptr());
}

// A tensor (or parameter) with memory behind it: no subclass and no wrapper of a transform (vmap, grad, fake tensors).
const at::Tensor* plain_tensor(PyObject* o, at::ScalarType type)
{
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    return has_memory(t, type) ? &t : nullptr;
}

// A contiguous one on the GPU.
const at::Tensor* dev_tensor(PyObject* o, at::ScalarType type)
{
    const at::Tensor* t = plain_tensor(o, type);
    return t && t->is_cuda() && t->is_contiguous() ? t : nullptr;
}

// The same of a tensor that comes from the autograd engine: a gradient, or what a saved-tensor hook handed back.
bool is_dev(const at::Tensor& t, at::ScalarType type)
{
    return t.defined() && !t.key_set().has(c10::DispatchKey::Python) && has_memory(t, type) && t.is_cuda() && t.is_contiguous();
}

const at::Tensor* dev_f32(PyObject* o) { return dev_tensor(o, at::kFloat); }

// The block list with its count: on the host (M) or on the device (count, M then the list's capacity).
struct Blocks {
    const at::Tensor* idx;
    int32_t M;
    const int32_t* count;
};

bool is_list(const at::Tensor& idx) { return idx.dim() == 2 && idx.size(1) == 3 && idx.size(0) <= INT32_MAX; }

bool blocks_of(PyObject* counts, PyObject* list, Blocks& b)
{
    b.idx = dev_tensor(list, at::kShort);
    if (!b.idx || !is_list(*b.idx)) return false;
    b.count = nullptr;
    if (THPVariable_Check(counts)) {
        const at::Tensor* c = plain_tensor(counts, at::kInt);
        if (!c || c->numel() < 1) return false;
        if (c->is_cuda()) {
            if (c->device() != b.idx->device()) return false;
            b.count = static_cast<const int32_t*>(c->data_ptr());
            b.M = (int32_t)b.idx->size(0);
            return true;
        }
        if (!c->is_cpu()) return false;
        b.M = *static_cast<const int32_t*>(c->const_data_ptr());
    } else if (PyList_CheckExact(counts) && PyList_GET_SIZE(counts) >= 1) {
        if (!int_of(PyList_GET_ITEM(counts, 0), &b.M)) return false;
    } else {
        return false;
    }
    return b.M >= 0 && b.M <= b.idx->size(0);
}

bool is_stack(const at::Tensor& t, int32_t M, int64_t C, const Pair& bsize, bool planar)
{
    return t.dim() == 4 && t.size(0) >= M && t.size(1) == (planar ? C : bsize.v[0]) &&
           t.size(2) == (planar ? bsize.v[0] : bsize.v[1]) && t.size(3) == (planar ? bsize.v[1] : C);
}

at::Tensor empty_f32(at::IntArrayRef size, const at::Tensor& like)
{
    return at::detail::empty_cuda(size, at::kFloat, like.device(), c10::nullopt);
}

at::Tensor empty_stack(int32_t M, int64_t C, const Pair& bsize, bool planar, const at::Tensor& like)
{
    return planar ? empty_f32({M, C, bsize.v[0], bsize.v[1]}, like) : empty_f32({M, bsize.v[0], bsize.v[1], C}, like);
}

void* stream_of(const at::Tensor& t) { return c10::hip::getCurrentHIPStream(t.get_device()).stream(); }

// Scratch of the calls of one stream, which run in order: one buffer per (device, stream) that only grows.  The GIL
// guards the table; a call enqueues its launches under the buffer's lock, so that another thread's on the same stream come
// before or after them and not in between.  A buffer that a call still holds when another thread grows it stays alive
// until that call's work has been enqueued, and torch's allocator hands its memory on in the order of the stream.
struct Scratch {
    at::Tensor buffer;
    std::recursive_mutex busy;   // (waited for without the GIL, which its holder may want)
};

std::map<std::pair<int, void*>, Scratch>* g_workspaces = nullptr;   // entries stay, release_workspaces() drops the buffers

Scratch& stream_scratch(int device)
{
    if (!g_workspaces) g_workspaces = new std::map<std::pair<int, void*>, Scratch>();
    return (*g_workspaces)[std::make_pair(device, (void*)c10::hip::getCurrentHIPStream((c10::DeviceIndex)device).stream())];
}

struct Workspace {
    at::Tensor buffer;
    std::recursive_mutex* busy = nullptr;
};

// (While the stream is being captured the scratch is a tensor of the graph's own pool: the graph keeps its address, and the
// kept buffer may grow or be released before a replay, or be in use by the stream's own calls during one.)
Workspace workspace(const at::Device& device, int64_t bytes)
{
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(c10::hip::getCurrentHIPStream(device.index()).stream(), &capture) != hipSuccess) (void)hipGetLastError();
    if (capture == hipStreamCaptureStatusActive) return {at::detail::empty_cuda({bytes}, at::kByte, device, c10::nullopt), nullptr};
    Scratch& s = stream_scratch(device.index());
    if (!s.buffer.defined() || s.buffer.numel() < bytes)
        s.buffer = at::detail::empty_cuda({bytes < (1 << 16) ? (1 << 16) : bytes}, at::kByte, device, c10::nullopt);
    return {s.buffer, &s.busy};
}

// Scratch of one call, as the tensors between torch's operators are: for the layers, whose stacks are large, may belong to a
// captured graph, and must not be shared with another thread that enqueues on the same stream.  Given back at the end of
// the call, in the order of the stream.
at::Tensor own_scratch(const at::Tensor& like, size_t bytes)
{
    return at::detail::empty_cuda({(int64_t)bytes}, at::kByte, like.device(), c10::nullopt);
}

// Runs a library call without the GIL, as ctypes does; raises on a status other than SBNET_OK.
template <typename F>
bool call(F f, std::recursive_mutex* busy = nullptr)
{
    int status;
    Py_BEGIN_ALLOW_THREADS
    if (busy) busy->lock();
    status = f();
    if (busy) busy->unlock();
    Py_END_ALLOW_THREADS
    if (status == SBNET_OK) return true;
    PyObject* r = PyObject_CallFunction(g_check, "i", status);
    if (r) {
        Py_DECREF(r);
        PyErr_SetString(PyExc_RuntimeError, "sbnet status was not raised");
    }
    return false;
}

[[noreturn]] void raise_pending()
{
    python_error e;
    e.persist();
    throw e;
}

// The same for code that C++ calls: throws what was raised.
template <typename F>
void run(F f, std::recursive_mutex* busy = nullptr)
{
    if (!call(f, busy)) raise_pending();
}

// A function of the module: N arguments, of which those after the first FEWEST may be missing (None), and no C++ exception
// through the interpreter's frames.
template <PyObject* (*F)(PyObject* const*), Py_ssize_t N, Py_ssize_t FEWEST = N>
PyObject* entry(PyObject*, PyObject* const* a, Py_ssize_t n)
{
    if (n > N || n < FEWEST) {
        PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", N, n);
        return nullptr;
    }
    PyObject* all[N];
    if constexpr (FEWEST < N) {
        for (Py_ssize_t i = 0; i < N; ++i) all[i] = i < n ? a[i] : Py_None;
        a = all;
    }
    try {
        return F(a);
    } catch (...) {
        torch::translate_exception_to_python(std::current_exception());
    }
    return nullptr;
}

// The same for an op: left to the general wrappers while something looks on at torch's operators.
template <PyObject* (*F)(PyObject* const*), Py_ssize_t N, Py_ssize_t FEWEST = N>
PyObject* op_entry(PyObject* self, PyObject* const* a, Py_ssize_t n)
{
    if (c10::impl::TorchDispatchModeTLS::any_modes_set()) Py_RETURN_NONE;
    return entry<F, N, FEWEST>(self, a, n);
}

// reduce_mask(mask, bcount, bsize, bstride, boffset, tol, avgpool, sync) -> (active_block_indices, bin_counts)
PyObject* reduce_mask(PyObject* const* a)
{
    const at::Tensor* mask = dev_f32(a[0]);
    Pair bc, bs, bt, bo;
    if (!mask || !pair_of(a[1], bc) || !pair_of(a[2], bs) || !pair_of(a[3], bt) || !pair_of(a[4], bo)) Py_RETURN_NONE;
    if (!(mask->dim() == 3 || (mask->dim() == 4 && mask->size(3) == 1)) || !PyFloat_CheckExact(a[5])) Py_RETURN_NONE;
    for (int i = 0; i < 3; ++i)
        if (mask->size(i) <= 0 || mask->size(i) > INT32_MAX) Py_RETURN_NONE;
    const int N = (int)mask->size(0), H = (int)mask->size(1), W = (int)mask->size(2);
    if (bc.v[0] <= 0 || bc.v[1] <= 0 || N > 32768 || bc.v[0] > 32768 || bc.v[1] > 32768) Py_RETURN_NONE;
    const int64_t T = (int64_t)N * bc.v[0] * bc.v[1];
    if (T > INT32_MAX) Py_RETURN_NONE;
    const float tol = (float)PyFloat_AS_DOUBLE(a[5]);
    const int avgpool = PyObject_IsTrue(a[6]), sync = PyObject_IsTrue(a[7]);
    if (avgpool < 0 || sync < 0) return nullptr;
    c10::DeviceGuard guard(mask->device());
    at::Tensor idx = at::detail::empty_cuda({T, 3}, at::kShort, mask->device(), c10::nullopt);
    at::Tensor count = sync ? at::empty({1}, at::kInt) : at::detail::empty_cuda({1}, at::kInt, mask->device(), c10::nullopt);
    int32_t* const cp = static_cast<int32_t*>(count.data_ptr());
    const Workspace scratch = workspace(mask->device(), (int64_t)sbnet_reduce_mask_workspace_bytes(N, bc.v, 2));
    const at::Tensor& ws = scratch.buffer;
    void* const stream = stream_of(*mask);
    if (!call([&] {
            return sbnet_reduce_mask(static_cast<const float*>(mask->data_ptr()), N, H, W, bc.v, 2, bs.v, 2, bt.v, 2, bo.v,
                                     2, tol, avgpool, static_cast<int16_t*>(idx.data_ptr()), sync ? cp : nullptr,
                                     sync ? nullptr : cp, ws.data_ptr(), (size_t)ws.numel(), stream);
        }, scratch.busy))
        return nullptr;
    PyObject* pi = THPVariable_Wrap(std::move(idx));
    PyObject* pc = THPVariable_Wrap(std::move(count));
    PyObject* t = pi && pc ? PyTuple_Pack(2, pi, pc) : nullptr;
    Py_XDECREF(pi);
    Py_XDECREF(pc);
    return t;
}

struct Gather {
    const at::Tensor* x;
    Blocks b;
    Pair bs, bt, bo;
    int transpose;
};

// x, bin_counts, active_block_indices, bsize, bstride, boffset, transpose; false where the general wrapper has to see to them.
bool gather_of(PyObject* const* a, Gather& g)
{
    g.x = dev_f32(a[0]);
    if (!g.x || g.x->dim() != 4 || !blocks_of(a[1], a[2], g.b) || g.b.idx->device() != g.x->device() || !pair_of(a[3], g.bs) ||
        !pair_of(a[4], g.bt) || !pair_of(a[5], g.bo) || g.bs.v[0] <= 0 || g.bs.v[1] <= 0)
        return false;
    g.transpose = PyObject_IsTrue(a[6]);
    return g.transpose >= 0;
}

at::Tensor run_gather(const Gather& g, const at::Tensor* out)
{
    const Blocks& b = g.b;
    c10::DeviceGuard guard(g.x->device());
    at::Tensor y = out ? *out : empty_stack(b.M, g.x->size(3), g.bs, g.transpose, *g.x);
    const float* const xp = static_cast<const float*>(g.x->data_ptr());
    const int16_t* const ip = static_cast<const int16_t*>(b.idx->data_ptr());
    float* const yp = static_cast<float*>(y.data_ptr());
    const int64_t* const dims = g.x->sizes().data();
    void* const stream = stream_of(*g.x);
    run([&] {
        return b.count ? sbnet_sparse_gather_device_count(xp, dims, 4, b.count, b.M, ip, g.bs.v, 2, g.bt.v, 2, g.bo.v, 2,
                                                          g.transpose, yp, stream)
                       : sbnet_sparse_gather(xp, dims, 4, b.M, ip, g.bs.v, 2, g.bt.v, 2, g.bo.v, 2, g.transpose, yp, stream);
    });
    return y;
}

// gather(x, bin_counts, active_block_indices, bsize, bstride, boffset, transpose, out) -> stack
PyObject* gather(PyObject* const* a)
{
    Gather g;
    if (!gather_of(a, g)) {
        if (PyErr_Occurred()) return nullptr;
        Py_RETURN_NONE;
    }
    const at::Tensor* out = nullptr;
    if (a[7] != Py_None) {
        out = dev_f32(a[7]);
        if (!out || out->device() != g.x->device() || !is_stack(*out, g.b.M, g.x->size(3), g.bs, g.transpose)) Py_RETURN_NONE;
    }
    return THPVariable_Wrap(run_gather(g, out));
}

at::Tensor run_gather_grad(const at::Tensor& g, const at::Tensor& idx, int32_t M, const int64_t* dims, const Pair& bs, const Pair& bt,
                           const Pair& bo, int transpose)
{
    c10::DeviceGuard guard(g.device());
    at::Tensor dx = empty_f32({dims[0], dims[1], dims[2], dims[3]}, g);
    const int64_t need = (int64_t)sbnet_sparse_scatter_workspace_bytes(M, dims, 4, bs.v, 2, bt.v, 2, bo.v, 2);
    const Workspace scratch = need ? workspace(g.device(), need) : Workspace();
    const at::Tensor& ws = scratch.buffer;
    const float* const gp = static_cast<const float*>(g.data_ptr());
    const int16_t* const ip = static_cast<const int16_t*>(idx.data_ptr());
    float* const dp = static_cast<float*>(dx.data_ptr());
    void* const stream = stream_of(g);
    run([&] {
        return sbnet_sparse_gather_grad(gp, M, ip, dp, dims, 4, bs.v, 2, bt.v, 2, bo.v, 2, transpose,
                                        need ? ws.data_ptr() : nullptr, need ? (size_t)ws.numel() : 0, stream);
    }, scratch.busy);
    return dx;
}

// gather_grad(grad, bin_counts, active_block_indices, x_shape, bsize, bstride, boffset, transpose) -> dx
PyObject* gather_grad(PyObject* const* a)
{
    const at::Tensor* g = dev_f32(a[0]);
    Blocks b;
    Pair bs, bt, bo;
    if (!g || !blocks_of(a[1], a[2], b) || b.count || b.idx->device() != g->device() || !PyTuple_Check(a[3]) ||
        PyTuple_GET_SIZE(a[3]) != 4 || !pair_of(a[4], bs) || !pair_of(a[5], bt) || !pair_of(a[6], bo))
        Py_RETURN_NONE;
    int64_t dims[4];
    for (int i = 0; i < 4; ++i) {
        int32_t d;
        if (!int_of(PyTuple_GET_ITEM(a[3], i), &d) || d <= 0) Py_RETURN_NONE;
        dims[i] = d;
    }
    const int transpose = PyObject_IsTrue(a[7]);
    if (transpose < 0) return nullptr;
    if (!is_stack(*g, b.M, dims[3], bs, transpose)) Py_RETURN_NONE;
    return THPVariable_Wrap(run_gather_grad(*g, *b.idx, b.M, dims, bs, bt, bo, transpose));
}

struct Scatter {
    const at::Tensor *x, *base;
    Blocks b;
    Pair bs, bt, bo;
    int add, atomic, transpose;
};

// x, bin_counts, active_block_indices, ybase, bsize, bstride, boffset, add, atomic, transpose
bool scatter_of(PyObject* const* a, Scatter& q)
{
    q.x = dev_f32(a[0]);
    q.base = dev_f32(a[3]);
    if (!q.x || !q.base || q.base->dim() != 4 || !blocks_of(a[1], a[2], q.b) || q.b.idx->device() != q.base->device() ||
        q.x->device() != q.base->device() || !pair_of(a[4], q.bs) || !pair_of(a[5], q.bt) || !pair_of(a[6], q.bo))
        return false;
    q.add = PyObject_IsTrue(a[7]);
    q.atomic = PyObject_IsTrue(a[8]);
    q.transpose = PyObject_IsTrue(a[9]);
    if (q.add < 0 || q.atomic < 0 || q.transpose < 0) return false;
    if (q.b.count && q.x->dim() > 0 && q.x->size(0) < q.b.M) q.b.M = (int32_t)q.x->size(0);
    return is_stack(*q.x, q.b.M, q.base->size(3), q.bs, q.transpose);
}

at::Tensor run_scatter(const Scatter& q, bool in_place)
{
    const Blocks& b = q.b;
    const Pair &bs = q.bs, &bt = q.bt, &bo = q.bo;
    const bool overlap = bt.v[0] < bs.v[0] || bt.v[1] < bs.v[1];
    c10::DeviceGuard guard(q.base->device());
    const int64_t* const dims = q.base->sizes().data();
    const bool wants = (q.add && q.atomic) || !in_place || (!q.add && overlap);
    const int64_t need = wants ? (int64_t)sbnet_sparse_scatter_workspace_bytes(b.M, dims, 4, bs.v, 2, bt.v, 2, bo.v, 2) : 0;
    const Workspace scratch = need ? workspace(q.base->device(), need) : Workspace();
    const at::Tensor& ws = scratch.buffer;
    void* const wp = need ? ws.data_ptr() : nullptr;
    const size_t wn = need ? (size_t)ws.numel() : 0;
    at::Tensor y = in_place ? *q.base : empty_f32(q.base->sizes(), *q.base);
    const float *const xp = static_cast<const float*>(q.x->data_ptr()), *const bp = static_cast<const float*>(q.base->data_ptr());
    const int16_t* const ip = static_cast<const int16_t*>(b.idx->data_ptr());
    float* const yp = static_cast<float*>(y.data_ptr());
    void* const stream = stream_of(*q.base);
    run([&] {
        if (in_place)
            return b.count ? sbnet_sparse_scatter_var_device_count(xp, b.count, b.M, ip, yp, dims, 4, bs.v, 2, bt.v, 2,
                                                                   bo.v, 2, q.add, q.atomic, q.transpose, wp, wn, stream)
                           : sbnet_sparse_scatter_var(xp, b.M, ip, yp, dims, 4, bs.v, 2, bt.v, 2, bo.v, 2, q.add, q.atomic,
                                                      q.transpose, wp, wn, stream);
        return b.count ? sbnet_sparse_scatter_device_count(xp, b.count, b.M, ip, bp, dims, 4, bs.v, 2, bt.v, 2, bo.v, 2,
                                                           q.add, q.atomic, q.transpose, yp, wp, wn, stream)
                       : sbnet_sparse_scatter(xp, b.M, ip, bp, dims, 4, bs.v, 2, bt.v, 2, bo.v, 2, q.add, q.atomic,
                                              q.transpose, yp, wp, wn, stream);
    }, scratch.busy);
    return y;
}

// scatter(x, bin_counts, active_block_indices, ybase, bsize, bstride, boffset, add, atomic, transpose, use_var) -> y
PyObject* scatter(PyObject* const* a)
{
    Scatter q;
    if (!scatter_of(a, q)) {
        if (PyErr_Occurred()) return nullptr;
        Py_RETURN_NONE;
    }
    const int in_place = PyObject_IsTrue(a[10]);
    if (in_place < 0) return nullptr;
    at::Tensor y = run_scatter(q, in_place);
    if (in_place) {
        Py_INCREF(a[3]);   // the caller's own tensor object, as the Python wrapper returns it
        return a[3];
    }
    return THPVariable_Wrap(std::move(y));
}

// The gradient of the base of plain writes; an undefined tensor for a geometry that the one pass does not take.
at::Tensor run_base_grad(const at::Tensor& g, const at::Tensor& idx, int32_t M, const Pair& bs, const Pair& bt, const Pair& bo)
{
    if (reinterpret_cast<uintptr_t>(g.data_ptr()) & 15) return at::Tensor();
    const int64_t* const dims = g.sizes().data();
    const size_t need = sbnet_sparse_scatter_base_grad_workspace_bytes(M, dims, bs.v, bt.v, bo.v);
    if (!need) return at::Tensor();
    c10::DeviceGuard guard(g.device());
    at::Tensor d = empty_f32(g.sizes(), g);
    at::Tensor ws = own_scratch(g, need);
    const float* const gp = static_cast<const float*>(g.data_ptr());
    const int16_t* const ip = static_cast<const int16_t*>(idx.data_ptr());
    float* const dp = static_cast<float*>(d.data_ptr());
    void *const wp = ws.data_ptr(), *const stream = stream_of(g);
    run([&] { return sbnet_sparse_scatter_base_grad(gp, M, ip, dp, dims, bs.v, bt.v, bo.v, wp, need, stream); });
    return d;
}

// scatter_base_grad(grad, bin_counts, active_block_indices, bsize, bstride, boffset) -> gradient of the base of plain writes
PyObject* scatter_base_grad(PyObject* const* a)
{
    const at::Tensor* g = dev_f32(a[0]);
    Blocks b;
    Pair bs, bt, bo;
    if (!g || g->dim() != 4 || !blocks_of(a[1], a[2], b) || b.count || b.idx->device() != g->device() || !pair_of(a[3], bs) ||
        !pair_of(a[4], bt) || !pair_of(a[5], bo))
        Py_RETURN_NONE;
    at::Tensor d = run_base_grad(*g, *b.idx, b.M, bs, bt, bo);
    if (!d.defined()) Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(d));
}

// Contiguous, on the GPU, float32, with no gradient asked for, and not under autocast, where the layers' convolutions
// would compute in another type.
const at::Tensor* plain_f32(PyObject* o)
{
    const at::Tensor* t = dev_f32(o);
    return t && !at::autocast::is_autocast_enabled(at::kCUDA) && !(t->requires_grad() && at::GradMode::is_enabled()) ? t : nullptr;
}

constexpr int64_t CONV_MOST = 1ll << 28, ROWS_MOST = 1ll << 28;   // elements, output pixels: inside what the kernels take

// Kernel dimensions as int32, false where an input of C channels and R x S pixels does not take it.
bool kernel_of(const at::Tensor& w, int64_t C, int64_t R, int64_t S, int32_t* dims)
{
    if (w.dim() != 4 || w.size(2) != C || C > 4096 || w.size(0) > R || w.size(1) > S || w.numel() <= 0 || w.numel() >= CONV_MOST) return false;
    for (int i = 0; i < 4; ++i) dims[i] = (int32_t)w.size(i);
    return true;
}

bool positive(const Pair& p) { return p.v[0] > 0 && p.v[1] > 0; }

// Whether a convolution of `rows` output pixels is left to the library as the faster way (MI355X; us for library / own, the
// layer in place on planar stacks, 17x17 and 24x24 blocks).
bool library_is_faster(const int32_t* w, int64_t rows, bool aligned)
{
    const int64_t k = (int64_t)w[0] * w[1] * w[2], K = w[3];
    if (aligned && w[2] % 4 == 0 && K % 4 == 0) {
        // 3x3: the library's transforms save multiplications, which pays for many pixels of many channels.  128 channels:
        // 66 / 61 at 4 GFLOP, 386 / 358 at 32, 691 / 764 at 69, 1391 / 1512 at 137; 256: 368 / 354, 676 / 680 at 64,
        // 2635 / 2904 at 276; 512: 362 / 390 at 32, 1368 / 1476 at 129, 9874 / 12969 at 1105.  With 80 channels or fewer the
        // two meet without crossing (406 / 415 with 64 at 34).  1x1 and 5x5 products of any size go either way with the
        // block count (1x1, 512 channels: 644 / 570, 1284 / 1294; 5x5, 256: 592 / 681, 1790 / 1407, 2169 / 2560).
        return w[0] == 3 && w[1] == 3 && w[2] > 80 && 2.0 * rows * k * K > 64e9;
    }
    // Single-float loads, at a third of the rate: only small products, in steps of 16 k times 16 channels.  30 channels,
    // 3x3: 39 / 34 at 1.8 M steps, 53 / 55 at 3.7, 144 / 196 at 16; 50: 33 / 30 at 1.7, 46 / 51 at 3.2; 130: 64 / 65 at 4.5,
    // 89 / 134 at 9.6.  Channels that fill no fragment read as many pixels for less: 3 channels, 3x3: 36 / 33 at 0.5,
    // 57 / 56 at 0.9 (44 / 56 on NHWC stacks); 7x7: 50 / 38 at 0.9, 83 / 99 at 3.3.
    return rows * ((k + 15) / 16) * ((K + 15) / 16) > (K < 16 ? 900000 : 2500000);
}

// block_conv(x, w, bin_counts, active_block_indices, bsize, bstride, boffset) -> NHWC stack
PyObject* block_conv(PyObject* const* a)
{
    const at::Tensor *x = plain_f32(a[0]), *w = plain_f32(a[1]);
    Blocks b;
    Pair bs, bt, bo;
    int32_t wd[4];
    if (!x || !w || x->dim() != 4 || x->numel() <= 0 || x->numel() >= 2 * CONV_MOST || w->device() != x->device() ||
        !blocks_of(a[2], a[3], b) || b.idx->device() != x->device() || !pair_of(a[4], bs) || !pair_of(a[5], bt) ||
        !pair_of(a[6], bo) || !positive(bs) || !positive(bt) || !kernel_of(*w, x->size(3), bs.v[0], bs.v[1], wd))
        Py_RETURN_NONE;
    const int64_t R = bs.v[0] - wd[0] + 1, S = bs.v[1] - wd[1] + 1;
    if (R * S >= ROWS_MOST || b.M * R * S >= ROWS_MOST || b.M * R * S * wd[3] >= 2 * CONV_MOST) Py_RETURN_NONE;
    // (of a count on the device only the capacity is known, which the library would compute in full)
    if (!b.count && library_is_faster(wd, b.M * R * S, (reinterpret_cast<uintptr_t>(x->const_data_ptr()) & 15) == 0)) Py_RETURN_NONE;
    c10::DeviceGuard guard(x->device());
    at::Tensor q = empty_f32({b.M, R, S, wd[3]}, *x);
    const float *const xp = static_cast<const float*>(x->data_ptr()), *const kp = static_cast<const float*>(w->data_ptr());
    const int16_t* const ip = static_cast<const int16_t*>(b.idx->data_ptr());
    float* const qp = static_cast<float*>(q.data_ptr());
    const int64_t* const dims = x->sizes().data();
    void* const stream = stream_of(*x);
    if (b.M && !call([&] { return sbnet_block_conv(xp, dims, b.M, b.count, ip, bs.v, bt.v, bo.v, kp, wd, qp, stream); }))
        return nullptr;
    return THPVariable_Wrap(std::move(q));
}

// block_bottleneck(x, [w1, w2, w3], [gamma, beta, mean, var] * 3, bin_counts, active_block_indices, bsize, bstride,
//                  boffset, out_stride, eps, no_activation, in_place) -> NHWC stack, or x with the result added; with
// no_activation the first four are not looked at
PyObject* block_bottleneck(PyObject* const* a)
{
    const at::Tensor* x = plain_f32(a[0]);
    Blocks b;
    Pair bs, bt, bo, os;
    if (!x || x->dim() != 4 || x->numel() <= 0 || x->numel() >= 2 * CONV_MOST || !PyList_CheckExact(a[1]) ||
        PyList_GET_SIZE(a[1]) != 3 || !PyList_CheckExact(a[2]) || PyList_GET_SIZE(a[2]) != 12 || !blocks_of(a[3], a[4], b) ||
        b.idx->device() != x->device() || !pair_of(a[5], bs) || !pair_of(a[6], bt) || !pair_of(a[7], bo) ||
        !pair_of(a[8], os) || !positive(bs) || !positive(bt) || !PyFloat_CheckExact(a[9]))
        Py_RETURN_NONE;
    const int no_activation = PyObject_IsTrue(a[10]), in_place = PyObject_IsTrue(a[11]);
    if (no_activation < 0 || in_place < 0) return nullptr;
    const float *weights[3], *norms[12];
    int32_t wd[12];
    int64_t R = bs.v[0], S = bs.v[1], C = x->size(3);
    for (int i = 0; i < 3; ++i) {
        const at::Tensor* w = plain_f32(PyList_GET_ITEM(a[1], i));
        if (!w || w->device() != x->device() || !kernel_of(*w, C, R, S, wd + 4 * i)) Py_RETURN_NONE;
        weights[i] = static_cast<const float*>(w->data_ptr());
        for (int j = 0; j < 4; ++j) {
            norms[4 * i + j] = nullptr;
            if (i == 0 && no_activation) continue;
            const at::Tensor* t = plain_f32(PyList_GET_ITEM(a[2], 4 * i + j));
            if (!t || t->device() != x->device() || t->numel() != C) Py_RETURN_NONE;
            norms[4 * i + j] = static_cast<const float*>(t->data_ptr());
        }
        R -= wd[4 * i] - 1;
        S -= wd[4 * i + 1] - 1;
        C = wd[4 * i + 3];
        if (R * S >= ROWS_MOST || b.M * R * S >= ROWS_MOST || b.M * R * S * C >= 2 * CONV_MOST) Py_RETURN_NONE;
    }
    if (in_place && (C != x->size(3) || os.v[0] != R || os.v[1] != S)) Py_RETURN_NONE;
    c10::DeviceGuard guard(x->device());
    at::Tensor q = in_place ? *x : empty_f32({b.M, R, S, C}, *x);
    at::Tensor ws = own_scratch(*x, sbnet_block_bottleneck_workspace_bytes(b.M, bs.v, wd));
    const float* const xp = static_cast<const float*>(x->data_ptr());
    const int16_t* const ip = static_cast<const int16_t*>(b.idx->data_ptr());
    float* const qp = static_cast<float*>(q.data_ptr());
    const int64_t* const dims = x->sizes().data();
    const float eps = (float)PyFloat_AS_DOUBLE(a[9]);
    void* const stream = stream_of(*x);
    if (b.M && !call([&] {
            return sbnet_block_bottleneck(xp, dims, b.M, b.count, ip, bs.v, bt.v, bo.v, weights, wd, norms, eps,
                                          in_place ? nullptr : qp, in_place ? qp : nullptr, os.v, ws.data_ptr(),
                                          (size_t)ws.numel(), stream);
        }))
        return nullptr;
    if (in_place) {
        Py_INCREF(a[0]);
        return a[0];
    }
    return THPVariable_Wrap(std::move(q));
}

// The gradients of a residual function on planar stacks: dp, dw1-3, (dgamma, dbeta)1-3, undefined what is not wanted.  saved:
// [z, act, mean, inv, kernel [K,C,kh,kw], gamma] * 3.  False where the kernels do not take the sizes.
bool run_bottleneck_grad(const at::Tensor* dq, const at::Tensor* const* t, const bool* wanted, at::Tensor* res)
{
    const float* ptr[6][3];
    for (int i = 0; i < 18; ++i) {
        if (!t[i] || t[i]->device() != dq->device()) return false;
        ptr[i % 6][i / 6] = static_cast<const float*>(t[i]->data_ptr());
    }
    if (t[0]->dim() != 4 || t[0]->size(0) > INT32_MAX) return false;
    const int64_t M = t[0]->size(0);
    int64_t C = t[0]->size(1), R = t[0]->size(2), S = t[0]->size(3);
    if (M <= 0 || C <= 0 || R <= 0 || S <= 0 || R > INT32_MAX || S > INT32_MAX) return false;
    const int32_t bs[2] = {(int32_t)R, (int32_t)S};
    int32_t wd[12];
    for (int i = 0; i < 3; ++i) {
        const at::Tensor* const* q = t + 6 * i;
        const at::Tensor* w = q[4];
        if (q[0]->dim() != 4 || q[0]->sizes() != at::IntArrayRef({M, C, R, S}) || q[1]->sizes() != q[0]->sizes() ||
            q[0]->numel() >= 2 * CONV_MOST || q[2]->numel() != C || q[3]->numel() != C || q[5]->numel() != C || w->dim() != 4 ||
            w->size(1) != C || w->size(2) > R || w->size(3) > S || w->numel() <= 0 || w->numel() >= CONV_MOST)
            return false;
        wd[4 * i] = (int32_t)w->size(2);
        wd[4 * i + 1] = (int32_t)w->size(3);
        wd[4 * i + 2] = (int32_t)C;
        wd[4 * i + 3] = (int32_t)w->size(0);
        R -= w->size(2) - 1;
        S -= w->size(3) - 1;
        C = w->size(0);
    }
    if (dq->sizes() != at::IntArrayRef({M, C, R, S}) || dq->numel() >= 2 * CONV_MOST) return false;
    const size_t need = sbnet_bottleneck_grad_workspace_bytes((int32_t)M, bs, wd);
    if (!need) return false;
    c10::DeviceGuard guard(dq->device());
    float *out[10];
    if (wanted[0]) res[0] = empty_f32(t[0]->sizes(), *dq);
    for (int i = 0; i < 3; ++i) {
        const int32_t* d = wd + 4 * i;
        if (wanted[1 + i]) res[1 + i] = empty_f32({d[0], d[1], d[2], d[3]}, *dq);
        if (wanted[4 + 2 * i]) res[4 + 2 * i] = empty_f32({d[2]}, *dq);
        if (wanted[5 + 2 * i]) res[5 + 2 * i] = empty_f32({d[2]}, *dq);
    }
    for (int i = 0; i < 10; ++i) out[i] = wanted[i] ? static_cast<float*>(res[i].data_ptr()) : nullptr;
    float *const dgamma[3] = {out[4], out[6], out[8]}, *const dbeta[3] = {out[5], out[7], out[9]};
    at::Tensor ws = own_scratch(*dq, need);
    const float* const dqp = static_cast<const float*>(dq->data_ptr());
    void *const wp = ws.data_ptr(), *const stream = stream_of(*dq);
    run([&] {
        return sbnet_bottleneck_grad(dqp, (int32_t)M, bs, ptr[0], ptr[1], ptr[2], ptr[3], ptr[5], ptr[4], wd, out[0],
                                     out + 1, dgamma, dbeta, wp, need, stream);
    });
    return true;
}

PyObject* or_none(at::Tensor&& t)
{
    if (t.defined()) return THPVariable_Wrap(std::move(t));
    Py_RETURN_NONE;
}

// bottleneck_grad(dq, [z, act, mean, inv, kernel [K,C,kh,kw], gamma] * 3, wanted) -> (dp, dw1, dw2, dw3, dgamma1, dbeta1,
// ...), on planar stacks, or None where the kernels do not take the sizes.  wanted: a tuple with the truth of each of the
// ten, those not wanted are None; all where it is missing.
PyObject* bottleneck_grad(PyObject* const* a)
{
    const at::Tensor* dq = dev_f32(a[0]);
    if (!dq || dq->dim() != 4 || !PyList_CheckExact(a[1]) || PyList_GET_SIZE(a[1]) != 18) Py_RETURN_NONE;
    bool wanted[10];
    if (a[2] != Py_None && (!PyTuple_CheckExact(a[2]) || PyTuple_GET_SIZE(a[2]) != 10)) Py_RETURN_NONE;
    for (int i = 0; i < 10; ++i) wanted[i] = a[2] == Py_None || PyTuple_GET_ITEM(a[2], i) == Py_True;
    const at::Tensor* t[18];
    for (int i = 0; i < 18; ++i) t[i] = dev_f32(PyList_GET_ITEM(a[1], i));
    at::Tensor res[10];
    if (!run_bottleneck_grad(dq, t, wanted, res)) Py_RETURN_NONE;
    PyObject* r = PyTuple_New(10);
    if (!r) return nullptr;
    for (int i = 0; i < 10; ++i) PyTuple_SET_ITEM(r, i, or_none(std::move(res[i])));
    return r;
}

// ---- the differentiable ops -------------------------------------------------------------------------------
//
// torch::autograd functions of the same steps as the ones in autograd.py and sparse_conv.py, for plain tensors: an autograd
// function in Python costs about 35 us of host time a call forward and 10-15 backward, and these steps are bound by that
// wherever the tensors are not large (a training step of a residual block spent 490 us in the host for 260 on the GPU).
// What looks on or transforms (dispatch and functorch modes, forward-mode tangents, tracing) is left to those.

using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// A backward pass's hold of the interpreter, which guards the scratch table and takes the errors.
struct Gil {
    PyGILState_STATE state = PyGILState_Ensure();
    ~Gil() { PyGILState_Release(state); }
};

// Whether a backward pass may hand the list it saved to the kernels beside a gradient: what comes back from a saved-tensor
// hook is whatever the hook made, and a gradient may be a transform's (a batch of them).  Anything else, and anything
// while modes look on, goes to the general wrappers, which convert, check and raise.
bool plain_list(const at::Tensor& idx, int32_t M, const at::Tensor& grad)
{
    return !c10::impl::TorchDispatchModeTLS::any_modes_set() && is_dev(idx, at::kShort) && is_list(idx) && M <= idx.size(0) &&
           is_dev(grad, at::kFloat) && grad.dim() == 4 && idx.device() == grad.device();
}

PyObject* tuple_of(at::IntArrayRef v)
{
    PyObject* t = PyTuple_New((Py_ssize_t)v.size());
    if (!t) raise_pending();
    for (size_t i = 0; i < v.size(); ++i) {
        PyObject* const o = PyLong_FromLongLong(v[i]);
        if (!o) {
            Py_DECREF(t);
            raise_pending();
        }
        PyTuple_SET_ITEM(t, (Py_ssize_t)i, o);
    }
    return t;
}

// Sizes that a function keeps: one entry of its context.
std::vector<int64_t> sizes_of(int32_t M, const Pair& bs, const Pair& bt, const Pair& bo, const at::Tensor& t, int flags)
{
    return {M, bs.v[0], bs.v[1], bt.v[0], bt.v[1], bo.v[0], bo.v[1], t.size(0), t.size(1), t.size(2), t.size(3), flags};
}

Pair pair_at(const std::vector<int64_t>& v, int i) { return {{(int32_t)v[i], (int32_t)v[i + 1]}}; }

struct GatherFunction : torch::autograd::Function<GatherFunction> {
    static at::Tensor forward(AutogradContext* ctx, const at::Tensor& x, const Gather* g)
    {
        ctx->save_for_backward({*g->b.idx});
        ctx->saved_data["sizes"] = sizes_of(g->b.M, g->bs, g->bt, g->bo, x, g->transpose);
        return run_gather(*g, nullptr);
    }

    static variable_list backward(AutogradContext* ctx, variable_list grads)
    {
        const Gil gil;
        const at::Tensor idx = ctx->get_saved_variables()[0], g = grads[0].contiguous();
        const std::vector<int64_t> v = ctx->saved_data["sizes"].toIntVector();
        const int32_t M = (int32_t)v[0];
        const Pair bs = pair_at(v, 1);
        if (plain_list(idx, M, g) && is_stack(g, M, v[10], bs, v[11]))
            return {run_gather_grad(g, idx, M, v.data() + 7, bs, pair_at(v, 3), pair_at(v, 5), (int)v[11]), at::Tensor()};
        THPObjectPtr grad(THPVariable_Wrap(g)), list(THPVariable_Wrap(idx)), sizes(tuple_of(v));
        if (!grad || !list) raise_pending();
        THPObjectPtr got(PyObject_CallFunctionObjArgs(g_gather_gradient, grad.get(), list.get(), sizes.get(), nullptr));
        if (!got) raise_pending();
        TORCH_CHECK(THPVariable_Check(got.get()), "a gradient");
        return {THPVariable_Unpack(got.get()), at::Tensor()};
    }
};

struct ScatterFunction : torch::autograd::Function<ScatterFunction> {
    static at::Tensor forward(AutogradContext* ctx, const at::Tensor& x, const at::Tensor& base, const Scatter* q)
    {
        ctx->save_for_backward({*q->b.idx});
        std::vector<int64_t> v = sizes_of(q->b.M, q->bs, q->bt, q->bo, base, q->transpose | q->add << 1);
        v.push_back(x.size(0));
        ctx->saved_data["sizes"] = std::move(v);
        return run_scatter(*q, false);
    }

    static variable_list backward(AutogradContext* ctx, variable_list grads)
    {
        const Gil gil;
        const at::Tensor idx = ctx->get_saved_variables()[0], grad = grads[0].contiguous();
        const std::vector<int64_t> v = ctx->saved_data["sizes"].toIntVector();
        const int32_t M = (int32_t)v[0];
        const Pair bs = pair_at(v, 1), bt = pair_at(v, 3), bo = pair_at(v, 5);
        const bool transpose = v[11] & 1, add = v[11] & 2;
        variable_list out(3);
        bool todo[2] = {ctx->needs_input_grad(0), ctx->needs_input_grad(1)};   // of the blocks, of the base
        if (plain_list(idx, M, grad) && grad.sizes() == at::IntArrayRef(v.data() + 7, 4)) {
            if (todo[0]) out[0] = run_gather({&grad, {&idx, M, nullptr}, bs, bt, bo, transpose}, nullptr);
            if (todo[1] && add) out[1] = grad;
            else if (todo[1] && !(at::GradMode::is_enabled() && grad.requires_grad())) out[1] = run_base_grad(grad, idx, M, bs, bt, bo);
            for (int i = 0; i < 2; ++i) todo[i] = todo[i] && !out[i].defined();
        }
        if (!todo[0] && !todo[1]) return out;
        // besides: a graph of the gradients is asked for, or a geometry that the one pass does not take
        THPObjectPtr g(THPVariable_Wrap(grad)), list(THPVariable_Wrap(idx)), sizes(tuple_of(v));
        if (!g || !list) raise_pending();
        THPObjectPtr got(PyObject_CallFunctionObjArgs(g_scatter_gradients, g.get(), list.get(), sizes.get(), todo[0] ? Py_True : Py_False,
                                                      todo[1] ? Py_True : Py_False, nullptr));
        if (!got) raise_pending();
        TORCH_CHECK(PyTuple_CheckExact(got.get()) && PyTuple_GET_SIZE(got.get()) == 2, "gradients of two inputs");
        for (int i = 0; i < 2; ++i) {
            PyObject* const o = PyTuple_GET_ITEM(got.get(), i);
            if (o != Py_None) out[i] = THPVariable_Unpack(o);
        }
        return out;
    }
};

// Nobody transforms or looks on at what torch does.
bool plain_autograd()
{
    return !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode);
}

// gather_autograd(x, bin_counts, active_block_indices, bsize, bstride, boffset, transpose) -> stack with a gradient
PyObject* gather_autograd(PyObject* const* a)
{
    Gather g;
    if (!plain_autograd() || !gather_of(a, g) || g.b.count) {
        if (PyErr_Occurred()) return nullptr;
        Py_RETURN_NONE;
    }
    return THPVariable_Wrap(GatherFunction::apply(*g.x, (const Gather*)&g));
}

// scatter_autograd(x, bin_counts, active_block_indices, ybase, bsize, bstride, boffset, add, atomic, transpose) -> y
PyObject* scatter_autograd(PyObject* const* a)
{
    Scatter q;
    if (!plain_autograd() || !scatter_of(a, q) || q.b.count) {
        if (PyErr_Occurred()) return nullptr;
        Py_RETURN_NONE;
    }
    return THPVariable_Wrap(ScatterFunction::apply(*q.x, *q.base, (const Scatter*)&q));
}

// A residual function's running statistics and the batch norms' numbers.
struct Residual {
    at::Tensor mean[3], var[3];   // undefined: none
    double momentum, eps;
};

// The status of a call that is made without the interpreter.
void checked(int status)
{
    TORCH_CHECK(status == SBNET_OK, sbnet_status_string(status), " (hipError_t ", sbnet_last_hip_error(), ")");
}

// Kernels [kh,kw,C,K] as the library takes them, [K,C,kh,kw].
void kernels_of(const at::Tensor* const* w, at::Tensor* out)
{
    const float* from[3];
    float* to[3];
    int32_t dims[12];
    bool own = true;
    for (int i = 0; i < 3; ++i) {
        own = own && w[i]->numel() > 0 && w[i]->numel() < CONV_MOST && w[i]->device() == w[0]->device();
        for (int j = 0; j < 4 && own; ++j) dims[4 * i + j] = (int32_t)w[i]->size(j);
    }
    if (!own) {
        for (int i = 0; i < 3; ++i) out[i] = w[i]->permute({3, 2, 0, 1}).contiguous();
        return;
    }
    c10::DeviceGuard guard(w[0]->device());
    for (int i = 0; i < 3; ++i) {
        out[i] = empty_f32({dims[4 * i + 3], dims[4 * i + 2], dims[4 * i], dims[4 * i + 1]}, *w[0]);
        from[i] = static_cast<const float*>(w[i]->const_data_ptr());
        to[i] = static_cast<float*>(out[i].data_ptr());
    }
    checked(sbnet_kernels_oihw(from, dims, to, 3, stream_of(*w[0])));
}

void relu(at::Tensor& t)
{
    if (!t.is_contiguous() || (reinterpret_cast<uintptr_t>(t.const_data_ptr()) & 15)) {
        t.relu_();
        return;
    }
    c10::DeviceGuard guard(t.device());
    checked(sbnet_relu(static_cast<float*>(t.data_ptr()), t.numel(), stream_of(t)));
}

struct ResidualFunction : torch::autograd::Function<ResidualFunction> {
    // The library's calls, one by one, as the layers make them.
    static at::Tensor forward(AutogradContext* ctx, const at::Tensor& p, const at::Tensor& w1, const at::Tensor& g1, const at::Tensor& b1,
                              const at::Tensor& w2, const at::Tensor& g2, const at::Tensor& b2, const at::Tensor& w3,
                              const at::Tensor& g3, const at::Tensor& b3, const Residual* r)
    {
        const at::Tensor *const w[3] = {&w1, &w2, &w3}, *const gamma[3] = {&g1, &g2, &g3}, *const beta[3] = {&b1, &b2, &b3};
        at::Tensor z = p, kernels[3];
        kernels_of(w, kernels);
        variable_list saved;
        for (int i = 0; i < 3; ++i) {
            auto bn = at::_batch_norm_impl_index(z, *gamma[i], *beta[i], r->mean[i], r->var[i], true, r->momentum, r->eps,
                                                 at::globalContext().userEnabledCuDNN());
            at::Tensor& act = std::get<0>(bn);
            relu(act);
            saved.insert(saved.end(), {z, act, std::get<1>(bn), std::get<2>(bn), kernels[i], *gamma[i]});
            z = at::conv2d(act, kernels[i], {}, at::IntArrayRef({1, 1}));
        }
        ctx->save_for_backward(std::move(saved));
        ctx->saved_data["layers"] = std::vector<at::Tensor>{w1, b1, w2, b2, w3, b3};   // for a graph of the gradients alone
        return z;
    }

    static variable_list backward(AutogradContext* ctx, variable_list grads)
    {
        const Gil gil;
        const variable_list saved = ctx->get_saved_variables();
        // of p and, per layer, kernel, gamma and beta, as the inputs are; the kernels' gradients stand first in what comes back
        bool needs[10], wanted[10];
        for (int i = 0; i < 10; ++i) needs[i] = ctx->needs_input_grad(i);
        constexpr int AT[10] = {0, 1, 4, 5, 2, 6, 7, 3, 8, 9};   // where input i's gradient is
        for (int i = 0; i < 10; ++i) wanted[AT[i]] = needs[i];
        variable_list out(11);
        const bool graph = at::GradMode::is_enabled();
        if (!graph) {
            const at::Tensor dq = grads[0].contiguous();
            const at::Tensor* t[18];
            bool plain = !c10::impl::TorchDispatchModeTLS::any_modes_set() && is_dev(dq, at::kFloat) && dq.dim() == 4;
            for (int i = 0; i < 18; ++i) {
                t[i] = &saved[i];
                plain = plain && is_dev(saved[i], at::kFloat);
            }
            at::Tensor res[10];
            if (plain && run_bottleneck_grad(&dq, t, wanted, res)) {
                for (int i = 0; i < 10; ++i) out[i] = res[AT[i]];
                return out;
            }
        }
        // a graph of the gradients is asked for, or sizes that the kernels do not take: through the layers one by one
        const std::vector<at::Tensor> layers = ctx->saved_data["layers"].toTensorVector();
        THPObjectPtr list(PyList_New(18)), pairs(PyList_New(6)), need(PyTuple_New(10)), dq(THPVariable_Wrap(grads[0]));
        if (!list || !pairs || !need || !dq) raise_pending();
        for (int i = 0; i < 18; ++i) PyList_SET_ITEM(list.get(), i, THPVariable_Wrap(saved[i]));
        for (int i = 0; i < 6; ++i) PyList_SET_ITEM(pairs.get(), i, THPVariable_Wrap(layers[i]));
        for (int i = 0; i < 10; ++i) PyTuple_SET_ITEM(need.get(), i, PyBool_FromLong(needs[i]));
        THPObjectPtr got(PyObject_CallFunctionObjArgs(g_by_layers, list.get(), pairs.get(), need.get(), dq.get(), graph ? Py_True : Py_False, nullptr));
        if (!got) raise_pending();
        TORCH_CHECK(PyList_CheckExact(got.get()) && PyList_GET_SIZE(got.get()) == 10, "gradients of ten inputs");
        for (int i = 0; i < 10; ++i) {
            PyObject* const o = PyList_GET_ITEM(got.get(), i);
            if (o != Py_None) out[i] = THPVariable_Unpack(o);
        }
        return out;
    }
};

// residual(p, [moving mean, moving variance] * 3, [kernel, gamma, beta] * 3, momentum, eps) -> the residual function of a planar
// stack with batch statistics, with own gradients
PyObject* residual(PyObject* const* a)
{
    const at::Tensor* p = dev_f32(a[0]);
    if (!plain_autograd() || !p || p->dim() != 4 || !PyList_CheckExact(a[1]) || PyList_GET_SIZE(a[1]) != 6 || !PyList_CheckExact(a[2]) ||
        PyList_GET_SIZE(a[2]) != 9 || !PyFloat_CheckExact(a[3]) || !PyFloat_CheckExact(a[4]))
        Py_RETURN_NONE;
    Residual r;
    r.momentum = PyFloat_AS_DOUBLE(a[3]);
    r.eps = PyFloat_AS_DOUBLE(a[4]);
    for (int i = 0; i < 6; ++i) {
        PyObject* const o = PyList_GET_ITEM(a[1], i);
        if (o == Py_None) continue;
        const at::Tensor* t = dev_f32(o);
        if (!t) Py_RETURN_NONE;
        (i & 1 ? r.var : r.mean)[i / 2] = *t;
    }
    const at::Tensor* t[9];
    for (int i = 0; i < 9; ++i) {
        t[i] = dev_f32(PyList_GET_ITEM(a[2], i));
        if (!t[i] || t[i]->dim() != (i % 3 ? 1 : 4)) Py_RETURN_NONE;
    }
    at::Tensor q;
    {
        const pybind11::gil_scoped_release free;   // (the library's calls may compile)
        q = ResidualFunction::apply(*p, *t[0], *t[1], *t[2], *t[3], *t[4], *t[5], *t[6], *t[7], *t[8], (const Residual*)&r);
    }
    return THPVariable_Wrap(std::move(q));
}

// all_plain(tensors) -> whether all are float32 tensors on the GPU, one behind the other in memory
PyObject* all_plain(PyObject* const* a)
{
    if (!PyList_CheckExact(a[0])) Py_RETURN_FALSE;
    for (Py_ssize_t i = 0; i < PyList_GET_SIZE(a[0]); ++i) {
        PyObject* const o = PyList_GET_ITEM(a[0], i);
        if (!THPVariable_Check(o)) Py_RETURN_FALSE;
        const at::Tensor& t = THPVariable_Unpack(o);
        if (!t.is_cuda() || t.scalar_type() != at::kFloat || t.layout() != at::kStrided || !t.is_contiguous()) Py_RETURN_FALSE;
    }
    Py_RETURN_TRUE;
}

// workspace(device index, bytes) -> uint8 tensor: the scratch of the current stream, for the wrappers in Python
PyObject* workspace_py(PyObject* const* a)
{
    const long dev = PyLong_AsLong(a[0]);
    const long long bytes = PyLong_AsLongLong(a[1]);
    if (PyErr_Occurred()) return nullptr;
    const at::Device device(at::kCUDA, (c10::DeviceIndex)dev);
    c10::DeviceGuard guard(device);
    return THPVariable_Wrap(workspace(device, bytes).buffer);
}

// lock_workspace(device index) -> what unlock_workspace() takes: the lock of the current stream's scratch
PyObject* lock_workspace(PyObject* const* a)
{
    const long dev = PyLong_AsLong(a[0]);
    if (PyErr_Occurred()) return nullptr;
    std::recursive_mutex* const busy = &stream_scratch((int)dev).busy;
    PyObject* const held = PyCapsule_New(busy, nullptr, nullptr);
    if (!held) return nullptr;
    Py_BEGIN_ALLOW_THREADS
    busy->lock();
    Py_END_ALLOW_THREADS
    return held;
}

PyObject* unlock_workspace(PyObject* const* a)
{
    void* const busy = PyCapsule_GetPointer(a[0], nullptr);
    if (!busy) return nullptr;
    static_cast<std::recursive_mutex*>(busy)->unlock();
    Py_RETURN_NONE;
}

PyObject* release_workspaces(PyObject*, PyObject*)
{
    if (g_workspaces)
        for (auto& w : *g_workspaces) w.second.buffer.reset();
    Py_RETURN_NONE;
}

PyObject* has_workspaces(PyObject*, PyObject*)
{
    bool any = false;
    if (g_workspaces)
        for (auto& w : *g_workspaces) any = any || w.second.buffer.defined();
    return PyBool_FromLong(any);
}

PyObject* set_check(PyObject*, PyObject* f)
{
    Py_INCREF(f);
    Py_XSETREF(g_check, f);
    Py_RETURN_NONE;
}

PyObject* set_by_layers(PyObject*, PyObject* f)
{
    Py_INCREF(f);
    Py_XSETREF(g_by_layers, f);
    Py_RETURN_NONE;
}

// set_gradients(gather_gradient, scatter_gradients)
PyObject* set_gradients(PyObject* const* a)
{
    PyObject** const at[2] = {&g_gather_gradient, &g_scatter_gradients};
    for (int i = 0; i < 2; ++i) {
        Py_INCREF(a[i]);
        Py_XSETREF(*at[i], a[i]);
    }
    Py_RETURN_NONE;
}

template <typename F>
PyCFunction fast(F f) { return reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(f)); }

PyMethodDef methods[] = {
    {"reduce_mask", fast(op_entry<reduce_mask, 8>), METH_FASTCALL, nullptr},
    {"gather", fast(op_entry<gather, 8>), METH_FASTCALL, nullptr},
    {"gather_grad", fast(op_entry<gather_grad, 8>), METH_FASTCALL, nullptr},
    {"scatter", fast(op_entry<scatter, 11>), METH_FASTCALL, nullptr},
    {"scatter_base_grad", fast(op_entry<scatter_base_grad, 6>), METH_FASTCALL, nullptr},
    {"block_conv", fast(op_entry<block_conv, 7>), METH_FASTCALL, nullptr},
    {"block_bottleneck", fast(op_entry<block_bottleneck, 12>), METH_FASTCALL, nullptr},
    {"bottleneck_grad", fast(op_entry<bottleneck_grad, 3, 2>), METH_FASTCALL, nullptr},
    {"gather_autograd", fast(op_entry<gather_autograd, 7>), METH_FASTCALL, nullptr},
    {"scatter_autograd", fast(op_entry<scatter_autograd, 10>), METH_FASTCALL, nullptr},
    {"residual", fast(op_entry<residual, 5>), METH_FASTCALL, nullptr},
    {"all_plain", fast(entry<all_plain, 1>), METH_FASTCALL, nullptr},
    {"workspace", fast(entry<workspace_py, 2>), METH_FASTCALL, nullptr},
    {"lock_workspace", fast(entry<lock_workspace, 1>), METH_FASTCALL, nullptr},
    {"unlock_workspace", fast(entry<unlock_workspace, 1>), METH_FASTCALL, nullptr},
    {"release_workspaces", release_workspaces, METH_NOARGS, nullptr},
    {"has_workspaces", has_workspaces, METH_NOARGS, nullptr},
    {"set_check", set_check, METH_O, nullptr},
    {"set_by_layers", set_by_layers, METH_O, nullptr},
    {"set_gradients", fast(entry<set_gradients, 2>), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) { return PyModule_Create(&module_def); }
