"""The differentiable ops in native code against the autograd functions in Python whose place they take, and what still goes to
those."""
import pytest
import torch
from torch.autograd import forward_ad
from torch.utils._python_dispatch import TorchDispatchMode

import sbnet_amd
from sbnet_amd import SparseGatherFunction, SparseScatterFunction, ops
from sbnet_amd import sparse_conv as sc

DEV = "cuda:0"
BS, BT, BO = [6, 6], [4, 5], [-1, -2]


def make(C=12, M=5, transpose=False, seed=0, device=DEV):
    g = torch.Generator(device=device).manual_seed(seed)
    idx = torch.tensor([(0, i, (2 * i) % 3) for i in range(M)], dtype=torch.int16, device=device)
    x = torch.randn(1, 24, 20, C, device=device, generator=g)
    q = torch.randn(*((M, C, *BS) if transpose else (M, *BS, C)), device=device, generator=g)
    return x, q, idx, torch.tensor([M], dtype=torch.int32)


def test_tensors_that_are_not_plain_are_left_alone():
    x, q, idx, cnt = make(device="cpu")
    native = ops._load_native()
    x.requires_grad_()
    assert native.gather_autograd(x, cnt, idx, BS, BT, BO, False) is None
    assert native.scatter_autograd(q, cnt, idx, x, BS, BT, BO, False, False, False) is None
    assert native.residual(q, [None] * 6, [q] * 9, 0.1, 1e-3) is None
    assert not native.all_plain([x, q])


@pytest.mark.gpu
@pytest.mark.parametrize("add", [False, True])
@pytest.mark.parametrize("transpose", [False, True])
@pytest.mark.parametrize("wanted", ["x", "q", "xq"])
def test_gradients_are_those_of_the_functions_in_python(wanted, transpose, add):
    x, q, idx, cnt = make(transpose=transpose)
    x.requires_grad_("x" in wanted)
    q.requires_grad_("q" in wanted)
    leaves = [t for t in (x, q) if t.requires_grad]
    results = []
    for python in (False, True):
        if python:
            p = SparseGatherFunction.apply(x, cnt, idx, BS, BT, BO, transpose)
            y = SparseScatterFunction.apply(q, cnt, idx, x, BS, BT, BO, add, True, transpose)
        else:
            p = sbnet_amd.sparse_gather(x, cnt, idx, BS, BT, BO, transpose=transpose)
            y = sbnet_amd.sparse_scatter(q, cnt, idx, x, BS, BT, BO, add=add, atomic=True, transpose=transpose)
            assert "Function" in y.grad_fn.name() and "Sparse" not in y.grad_fn.name()
        assert p.requires_grad == x.requires_grad and y.requires_grad
        # gradients that are not contiguous; an unused output; twice, with the graph kept
        dy = torch.linspace(-1, 1, y.shape[3], device=DEV).expand(y.shape)
        grads = torch.autograd.grad(y, leaves, dy, retain_graph=True)
        grads += torch.autograd.grad([y] + [p] * p.requires_grad, leaves, [dy] + [p.detach()] * p.requires_grad)
        results.append((p.detach(), y.detach(), *grads))
    for a, b in zip(*results):
        assert torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("add", [False, True])
def test_gradient_of_the_bases_gradient(add):
    x, q, idx, cnt = make()
    results = []
    for op in (sbnet_amd.sparse_scatter, SparseScatterFunction.apply):
        base, dy = x.clone().requires_grad_(), torch.cos(x).requires_grad_()
        y = op(q, cnt, idx, base, BS, BT, BO, add, True, False)
        g, = torch.autograd.grad(y, base, dy, create_graph=True)
        results.append((g.detach(), torch.autograd.grad(g, dy, x)[0]))
    for a, b in zip(*results):
        assert torch.equal(a, b)


@pytest.mark.gpu
def test_hooks_of_saved_tensors_see_the_list():
    x, q, idx, cnt = make()
    x.requires_grad_()
    seen = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: seen.append(t.shape) or t.cpu(), lambda t: t.to(DEV)):
        p = sbnet_amd.sparse_gather(x, cnt, idx, BS, BT, BO)
        y = sbnet_amd.sparse_scatter(q, cnt, idx, x, BS, BT, BO, add=True, atomic=True)
    assert seen == [idx.shape, idx.shape]
    got, = torch.autograd.grad([p, y], x, [p.detach(), y.detach()])
    want, = torch.autograd.grad([sbnet_amd.sparse_gather(x, cnt, idx, BS, BT, BO)], x, [p.detach()])
    assert torch.equal(got, want + y.detach())


def scatter_native(x, q, idx, cnt, add=True):
    return sbnet_amd.sparse_scatter(q, cnt, idx, x, BS, BT, BO, add=add, atomic=True)


def scatter_python(x, q, idx, cnt, add=True):
    return SparseScatterFunction.apply(q, cnt, idx, x, BS, BT, BO, add, True, False)


def gather_native(x, q, idx, cnt):
    return sbnet_amd.sparse_gather(x, cnt, idx, BS, BT, BO)


def gather_python(x, q, idx, cnt):
    return SparseGatherFunction.apply(x, cnt, idx, BS, BT, BO, False)


@pytest.mark.gpu
@pytest.mark.parametrize("op", [gather_native, gather_python, scatter_native, scatter_python])
@pytest.mark.parametrize("change,error,text", [
    (lambda t: t[:3].clone(), ops.InvalidArgument, "outside the block list of 3 rows"),
    (lambda t: t[:, :2].clone(), ops.InvalidArgument, "must have shape"),
    (lambda t: t.view(-1), ops.InvalidArgument, "must have shape"),
    (lambda t: t.int(), TypeError, "int16 tensor on the GPU"),
    (lambda t: t.cpu(), TypeError, "int16 tensor on the GPU"),
], ids=["shorter", "narrower", "flat", "int32", "cpu"])
def test_a_list_that_a_hook_hands_back_otherwise_is_refused(op, change, error, text):
    x, q, idx, cnt = make()
    q.requires_grad_()
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, change):
        y = op(x.requires_grad_(), q, idx, cnt)
    with pytest.raises(error, match=text):
        torch.autograd.grad(y.sum(), [x] if "gather" in op.__name__ else [x, q])


@pytest.mark.gpu
@pytest.mark.parametrize("op", [scatter_native, scatter_python])
def test_a_batch_of_gradients_passes_through_an_adds_base(op):
    """The base's gradient of an add is the gradient itself, whatever tensor that is."""
    x, q, idx, cnt = make()
    y = op(x.requires_grad_(), q, idx, cnt)
    dy = torch.randn(3, *y.shape, device=DEV)
    got, = torch.autograd.grad(y, x, dy, is_grads_batched=True)
    assert torch.equal(got, dy)


@pytest.mark.gpu
def test_modes_of_the_backward_pass_look_on():
    """What runs under a mode is left to the general wrappers, whose results are the same."""
    seen = []

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))

    x, q, idx, cnt = make()
    x.requires_grad_()
    q.requires_grad_()
    for op, leaves in ((gather_native, [x]), (scatter_native, [x, q]), (lambda *a: scatter_native(*a, add=False), [x, q])):
        y = op(x, q, idx, cnt)
        want = torch.autograd.grad(y, leaves, y.detach(), retain_graph=True)
        with Mode():
            got = torch.autograd.grad(y, leaves, y.detach())
        for a, b in zip(got, want):
            assert torch.equal(a, b)
    assert torch.ops.aten.empty.memory_format in seen   # (the general wrapper's own results)


@pytest.mark.gpu
def test_what_looks_on_or_transforms_goes_to_the_functions_in_python():
    x, q, idx, cnt = make()

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    x.requires_grad_()
    with Mode():
        assert "SparseGatherFunction" in sbnet_amd.sparse_gather(x, cnt, idx, BS, BT, BO).grad_fn.name()
        assert "SparseScatterFunction" in sbnet_amd.sparse_scatter(q, cnt, idx, x, BS, BT, BO, add=True, atomic=True).grad_fn.name()
    with forward_ad.dual_level(), pytest.raises(RuntimeError):   # (no rule for forward mode: refused, not dropped)
        sbnet_amd.sparse_gather(forward_ad.make_dual(x, torch.ones_like(x)), cnt, idx, BS, BT, BO)
    with pytest.raises(RuntimeError):                             # (functorch wants setup_context)
        torch.func.grad(lambda t: sbnet_amd.sparse_gather(t, cnt, idx, BS, BT, BO).sum())(x.detach())
    # a count on the device
    y = sbnet_amd.sparse_gather(x, cnt.to(DEV), idx, BS, BT, BO)
    assert "SparseGatherFunction" in y.grad_fn.name()


@pytest.mark.gpu
def test_a_changed_list_is_noticed():
    x, _, idx, cnt = make()
    y = sbnet_amd.sparse_gather(x.requires_grad_(), cnt, idx, BS, BT, BO)
    idx.add_(0)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        torch.autograd.grad(y.sum(), x)


@pytest.mark.gpu
@pytest.mark.parametrize("shapes", [[(1, 1, 4, 4)], [(3, 3, 20, 12), (1, 5, 7, 3)], [(1, 1, 256, 64), (3, 3, 64, 64), (7, 7, 1, 33)]],
                         ids=str)
def test_kernels_in_the_librarys_order(shapes):
    import ctypes
    import numpy as np
    from sbnet_amd import _lib
    w = [torch.randn(*s, device=DEV) for s in shapes]
    out = [torch.empty(s[3], s[2], s[0], s[1], device=DEV) for s in shapes]
    n = len(w)
    pointers = lambda ts: ctypes.cast((ctypes.c_void_p * 4)(*(t.data_ptr() for t in ts)), ctypes.c_void_p)
    fn = _lib.load().sbnet_kernels_oihw
    call = lambda d, k: fn(pointers(w), ops._pair(d.reshape(-1))[1], pointers(out), k, ops._stream())
    dims = np.array(shapes, np.int32)
    assert call(dims, n) == 0
    for a, b in zip(out, w):
        assert torch.equal(a, b.permute(3, 2, 0, 1))
    assert call(dims, 4) == call(dims, 0) == call(dims * 0, n) == _lib.SBNET_EINVAL_ARG


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 3, 4, 4095, 4096, 4099, 100001])
def test_relu_is_the_librarys(n):
    from sbnet_amd import _lib
    x = torch.randn(n, device=DEV)
    special = torch.tensor([float("nan"), -0.0, 0.0, float("inf"), -float("inf"), -1e-45, 1e-45], device=DEV)[:n]
    x[n - len(special):] = special
    want = torch.relu(x)
    fn = _lib.load().sbnet_relu
    assert fn(x.data_ptr(), n, ops._stream()) == 0
    assert torch.equal(x.view(torch.int32), want.view(torch.int32))
    assert fn(x.data_ptr() + 4, 1, ops._stream()) == _lib.SBNET_EINVAL_ARG


# ---- the residual function ----------------------------------------------------------------------------------------

class LooksOn(TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


def residual_native(p, params):
    q = sc._residual_in_training(p, params)
    assert "ResidualFunction" in q.grad_fn.name() and "InTraining" not in q.grad_fn.name()
    return q


def residual_python(p, params):
    with LooksOn():     # which the native function leaves to the one in Python
        q = sc._residual_in_training(p, params)
    assert "_ResidualInTraining" in q.grad_fn.name()
    return q


def make_residual(stats=True, seed=3):
    params = sc.BottleneckParams([(1, 1, 16, 8), (3, 3, 8, 8), (1, 1, 8, 16)], DEV, seed=seed)
    g = torch.Generator(device=DEV).manual_seed(seed)
    if not stats:
        params.bn = [sc.BatchNormParams(b.gamma, b.beta, None, None) for b in params.bn]
    return params, torch.randn(6, 16, 9, 9, device=DEV, generator=g).requires_grad_()


def same(got, want):
    """The same kernels on the same values, but for the order of the batch norms' sums, which are added up in double: a unit in
    the last place of a coefficient, 2^-24 of each term, and what the later layers make of it."""
    assert len(got) == len(want)
    for a, b in zip(got, want):
        assert a.shape == b.shape and torch.linalg.vector_norm(a - b) <= 1e-6 * torch.linalg.vector_norm(b) + 1e-9


def leaves_of(p, params):
    return [p] + params.parameters()


@pytest.mark.gpu
@pytest.mark.parametrize("wanted", ["all", "input", "kernels", "norms"])
@pytest.mark.parametrize("create_graph", [False, True])
def test_residual_function_is_the_one_in_python(wanted, create_graph):
    results = []
    for op in (residual_native, residual_python):
        params, p = make_residual()
        for i, t in enumerate(leaves_of(p, params)):
            t.requires_grad_(wanted == "all" or (wanted == "input") == (i == 0) and (wanted == "kernels") == (1 <= i <= 3))
        leaves = [t for t in leaves_of(p, params) if t.requires_grad]
        q = op(p, params)
        dq = torch.linspace(-1, 1, q.numel(), device=DEV).view(q.shape)
        grads = torch.autograd.grad(q, leaves, dq, create_graph=create_graph)
        stats = [t for b in params.bn for t in (b.moving_mean, b.moving_var)]
        if create_graph:
            grads += torch.autograd.grad(sum((g * g).sum() for g in grads), leaves)
        results.append([q.detach(), *stats, *(g.detach() for g in grads)])
    same(*results)


@pytest.mark.gpu
@pytest.mark.parametrize("op", [residual_native, residual_python])
def test_residual_function_under_hooks_of_saved_tensors(op):
    params, p = make_residual()
    want = torch.autograd.grad(op(p, params).square().sum(), leaves_of(p, params))
    kept = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: kept.append(t.shape) or t.cpu(), lambda t: t.to(DEV)):
        q = op(p, params)
    assert len(kept) == 18
    same(torch.autograd.grad(q.square().sum(), leaves_of(p, params)), want)
    # what comes back in another order of memory goes through the layers: other kernels' sums, of up to 486 pixels and 144 taps
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t.to(memory_format=torch.channels_last) if t.dim() == 4 else t):
        q = op(p, params)
    for a, b in zip(torch.autograd.grad(q.square().sum(), leaves_of(p, params)), want):
        assert torch.linalg.vector_norm(a - b) <= 1e-4 * torch.linalg.vector_norm(b)


@pytest.mark.gpu
@pytest.mark.parametrize("op", [residual_native, residual_python])
def test_residual_function_in_a_checkpoint(op):
    from torch.utils.checkpoint import checkpoint
    params, p = make_residual(stats=False)
    want = torch.autograd.grad(op(p, params).square().sum(), leaves_of(p, params))
    q = checkpoint(lambda t: op(t, params), p, use_reentrant=False)
    same(torch.autograd.grad(q.square().sum(), leaves_of(p, params)), want)


@pytest.mark.gpu
@pytest.mark.parametrize("op", [residual_native, residual_python])
def test_residual_function_takes_a_batch_of_gradients(op):
    """Through the layers, one by one: sums of up to 486 pixels and 144 taps in another order."""
    params, p = make_residual(stats=False)
    q = op(p, params)
    dq = torch.randn(3, *q.shape, device=DEV)
    got = torch.autograd.grad(q, leaves_of(p, params), dq, is_grads_batched=True, retain_graph=True)
    for i in range(3):
        for a, b in zip(got, torch.autograd.grad(q, leaves_of(p, params), dq[i], retain_graph=True)):
            assert torch.linalg.vector_norm(a[i] - b) <= 1e-4 * torch.linalg.vector_norm(b)


@pytest.mark.gpu
def test_residual_functions_of_two_threads():
    """The forward pass runs without the interpreter's lock."""
    from concurrent.futures import ThreadPoolExecutor

    def job(seed):
        params, p = make_residual(seed=seed)
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            out = []
            for _ in range(5):
                q = residual_native(p, params)
                out = [q.detach(), *torch.autograd.grad(q.square().sum(), leaves_of(p, params))]
            stream.synchronize()
        return [t.cpu() for t in out]

    want = [job(seed) for seed in (1, 2)]
    with ThreadPoolExecutor(2) as pool:
        got = list(pool.map(job, (1, 2)))
    for a, b in zip(got, want):
        same(a, b)
