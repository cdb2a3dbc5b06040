"""The gradient of a bottleneck's residual function (sbnet_amd/csrc/sbnet_block_grad.hip) against the same steps in float64.

The bound travels with the values: each step passes on the error it received through the absolute values of its
coefficients and adds its own sums' n * 2^-24 * sum |a| * |b| (any order of the sum); batch norm's own arithmetic is a
handful of roundings per value.
"""
import types

import numpy as np
import pytest
import torch
import torch.nn.functional as F

import sbnet_amd
from sbnet_amd import ops
from sbnet_amd import sparse_conv as sc

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
U = 2.0 ** -24


def forward32(rng, M, bsize, ksizes):
    """Stacks, activations, statistics and kernels of a forward pass, in float32: [z, act, mean, inv, kernel, gamma] * 3."""
    out = []
    z = torch.from_numpy(rng.standard_normal((M, ksizes[0][2], *bsize)).astype(np.float32))
    for kh, kw, C, K in ksizes:
        mean, var = z.mean((0, 2, 3)), z.var((0, 2, 3), unbiased=False)
        inv = 1 / (var + sc.BN_EPS).sqrt()
        gamma = torch.from_numpy(rng.uniform(-1.5, 1.5, C).astype(np.float32))   # both signs
        beta = torch.from_numpy(rng.uniform(-0.3, 0.3, C).astype(np.float32))
        col = lambda t: t.view(1, -1, 1, 1)
        act = torch.relu((z - col(mean)) * col(inv) * col(gamma) + col(beta))
        w = torch.from_numpy((rng.standard_normal((K, C, kh, kw)) / np.sqrt(kh * kw * C)).astype(np.float32))
        out += [z, act, mean, inv, w, gamma]
        z = F.conv2d(act, w)
    return out, torch.from_numpy(rng.standard_normal(z.shape).astype(np.float32))


def wgrad64(act, dz, kh, kw):
    R, S = dz.shape[2:]
    return torch.stack([torch.stack([torch.einsum("mcrs,mkrs->ck", act[:, :, i:i + R, j:j + S], dz) for j in range(kw)])
                        for i in range(kh)])


def backward64(saved, dq):
    dz, err = dq.double(), torch.zeros(dq.shape, dtype=torch.float64)
    dws, norms = [], []
    for i in (2, 1, 0):
        z, act, mean, inv, w, gamma = (t.double() for t in saved[6 * i:6 * i + 6])
        kh, kw = w.shape[2:]
        P = dz.shape[0] * dz.shape[2] * dz.shape[3]
        dws.insert(0, (wgrad64(act, dz, kh, kw), wgrad64(act, err + P * U * dz.abs(), kh, kw)))
        taps = w[0, 0].numel() * w.shape[0]
        mask = (act > 0).double()
        err = F.conv_transpose2d(err + taps * U * dz.abs(), w.abs()) * mask
        g = F.conv_transpose2d(dz, w) * mask
        col = lambda t: t.view(1, -1, 1, 1)
        xhat = (z - col(mean)) * col(inv)
        n = z.numel() // z.shape[1]
        s1, s2 = g.sum((0, 2, 3)), (g * xhat).sum((0, 2, 3))
        # 16 values in float32, the rest in double; xhat itself is off by the rounding of z - mean and of the product
        e1 = (err + 20 * U * g.abs()).sum((0, 2, 3))
        e2 = ((err + 24 * U * g.abs()) * xhat.abs()).sum((0, 2, 3))
        norms.insert(0, ((s2, e2 + U * s2.abs()), (s1, e1 + U * s1.abs())))
        scale = col(gamma * inv)
        dz = scale * (g - col(s1) / n - xhat * col(s2) / n)
        err = scale.abs() * (err + col(e1) / n + xhat.abs() * col(e2) / n + 8 * U * (g.abs() + col(s1.abs()) / n + (xhat * col(s2)).abs() / n))
    return (dz, err), dws, norms


CASES = [
    # M, bsize, kernels [kh, kw, C, K]                                      what the size is for
    (1, (3, 4), [[1, 1, 4, 4], [3, 3, 4, 4], [1, 1, 4, 4]]),              # twelve pixels, two of them in the end
    (2, (5, 6), [[1, 1, 12, 8], [3, 3, 8, 8], [1, 1, 8, 12]]),            # four taps share a step of sixteen k
    (7, (11, 11), [[1, 1, 96, 24], [3, 3, 24, 24], [1, 1, 24, 96]]),      # channels between fragments; 32-wide kernel tiles
    (40, (11, 11), [[1, 1, 64, 36], [3, 3, 36, 36], [1, 1, 36, 64]]),     # 64-wide tiles, the last a quarter full
    (3, (9, 7), [[3, 1, 20, 16], [1, 5, 16, 28], [3, 3, 28, 20]]),        # unequal and multiple taps everywhere
    (5, (8, 8), [[1, 1, 260, 132], [3, 3, 132, 132], [1, 1, 132, 260]]),  # second chunk of channels in the batch norm's backward
    (300, (14, 14), [[1, 1, 16, 16], [3, 3, 16, 16], [1, 1, 16, 16]]),    # enough pixels that k is not split
    (100, (18, 18), [[1, 1, 16, 16], [3, 3, 16, 32], [1, 1, 32, 16]]),    # 2025 wave tiles of 16, 32 and 48 channels and 18
    (100, (18, 18), [[1, 1, 16, 32], [3, 3, 32, 32], [1, 1, 32, 16]]),    # steps in the middle: k split in two
    (100, (18, 18), [[1, 1, 16, 48], [3, 3, 48, 32], [1, 1, 32, 16]]),
]


@pytest.mark.parametrize("M,bsize,ksizes", CASES, ids=lambda v: "x".join(str(t) for t in v) if isinstance(v, tuple) else None)
def test_gradients_of_a_bottleneck(M, bsize, ksizes):
    saved, dq = forward32(np.random.default_rng(M), M, bsize, ksizes)
    native = ops._load_native()
    got = native.bottleneck_grad(dq.to(DEV), [t.to(DEV) for t in saved])
    assert got is not None
    dp, dws, norms = backward64(saved, dq)
    want = [dp, *dws, *(pair for n in norms for pair in n)]
    for k, (value, (exact, bound)) in enumerate(zip(got, want)):
        assert value.shape == exact.shape, k
        err = (value.cpu().double() - exact).abs()
        assert bool((err <= 2 * bound + 1e-30).all()), (k, float((err / (2 * bound + 1e-30)).max()))


@pytest.mark.parametrize("frozen", [False, True])
def test_large_steps_take_the_librarys_gradients(frozen):
    params = sc.BottleneckParams([[1, 1, 256, 64], [3, 3, 64, 64], [1, 1, 64, 256]], DEV)
    for w in params.w:
        w.requires_grad_(not frozen)
    most = sc.OWN_GRADIENT_MOST_FROZEN if frozen else sc.OWN_GRADIENT_MOST
    blocks = int(most / (2 * 17 * 17 * sum(w.numel() for w in params.w)))
    for M, own in ((blocks, True), (blocks + 1, False)):
        assert sc._own_residual_gradient(torch.empty(M, 256, 17, 17, device=DEV), params) == own


ALL = range(10)


@pytest.mark.parametrize("wanted", [(), (0,), (1,), (2,), (3,), (4,), (7,), (9,), (1, 3), (2, 4), (0, 2, 8), (1, 2, 3), (4, 5, 6, 7, 8, 9)])
def test_gradients_that_are_not_wanted(wanted):
    """Any of dp, dw1-3 and the batch norms' six alone: the others are None, and what they need is not in the way."""
    M, bsize, ksizes = CASES[2]
    saved, dq = forward32(np.random.default_rng(M), M, bsize, ksizes)
    dp, dws, norms = backward64(saved, dq)
    want = [dp, *dws, *(pair for n in norms for pair in n)]
    got = ops._load_native().bottleneck_grad(dq.to(DEV), [t.to(DEV) for t in saved], tuple(k in wanted for k in ALL))
    for k, (value, (exact, bound)) in enumerate(zip(got, want)):
        assert (value is not None) == (k in wanted)
        if value is not None:
            err = (value.cpu().double() - exact).abs()
            assert bool((err <= 2 * bound + 1e-30).all()), (k, float((err / (2 * bound + 1e-30)).max()))


def test_frozen_kernels_and_input():
    """What requires no gradient gets none; the rest is what it is with everything wanted."""
    results = []
    for frozen in (False, True):
        bp, ind, params, x = make_block()
        if frozen:
            x = x.detach()
            for w in params.w:
                w.requires_grad_(False)
        y = sc.sparse_res_block_bottleneck(x, params, ind, bp, [1, 1, 1, 1], True, data_format="NCHW")
        results.append(torch.autograd.grad(y, [t for b in params.bn for t in b[:2]], torch.cos(y.detach())))
    for a, b in zip(*results):   # (the order in which the sums' atomics arrive is free)
        assert float((a - b).norm()) <= 1e-5 * float(a.norm())


def make_block(C=16, mid=8):
    ksizes = [[1, 1, C, mid], [3, 3, mid, mid], [1, 1, mid, C]]
    bp = sbnet_amd.calc_block_params_res_block([1, 30, 33, C], [1, 9, 9, 1], ksizes, [1, 1, 1, 1], "SAME")
    mask = torch.zeros(1, 30, 33, 1, device=DEV)
    mask[:, 5:20, 8:25] = 1
    x = torch.randn(1, 30, 33, C, device=DEV, generator=torch.Generator(DEV).manual_seed(1))
    return bp, sc.convert_mask_to_indices_custom(mask, bp, 0.0), sc.BottleneckParams(ksizes, DEV, seed=3), x.requires_grad_()


def step(composed, create_graph=False):
    """Output, gradients and running statistics of one training step; `composed`: through the layers one by one."""
    bp, ind, params, x = make_block()
    keep, sc._own_residual_gradient = sc._own_residual_gradient, (lambda p, q: False) if composed else sc._own_residual_gradient
    try:
        y = sc.sparse_res_block_bottleneck(x, params, ind, bp, [1, 1, 1, 1], True, data_format="NCHW")
    finally:
        sc._own_residual_gradient = keep
    tensors = [x, *params.parameters()]
    grads = torch.autograd.grad(y, tensors, torch.cos(y.detach()), create_graph=create_graph)
    if create_graph:
        grads = grads + torch.autograd.grad(sum((g * g).sum() for g in grads[1:]), tensors)
    return y.detach(), [g.detach() for g in grads], [t for b in params.bn for t in (b.moving_mean, b.moving_var)]


def test_step_equals_composed_step():
    (y, g, s), (y0, g0, s0) = step(False), step(True)
    assert torch.equal(y, y0) and all(torch.equal(a, b) for a, b in zip(s, s0))   # the forward pass is the same calls
    for a, b in zip(g, g0):   # two float32 results of 200-pixel sums, each within its own bound of the exact one
        assert float((a - b).norm()) <= 4 * 25 ** 2 * U * 81 ** 0.5 * float(b.norm()), float((a - b).norm() / b.norm())


def test_gradient_of_a_gradient_goes_through_the_layers():
    (_, g, _), (_, g0, _) = step(False, True), step(True, True)
    for a, b in zip(g, g0):
        assert float((a - b).norm()) <= 1e-4 * float(b.norm())


def test_kernel_changed_between_forward_and_backward():
    """The forward pass keeps its own copy of a kernel: an optimizer's step before backward changes no gradient."""
    bp, ind, params, x = make_block()
    tensors = [x, *params.parameters()]
    y = sc.sparse_res_block_bottleneck(x, params, ind, bp, [1, 1, 1, 1], True, data_format="NCHW")
    first = torch.autograd.grad(y, tensors, torch.ones_like(y), retain_graph=True)
    with torch.no_grad():
        for w in params.w:
            w.add_(1.0)
    second = torch.autograd.grad(y, tensors, torch.ones_like(y))
    for a, b in zip(first, second):
        assert float((a - b).norm()) <= 1e-6 * float(a.norm())


@pytest.mark.parametrize("create_graph", [False, True])
def test_kernels_and_betas_changed_between_forward_and_backward(create_graph):
    """No gradient depends on what a beta or a kernel is by the time of backward; nor does a gradient's gradient."""
    results = []
    for change in (False, True):
        bp, ind, params, x = make_block()
        tensors = [x, *params.parameters()]
        y = sc.sparse_res_block_bottleneck(x, params, ind, bp, [1, 1, 1, 1], True, data_format="NCHW")
        if change:
            with torch.no_grad():
                for t in [*params.w, *(b.beta for b in params.bn)]:
                    t.add_(1.0)
        grads = torch.autograd.grad(y, tensors, torch.ones_like(y), create_graph=create_graph)
        if create_graph:
            grads = grads + torch.autograd.grad(sum((g * g).sum() for g in grads), tensors)
        results.append([g.detach() for g in grads])
    # The same sums, in an order that the library is free in: six of them one behind the other, over up to 2025 pixels, are
    # off by about 6 * 2025 ** 0.5 * 2^-24 = 1.6e-5, the gradients' own cancellation not counted.
    for a, b in zip(*results):
        assert float((a - b).norm()) <= 1e-4 * float(a.norm())


@pytest.mark.parametrize("is_training,no_activation", [(True, False), (True, True), (False, True)])
def test_blocks_without_running_statistics_or_a_first_batch_norm(is_training, no_activation):
    """What a block does not use may be absent, and the batch norms' parameters may come in any object with their names."""
    bp, ind, params, x = make_block()
    x = x.detach()
    with torch.no_grad():
        want = sc.sparse_res_block_bottleneck(x, params, ind, bp, [1, 1, 1, 1], is_training, "NCHW", no_activation=no_activation)
    params.bn = [types.SimpleNamespace(**b._asdict()) for b in params.bn]
    for b in params.bn if is_training else ():
        b.moving_mean = b.moving_var = None
    if no_activation:
        params.bn[0] = None
    for grad in (False, is_training):
        with torch.set_grad_enabled(grad):
            y = sc.sparse_res_block_bottleneck(x, params, ind, bp, [1, 1, 1, 1], is_training, "NCHW", no_activation=no_activation)
        assert torch.equal(y, want)
