"""The block convolutions (sbnet_amd/csrc/sbnet_conv.hip) against float64 convolutions of the gathered blocks.

The bound on a float32 sum of n products in any order is n * 2^-24 * sum |a| * |w| (plus rounding of the operands,
none here); through batch norm and ReLU the same argument runs with the folded scale, so the tests compare with that
bound evaluated per element on the absolute values, in float64.
"""
import threading

import numpy as np
import pytest
import torch
import torch.nn.functional as F
from torch.utils.flop_counter import FlopCounterMode

import sbnet_amd
from sbnet_amd import ops
from sbnet_amd import sparse_conv as sc
from sbnet_amd.block_params import BlockParams

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
U = 2.0 ** -24


def blocks64(x, idx, bsize, bstride, boffset):
    """Gathered blocks [M,C,R,S] in float64 on the CPU, zeros outside the image."""
    R, S = bsize
    xp = F.pad(x.double().permute(0, 3, 1, 2), (64, 64, 64, 64))
    out = [xp[n, :, 64 + boffset[0] + bh * bstride[0]:, 64 + boffset[1] + bw * bstride[1]:][:, :R, :S] for n, bh, bw in idx.tolist()]
    return torch.stack(out)


def make_blocks(rng, N, H, W, bsize, bstride, boffset, M):
    """M distinct blocks, borders included, in random order."""
    bc = [1 + (H - boffset[0] - 1) // bstride[0], 1 + (W - boffset[1] - 1) // bstride[1]]
    T = N * bc[0] * bc[1]
    pick = rng.permutation(T)[:M]
    idx = np.stack([pick // (bc[0] * bc[1]), pick // bc[1] % bc[0], pick % bc[1]], 1).astype(np.int16)
    return torch.from_numpy(idx)


CONVS = [
    # N, H, W, C, K, kh, kw, bsize, M      what the size is for
    (1, 20, 24, 1, 1, 1, 1, (5, 5), 6),     # one channel, one k
    (2, 31, 29, 3, 5, 3, 3, (6, 9), 9),     # no vector width
    (1, 40, 40, 8, 2, 3, 3, (7, 7), 11),    # four-wide input, narrow output
    (1, 33, 50, 10, 10, 5, 3, (9, 11), 7),  # k not a multiple of 16, unequal kernel sides
    (1, 40, 60, 4, 4, 3, 3, (10, 10), 8),   # four taps share a step
    (1, 64, 64, 12, 20, 1, 1, (8, 8), 20),  # last step three quarters full, second channel fragment a quarter full
    (1, 64, 48, 24, 24, 3, 3, (17, 17), 5),
    (3, 40, 40, 48, 48, 3, 3, (8, 8), 30),
    (1, 50, 50, 130, 36, 3, 3, (9, 9), 6),  # channels no multiple of four
    (1, 60, 60, 132, 68, 1, 1, (6, 6), 40),
    (1, 300, 300, 16, 64, 3, 3, (12, 12), 700),   # enough tiles that k is not split
    (1, 300, 300, 7, 33, 3, 3, (12, 12), 700),
    (1, 260, 260, 32, 16, 3, 3, (18, 18), 110),   # 1760 wave tiles of 16, 32 and 48 channels: k split in two
    (1, 260, 260, 32, 32, 3, 3, (18, 18), 110),
    (1, 260, 260, 32, 48, 3, 3, (18, 18), 110),
]


@pytest.mark.parametrize("device_count", [False, True])
@pytest.mark.parametrize("case", CONVS, ids=lambda c: "x".join(str(v) for v in c[:7]))
def test_block_conv(case, device_count):
    N, H, W, C, K, kh, kw, bsize, M = case
    rng = np.random.default_rng(C * 100 + K)
    bstride, boffset = (bsize[0] - kh + 1, bsize[1] - kw + 1), (-(kh // 2), -(kw // 2))
    idx = make_blocks(rng, N, H, W, bsize, bstride, boffset, M)
    M = idx.shape[0]
    x = torch.from_numpy(rng.standard_normal((N, H, W, C)).astype(np.float32))
    w = torch.from_numpy(rng.standard_normal((kh, kw, C, K)).astype(np.float32))
    listed = torch.cat([idx, torch.full((3, 3), 77, dtype=torch.int16)]) if device_count else idx
    count = torch.tensor([M], dtype=torch.int32)
    bp = BlockParams(bsize=list(bsize), bsize_out=list(bstride), boffset=list(boffset), bcount=None, bstrides=list(bstride))
    q = sc._block_conv(x.to(DEV), w.to(DEV), sbnet_amd.ReduceMaskResult(listed.to(DEV), count.to(DEV) if device_count else count), bp)
    assert q is not None and q.shape[1:] == (bstride[0], bstride[1], K)
    p = blocks64(x, idx, bsize, bstride, boffset)
    w64 = w.double().permute(3, 2, 0, 1)
    want = F.conv2d(p, w64).permute(0, 2, 3, 1)
    bound = kh * kw * C * U * F.conv2d(p.abs(), w64.abs()).permute(0, 2, 3, 1)
    err = (q[:M].cpu().double() - want).abs()
    assert bool((err <= bound + 1e-30).all()), float((err / (bound + 1e-30)).max())


@pytest.mark.parametrize("C,k,M,bsize,own", [
    (12, 3, 3000, 18, True),      # narrow: however many pixels
    (96, 3, 1500, 18, True),      # 63.7 GFLOP
    (96, 3, 1550, 18, False),     # 65.8
    (80, 3, 2400, 18, True),
    (128, 1, 1500, 17, True),     # one tap
    (30, 3, 280, 18, True),       # 2.4 and 2.6 million steps of 16 k times 16 channels
    (30, 3, 300, 18, False),
    (3, 7, 350, 22, True),        # 0.90 and 0.92
    (3, 7, 360, 22, False),
])
def test_where_the_library_takes_over(C, k, M, bsize, own):
    """The route of a product by its size; the two sides agree within the bound of a sum in any order, 2 * k * k * C * 2^-24
    of the sum of absolute products."""
    idx = torch.stack([torch.zeros(M, dtype=torch.int64), torch.arange(M) // 40, torch.arange(M) % 40], 1).to(torch.int16).to(DEV)
    out = bsize - k + 1
    bp = BlockParams(bsize=[bsize] * 2, bsize_out=[out] * 2, boffset=[-(k // 2)] * 2, bcount=None, bstrides=[out] * 2)
    g = torch.Generator(DEV).manual_seed(C)
    x = torch.rand(1, (M // 40 + 1) * out, 40 * out, C, device=DEV, generator=g)   # (positive: the sum itself)
    w = torch.rand(k, k, C, C, device=DEV, generator=g)
    ind = sbnet_amd.ReduceMaskResult(idx, torch.tensor([M], dtype=torch.int32))
    assert (sc._block_conv(x, w, ind, bp) is not None) == own
    on_device = sbnet_amd.ReduceMaskResult(idx, torch.tensor([M], dtype=torch.int32, device=DEV))
    results = [sc.sparse_conv2d_custom(x, w, i, bp, [1, 1, 1, 1], transpose=t) for i in (ind, on_device) for t in (False, True)]
    for y in results[1:]:
        assert bool(((y - results[0]).abs() <= 2 * k * k * C * U * results[0]).all())


def bottleneck64(p, params, no_activation):
    """Residual function in float64 and, beside it, the accumulated rounding bound: each stage adds its own sum's bound and
    passes on the one it received through the absolute values of its scales and weights."""
    err = torch.zeros_like(p)
    for i, (w, bn) in enumerate(zip(params.w, params.bn)):
        if i or not no_activation:
            g, b, m, v = (t.detach().cpu().double().view(1, -1, 1, 1) for t in bn)
            scale = g / (v + sc.BN_EPS).sqrt()
            # the mean comes off first, so what is rounded is the distance from it
            err = scale.abs() * err + 8 * U * (((p - m) * scale).abs() + b.abs())
            p = torch.relu((p - m) * scale + b)
        w64 = w.detach().cpu().double().permute(3, 2, 0, 1)
        n = int((w64 != 0).sum((1, 2, 3)).max())   # (a product with zero rounds nothing)
        err = F.conv2d(err + n * U * p.abs(), w64.abs())
        p = F.conv2d(p, w64)
    return p.permute(0, 2, 3, 1), err.permute(0, 2, 3, 1)


@pytest.mark.parametrize("use_var", [False, True])
@pytest.mark.parametrize("no_activation", [False, True])
@pytest.mark.parametrize("C,mid,bsize,shape", [(6, 3, 5, (2, 23, 31)), (24, 8, 9, (1, 40, 52)), (96, 24, 17, (1, 70, 64)),
                                               (260, 64, 7, (1, 30, 30)), (16, 16, 24, (1, 220, 220))])
def test_bottleneck_in_inference(C, mid, bsize, shape, no_activation, use_var):
    check_bottleneck(C, mid, bsize, shape, no_activation, use_var)


def check_bottleneck(C, mid, bsize, shape, no_activation, use_var):
    """Returns the number of output pixels."""
    rng = np.random.default_rng(C)
    ksizes = [[1, 1, C, mid], [3, 3, mid, mid], [1, 1, mid, C]]
    bp = sbnet_amd.calc_block_params_res_block([shape[0], shape[1], shape[2], C], [1, bsize, bsize, 1], ksizes, [1, 1, 1, 1], "SAME")
    mask = torch.from_numpy((rng.random((*shape, 1)) < 0.02).astype(np.float32)).to(DEV)
    ind = sc.convert_mask_to_indices_custom(mask, bp, 0.0)
    M = int(ind.bin_counts[0])
    params = sc.BottleneckParams(ksizes, DEV, seed=C)
    with torch.no_grad():
        for bn in params.bn:
            for t, (lo, hi) in zip(bn, ((0.5, 1.5), (-0.3, 0.3), (-0.3, 0.3), (0.5, 1.5))):
                t.copy_(torch.from_numpy(rng.uniform(lo, hi, t.shape).astype(np.float32)))
    x = torch.from_numpy(rng.standard_normal((*shape, C)).astype(np.float32))
    xd = x.to(DEV)
    with torch.no_grad():
        assert sc._block_bottleneck(xd, params, ind, bp, no_activation, False) is not None
        y = sc.sparse_res_block_bottleneck(xd, params, ind, bp, [1, 1, 1, 1], False, no_activation=no_activation, use_var=use_var)
    assert (y.data_ptr() == xd.data_ptr()) == use_var
    idx = ind.active_block_indices[:M].cpu()
    q, bound = bottleneck64(blocks64(x, idx, bp.bsize, bp.bstrides, bp.boffset), params, no_activation)
    want, most = x.double().clone(), torch.zeros(x.shape, dtype=torch.float64)
    Ro, So = bp.bsize_out
    for i, (n, bh, bw) in enumerate(idx.tolist()):
        part = want[n, bh * Ro:(bh + 1) * Ro, bw * So:(bw + 1) * So]
        part += q[i, :part.shape[0], :part.shape[1]]
        most[n, bh * Ro:(bh + 1) * Ro, bw * So:(bw + 1) * So] = bound[i, :part.shape[0], :part.shape[1]] + U * part.abs()
    err = (y.cpu().double() - want).abs()
    assert bool((err <= most + 1e-30).all()), float((err / (most + 1e-30)).max())
    return M * Ro * So


@pytest.mark.parametrize("ratio", [10.0, 1000.0])
@pytest.mark.parametrize("C", [16, 18])
@pytest.mark.parametrize("no_activation", [False, True])
def test_batch_norm_of_values_far_from_zero(C, no_activation, ratio):
    """Channels whose mean is many times their spread, in front of the first convolution or, with kernels that only pass
    pixels on, behind it: the result is off by the rounding of the distance from the mean, not of the mean."""
    shape, ksizes = (1, 30, 41), [[1, 1, C, C], [3, 3, C, C], [1, 1, C, C]]
    bp = sbnet_amd.calc_block_params_res_block([*shape, C], [1, 9, 9, 1], ksizes, [1, 1, 1, 1], "SAME")
    ind = sc.convert_mask_to_indices_custom(torch.ones(*shape, 1, device=DEV), bp, 0.0)
    M = int(ind.bin_counts[0])
    params = sc.BottleneckParams(ksizes, DEV, seed=C)
    rng = np.random.default_rng(C)
    x = torch.from_numpy((ratio + rng.standard_normal((*shape, C))).astype(np.float32))
    with torch.no_grad():
        for w in params.w:
            w.zero_()[w.shape[0] // 2, w.shape[1] // 2].copy_(torch.eye(C))
        bn = params.bn[1 if no_activation else 0]
        bn.moving_mean.copy_(torch.from_numpy((ratio + 0.1 * rng.standard_normal(C)).astype(np.float32)))
        q = sc._block_bottleneck(x.to(DEV), params, ind, bp, no_activation, False)
    idx = ind.active_block_indices[:M].cpu()
    # (nothing is rounded in front of that batch norm; pixels outside the image are as far from the mean as it is from 0)
    want, bound = bottleneck64(blocks64(x, idx, bp.bsize, bp.bstrides, bp.boffset), params, no_activation)
    err = (q.cpu().double() - want).abs()
    assert bool((err <= bound + 1e-30).all()), float((err / (bound + 1e-30)).max())


@pytest.mark.parametrize("C,kh", [(18, 1), (20, 1), (20, 3), (18, 3), (5, 3)])   # k ends inside a step of sixteen
def test_infinite_shift_of_a_channel_stays_infinite(C, kh):
    """Infinities where the exact result has them, and no NaN out of the places past the last k."""
    shape, ksizes = (1, 30, 41), [[kh, kh, C, 8], [1, 1, 8, 8], [1, 1, 8, C]]
    bp = sbnet_amd.calc_block_params_res_block([*shape, C], [1, 9, 9, 1], ksizes, [1, 1, 1, 1], "SAME")
    ind = sc.convert_mask_to_indices_custom(torch.ones(*shape, 1, device=DEV), bp, 0.0)
    params = sc.BottleneckParams(ksizes, DEV, seed=C)
    with torch.no_grad():
        for w in params.w:
            w.abs_()
        params.bn[0].beta[-1] = float("inf")
        q = sc._block_bottleneck(torch.randn(*shape, C, device=DEV), params, ind, bp, False, False)
    assert bool((q == float("inf")).all())


ONE_LAUNCH = 1536 * 16   # output pixels from which on the last two convolutions share a launch, up to 128 channels in between


@pytest.mark.parametrize("use_var", [False, True])
@pytest.mark.parametrize("C,mid,bsize,shape,one", [
    (96, 24, 17, (1, 190, 205), True),      # one fragment of channels in between and half of another
    (40, 36, 17, (2, 140, 150), True),      # three, the last a quarter full
    (256, 64, 17, (1, 180, 175), True),     # four
    (132, 84, 17, (1, 180, 175), True),     # six; output tiles of 64 channels and a rest
    (64, 100, 17, (1, 180, 175), True),     # seven of eight
    (64, 128, 24, (1, 180, 185), True),     # eight
    (132, 84, 11, (1, 60, 44), False),      # few pixels: two launches
    (20, 132, 17, (1, 180, 175), False),    # more than one tile of channels in between: two launches
])
def test_last_two_convolutions_in_one_launch(C, mid, bsize, shape, one, use_var):
    assert (check_bottleneck(C, mid, bsize, shape, False, use_var) >= ONE_LAUNCH and mid <= 128) == one


def test_layers_under_autocast_take_the_layers_own_way():
    """Autocast makes the composed convolutions compute in half precision, which the scatter refuses: so does the layer."""
    bp = sbnet_amd.calc_block_params([1, 20, 20, 16], [1, 8, 8, 1], [3, 3, 16, 16], [1, 1, 1, 1], "SAME")
    ind = sc.convert_mask_to_indices_custom(torch.ones(1, 20, 20, 1, device=DEV), bp, 0.0)
    x, w = torch.randn(1, 20, 20, 16, device=DEV), torch.randn(3, 3, 16, 16, device=DEV)
    with torch.no_grad(), torch.autocast("cuda", dtype=torch.float16), pytest.raises(TypeError):
        sc.sparse_conv2d_custom(x, w, ind, bp, [1, 1, 1, 1])
    with torch.no_grad():
        sc.sparse_conv2d_custom(x, w, ind, bp, [1, 1, 1, 1])


def test_layers_under_a_dispatch_mode_take_the_layers_own_way():
    """What looks on at torch's operators (here: counts their operations) sees a layer's convolution."""
    bp = sbnet_amd.calc_block_params([1, 20, 20, 16], [1, 8, 8, 1], [3, 3, 16, 16], [1, 1, 1, 1], "SAME")
    ind = sc.convert_mask_to_indices_custom(torch.ones(1, 20, 20, 1, device=DEV), bp, 0.0)
    x, w = torch.randn(1, 20, 20, 16, device=DEV), torch.randn(3, 3, 16, 16, device=DEV)
    with torch.no_grad(), FlopCounterMode(display=False) as flops:
        sc.sparse_conv2d_custom(x, w, ind, bp, [1, 1, 1, 1])
    assert flops.get_total_flops() == 2 * int(ind.bin_counts[0]) * 36 * 9 * 16 * 16


def residual_layer(seed, shape=(1, 60, 70), C=32, mid=8, bsize=9):
    """A residual layer in place on a tensor, its input, and what it gives by itself."""
    ksizes = [[1, 1, C, mid], [3, 3, mid, mid], [1, 1, mid, C]]
    bp = sbnet_amd.calc_block_params_res_block([*shape, C], [1, bsize, bsize, 1], ksizes, [1, 1, 1, 1], "SAME")
    ind = sc.convert_mask_to_indices_custom(torch.ones(*shape, 1, device=DEV), bp, 0.0)
    params = sc.BottleneckParams(ksizes, DEV, seed=seed)
    x = torch.randn(*shape, C, device=DEV, generator=torch.Generator(DEV).manual_seed(seed))

    def layer(t):
        with torch.no_grad():
            return sc.sparse_res_block_bottleneck(t, params, ind, bp, [1, 1, 1, 1], False, use_var=True)

    return layer, x, layer(x.clone())


def test_layers_share_no_scratch_between_calls():
    """The stacks between a block's convolutions and the map of the base's gradient are tensors of the call, not a buffer kept
    for the stream: another thread on the stream, or a captured graph, would find another call's values in it."""
    layer, x, want = residual_layer(1)
    base = torch.zeros(1, 16, 16, 4, device=DEV, requires_grad=True)
    idx = torch.tensor([[0, 0, 0], [0, 1, 1]], dtype=torch.int16, device=DEV)
    y = sbnet_amd.sparse_scatter(torch.ones(2, 8, 8, 4, device=DEV), [2], idx, base, [8, 8], [8, 8], [0, 0], add=False)
    ops.release_workspaces()
    assert torch.equal(layer(x.clone()), want)
    torch.autograd.grad(y, base, torch.ones_like(y))
    assert not ops._load_native().has_workspaces()


def test_layers_from_two_threads_on_one_stream():
    work = [residual_layer(seed) for seed in (1, 2)]
    wrong = []

    def run(layer, x, want):
        for _ in range(100):
            if not torch.equal(layer(x.clone()), want):
                wrong.append(1)

    threads = [threading.Thread(target=run, args=w) for w in work]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


def test_captured_layers_own_their_stacks():
    """Two layers captured on one stream, replayed side by side, after the eager calls' scratch has been given back."""
    work = [residual_layer(seed) for seed in (1, 2)]
    side = torch.cuda.Stream()
    graphs = []
    for layer, x, _ in work:
        t, g = x.clone(), torch.cuda.CUDAGraph()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            layer(x.clone())
        torch.cuda.synchronize()
        with torch.cuda.graph(g, stream=side):
            layer(t)
        graphs.append((t, g, torch.cuda.Stream()))
    ops.release_workspaces()
    held = [torch.full((1 << 20,), 7.0, device=DEV) for _ in range(8)]
    for _ in range(4):
        for (t, _, _), (_, x, _) in zip(graphs, work):
            t.copy_(x)
        torch.cuda.synchronize()
        for _, g, stream in graphs:
            with torch.cuda.stream(stream):
                g.replay()
        torch.cuda.synchronize()
        for (t, _, _), (_, _, want) in zip(graphs, work):
            assert torch.equal(t, want)
    assert all(bool((h == 7.0).all()) for h in held)
