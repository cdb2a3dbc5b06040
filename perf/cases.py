"""Timing cases: what a program built on sbnet_amd has it do, through its public entry points.

Four kinds of case:

* pipeline    mask -> reduce_mask -> sparse_gather -> sparse_scatter[_var], the three ops as a network runs them once
              per frame.  The program's own layers sit between gather and scatter, so the stack that is scattered is
              part of the state.
* overlap     sparse_scatter_var(add, atomic) of overlapping blocks onto a base: accumulating detection windows.
* conv, res   the layers of sbnet_amd.sparse_conv: mask -> index list, then `depth` sparse convolutions or sparse
              bottleneck residual blocks on it, the first into a new tensor and the others in place on that (inference).
* train_ops,  forward and backward: of the gather and the copying scatter around a program's own layers, and of a
  train_res   whole sparse residual block with batch statistics.

Masks are what such programs have: road-like strokes (lidar birds-eye views), ellipses (detected objects), independent
cells (attention maps).  Everything is float32, the only type the ops take.
"""
import math

import torch

import sbnet_amd
from sbnet_amd import sparse_conv

DEVICE = "cuda:0"


# ---------------------------------------------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------------------------------------------

def _pipeline(name, shape, bsize, stride, offset, out, mask, density, avgpool=False, transpose=False, add=False,
              var=False, host_count=True, tol=0.5):
    """`out`: "same" scatters blocks of the gather's geometry; "valid" the centre of a 3x3 VALID convolution."""
    N, H, W, C = shape
    return dict(name=name, kind="pipeline", n=N, h=H, w=W, c=C, bh=bsize[0], bw=bsize[1], sh=stride[0], sw=stride[1],
                oh=offset[0], ow=offset[1], out=out, mask=mask, density=density, avgpool=avgpool, transpose=transpose,
                add=add, var=var, host_count=host_count, tol=tol)


def _layers(name, kind, shape, mid, bsize, mask, density, transpose, depth=1, k=3):
    N, H, W, C = shape
    return dict(name=name, kind=kind, n=N, h=H, w=W, c=C, mid=mid, bh=bsize, bw=bsize, mask=mask, density=density,
                transpose=transpose, depth=depth, k=k)


def listed():
    return [
        # The smallest step (plumbing-sized feature map, default layout, copying scatter): launches and host time.
        _pipeline("tiny_step", (1, 64, 64, 16), (10, 10), (8, 8), (-1, -1), "same", "cells", 0.5),
        # One lidar birds-eye-view frame at 30 % block density, planar stack, written back in place.
        _pipeline("bev_dense", (1, 800, 800, 128), (27, 27), (25, 25), (-1, -1), "same", "roads", 0.30,
                  transpose=True, var=True),
        # The same frame nearly empty, default layout, count left on the device.
        _pipeline("bev_sparse_nhwc", (1, 800, 800, 128), (27, 27), (25, 25), (-1, -1), "same", "roads", 0.05,
                  var=True, host_count=False),
        # A batch of mid-sized maps with average pooling, the convolution's output added to a copy of the input.
        _pipeline("ellipses_add", (4, 256, 256, 64), (18, 18), (16, 16), (-1, -1), "valid", "ellipses", 0.08,
                  avgpool=True, transpose=True, add=True, tol=0.05),
        # Many small images, many small blocks.
        _pipeline("small_images", (64, 128, 128, 32), (6, 6), (4, 4), (-1, -1), "valid", "cells", 0.33, avgpool=True,
                  transpose=True, add=True, tol=0.05),
        # Odd everything: channels no vector width divides, blocks that straddle the borders, gaps between blocks.
        _pipeline("odd_channels", (3, 301, 203, 15), (9, 13), (10, 14), (-3, -2), "same", "cells", 0.4,
                  transpose=True),
        # Overlapping windows accumulated into a large base; the largest case.
        dict(name="overlap_add", kind="overlap", n=2, h=512, w=512, c=256, bh=16, bw=16, sh=8, sw=8, density=0.25,
             transpose=False),
        # Forward and backward of the two block ops around a program's own layers, at one of the sizes the
        # reference times its ops on.
        dict(name="train_ops", kind="train_ops", n=1, h=300, w=480, c=256, bh=18, bw=18, sh=16, sw=16, oh=-1, ow=-1,
             mask="ellipses", density=0.3, avgpool=False, tol=0.5, transpose=True, add=False),
        # Two sparse 3x3 convolutions of a ResNet stage, default layout.
        _layers("conv_stage", "conv", (1, 200, 350, 48), 0, 17, "roads", 0.15, False, depth=2),
        # Three sparse bottleneck blocks of the first and of the last ResNet stage, inference.
        _layers("res_stage_first", "res", (1, 400, 700, 96), 24, 17, "roads", 0.10, True, depth=3),
        _layers("res_stage_last", "res", (1, 50, 88, 512), 128, 9, "ellipses", 0.3, False, depth=3),
        # Training step of one bottleneck block.  Planar stack, as everywhere for this kind: on a drawn size with an
        # NHWC stack (1x40x45x384, 15x15 blocks) the process ended with a segmentation fault that is not explained.
        _layers("train_res", "train_res", (1, 100, 175, 256), 64, 11, "ellipses", 0.2, True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _channels(rng, hi):
    """Mostly the multiples of 8 that networks use, now and then any number."""
    if rng.random() < 0.25:
        return _log_int(rng, 1, hi)
    return min(hi, 8 * max(1, _log_int(rng, 8, hi) // 8))


MOST_BYTES = 1.2e9   # of the listed cases' largest


def draw(rng):
    while True:
        kind = rng.choice(["pipeline"] * 5 + ["overlap", "train_ops", "conv", "res", "train_res"])
        if kind in ("pipeline", "train_ops"):
            c = dict(kind=kind, n=_log_int(rng, 1, 16), h=_log_int(rng, 48, 800), w=_log_int(rng, 48, 800),
                     c=_channels(rng, 256), bh=rng.randint(6, 32), mask=rng.choice(["cells", "roads", "ellipses"]),
                     density=round(math.exp(rng.uniform(math.log(0.03), math.log(0.5))), 3),
                     transpose=rng.random() < 0.5)
            c["bw"] = c["bh"] if rng.random() < 0.7 else rng.randint(6, 32)
            step = rng.choice(["halo", "halo", "tile", "gap"])   # 3x3 convolution blocks, tiles, blocks with gaps
            d = {"halo": -2, "tile": 0, "gap": rng.randint(1, 3)}[step]
            c["sh"], c["sw"] = c["bh"] + d, c["bw"] + d
            c["oh"] = c["ow"] = -1 if step == "halo" else rng.choice([0, -1, -2])
            if kind == "pipeline":
                c.update(out="valid" if step == "halo" and rng.random() < 0.6 else "same",
                         avgpool=rng.random() < 0.4, var=rng.random() < 0.5, host_count=rng.random() < 0.75)
                c["tol"] = 0.05 if c["avgpool"] else 0.5
                c["add"] = rng.random() < 0.5 and (c["out"] == "valid" or step != "halo")
            else:
                c.update(add=rng.random() < 0.5 and step != "halo", avgpool=False, tol=0.5)
        elif kind == "overlap":
            s = rng.randint(4, 16)
            c = dict(kind=kind, n=_log_int(rng, 1, 8), h=_log_int(rng, 64, 600), w=_log_int(rng, 64, 600),
                     c=_channels(rng, 256), bh=rng.randint(s + 1, 2 * s), sh=s, sw=s,
                     density=round(rng.uniform(0.05, 0.5), 3), transpose=rng.random() < 0.5)
            c["bw"] = c["bh"]
        else:
            stage = rng.choice([(400, 700, 96, 24), (200, 350, 192, 48), (100, 175, 256, 64), (50, 88, 384, 96),
                                (400, 700, 128, 32), (100, 175, 384, 96), (50, 88, 512, 128)])
            s = math.exp(rng.uniform(math.log(0.5), 0.0))
            c = dict(kind=kind, n=1, h=max(40, int(stage[0] * s)), w=max(40, int(stage[1] * s)),
                     c=stage[3] if kind == "conv" else stage[2], mid=0 if kind == "conv" else stage[3],
                     bh=rng.randint(7, 24), mask=rng.choice(["roads", "ellipses"]),
                     density=round(math.exp(rng.uniform(math.log(0.03), math.log(0.4))), 3),
                     transpose=rng.random() < 0.5 or kind == "train_res",
                     depth=rng.randint(1, 3) if kind != "train_res" else 1,
                     k=rng.choice([3, 3, 5, 1]) if kind == "conv" else 3)
            c["bw"] = c["bh"]
            if _layer_geometry(c) is None:
                continue
        if kind in ("pipeline", "train_ops") and not _budget_fits(c):
            continue
        if 4 * c["n"] * c["h"] * c["w"] * c["c"] <= 4.2e8 and work(c)["bytes"] <= MOST_BYTES and work(c)["flops"] <= 2e11:
            return c


# ---------------------------------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------------------------------

def _layer_geometry(case):
    """Block parameters as sbnet_amd.block_params gives them, or None where it refuses the sizes."""
    size = [case["n"], case["h"], case["w"], case["c"]]
    bsize, k = [1, case["bh"], case["bw"], 1], case["k"]
    try:
        return sbnet_amd.calc_block_params(size, bsize, [k, k, case["c"], case["c"]], [1, 1, 1, 1], "SAME")
    except ValueError:
        return None


def _grid(case):
    """bcount, bsize, bstride, boffset of a case that states its geometry."""
    oh, ow = case.get("oh", 0), case.get("ow", 0)
    return ([sbnet_amd.calc_block_count_covering(case["h"], oh, case["sh"]),
             sbnet_amd.calc_block_count_covering(case["w"], ow, case["sw"])],
            [case["bh"], case["bw"]], [case["sh"], case["sw"]], [oh, ow])


def _score(case, gen, ys, xs):
    """[N, len(ys), len(xs)]: the lower, the more a place matters.  Roads: the distance to a polyline that wanders through
    the image; ellipses: the normalised distance to the nearest of six centres; cells: independent values, images of a
    batch with more and with less."""
    N, H, W = case["n"], case["h"], case["w"]
    if case["mask"] == "cells":
        busy = torch.empty(N, 1, 1, device=DEVICE).uniform_(0.1, 1.0, generator=gen)
        return torch.rand(N, len(ys), len(xs), device=DEVICE, generator=gen) / busy
    yy, xx = ys.view(1, -1, 1), xs.view(1, 1, -1)

    def uniform(lo, hi):
        return torch.empty(N, 1, 1, device=DEVICE).uniform_(lo, hi, generator=gen)

    best = torch.full((N, len(ys), len(xs)), math.inf, device=DEVICE)
    if case["mask"] == "ellipses":
        for _ in range(6):
            cy, cx, ry, rx = uniform(0, H), uniform(0, W), uniform(0.5, 1.5), uniform(0.5, 1.5)
            best = torch.minimum(best, ((yy - cy) / ry) ** 2 + ((xx - cx) / rx) ** 2)
    else:
        step = 0.25 * min(H, W)
        py, px, heading = uniform(0, H), uniform(0, W), uniform(0, 2 * math.pi)
        for _ in range(12):
            heading = heading + uniform(-0.8, 0.8)
            dy, dx = step * torch.sin(heading), step * torch.cos(heading)
            t = (((yy - py) * dy + (xx - px) * dx) / (step * step)).clamp_(0, 1)
            best = torch.minimum(best, (yy - py - t * dy) ** 2 + (xx - px - t * dx) ** 2)
            py, px = (py + dy) % H, (px + dx) % W
    return best


def _pixel_mask(case, gen):
    """float32 [N,H,W,1] of zeros and ones, `density` of the pixels set.  The number of active blocks follows from it
    and is another for every seed."""
    H, W = case["h"], case["w"]
    score = _score(case, gen, torch.arange(H, device=DEVICE).float(), torch.arange(W, device=DEVICE).float()).view(-1)
    count = max(1, int(round(case["density"] * score.numel())))
    return (score <= score.kthvalue(count).values).float().view(case["n"], H, W, 1)


def _active(case):
    """Active blocks of a case that names its share of the blocks."""
    bcount = _grid(case)[0]
    return max(1, int(round(case["density"] * case["n"] * bcount[0] * bcount[1])))


def _own_pixels(case, axis):
    """For each row (axis 0) or column (1) of blocks, the pixels of the image that only its blocks read."""
    bcount, bsize, bstride, boffset = (v[axis] for v in _grid(case))
    size, overlap = (case["h"], case["w"])[axis], max(0, bsize - bstride)
    first = [boffset + i * bstride for i in range(bcount)]
    return [range(max(0, f + overlap), max(0, f + overlap, min(size, f + min(bsize, bstride)))) for f in first]


def _least_share(case):
    return 1.1 * case["tol"] if case["avgpool"] else 1e-6


def _budget_fits(case):
    rows, cols = ([len(own) for own in _own_pixels(case, axis)] for axis in (0, 1))
    least = _least_share(case) * case["bh"] * case["bw"]
    return case["n"] * sum(r * c >= least for r in rows for c in cols) >= _active(case)


def _block_mask(case, gen):
    """float32 [N,H,W,1] that activates `density` of the blocks, as a program does that ranks its blocks and spends a
    budget: in every chosen block those pixels are one that no other block reads.  Blocks of which too little lies in
    the image are not chosen."""
    bcount, bsize, bstride, boffset = _grid(case)
    member, centres = [], []   # member: [size, blocks], which pixels belong to each row or column of blocks alone
    for axis, size in enumerate((case["h"], case["w"])):
        m = torch.zeros(size, bcount[axis])
        for i, own in enumerate(_own_pixels(case, axis)):
            m[own.start:own.stop, i] = 1.0
        member.append(m.to(DEVICE))
        centres.append(boffset[axis] + bstride[axis] * torch.arange(bcount[axis], device=DEVICE).float() + bsize[axis] / 2)
    share = member[0].sum(0).view(-1, 1) * member[1].sum(0).view(1, -1) / (bsize[0] * bsize[1])
    score = _score(case, gen, *centres).masked_fill_(share.unsqueeze(0) < _least_share(case), math.inf)
    chosen = torch.zeros_like(score).view(-1)
    chosen[torch.topk(score.view(-1), _active(case), largest=False).indices] = 1.0
    return (member[0] @ chosen.view_as(score) @ member[1].t()).contiguous().unsqueeze(3)


def _randn(gen, *shape):
    return torch.randn(*shape, device=DEVICE, generator=gen)


def _stack(gen, M, R, S, C, transpose):
    return _randn(gen, *((M, C, R, S) if transpose else (M, R, S, C)))


def prepare(case, seed):
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    kind, C = case["kind"], case["c"]
    shape = (case["n"], case["h"], case["w"], C)
    s = dict(case=case)
    if kind == "pipeline":
        s["bcount"], s["bsize"], s["bstride"], s["boffset"] = _grid(case)
        s["mask"], s["x"] = _block_mask(case, gen), _randn(gen, *shape)
        if case["out"] == "valid":
            s["out_bsize"], s["out_boffset"] = [case["bh"] - 2, case["bw"] - 2], [case["oh"] + 1, case["ow"] + 1]
        else:
            s["out_bsize"], s["out_boffset"] = s["bsize"], s["boffset"]
        s["q"] = _stack(gen, _active(case), *s["out_bsize"], C, case["transpose"])
        s["base"] = s["x"].clone() if case["var"] else s["x"]
    elif kind == "overlap":
        bcount, s["bsize"], s["bstride"], s["boffset"] = _grid(case)
        order = torch.randperm(case["n"] * bcount[0] * bcount[1], device=DEVICE, generator=gen)[:_active(case)].sort().values
        s["indices"] = torch.stack([order // (bcount[0] * bcount[1]), order // bcount[1] % bcount[0], order % bcount[1]], 1).to(torch.int16)
        s["count"] = torch.tensor([len(order)], dtype=torch.int32)
        s["q"] = _stack(gen, len(order), case["bh"], case["bw"], C, case["transpose"])
        s["base"] = torch.zeros(*shape, device=DEVICE)
    elif kind == "train_ops":
        bcount, s["bsize"], s["bstride"], s["boffset"] = _grid(case)
        s["indices"] = sbnet_amd.reduce_mask(_block_mask(case, gen), bcount, s["bsize"], s["bstride"], s["boffset"], tol=0.5)
        stack = (gen, _active(case), case["bh"], case["bw"], C, case["transpose"])
        s["x"], s["q"] = _randn(gen, *shape).requires_grad_(), _stack(*stack).requires_grad_()
        s["dp"], s["dy"] = _stack(*stack), _randn(gen, *shape)
    else:
        s["geometry"] = _layer_geometry(case)
        s["mask"], s["x"] = _pixel_mask(case, gen), _randn(gen, *shape)
        k, mid = case["k"], case["mid"]
        if kind == "conv":
            s["w"] = [_randn(gen, k, k, C, C) / math.sqrt(k * k * C) for _ in range(case["depth"])]
        else:
            ksizes = [[1, 1, C, mid], [k, k, mid, mid], [1, 1, mid, C]]
            s["params"] = [sparse_conv.BottleneckParams(ksizes, DEVICE, seed=seed + i) for i in range(case["depth"])]
            for p in s["params"]:   # statistics and scales of a network that has been trained
                for bn in p.bn:
                    with torch.no_grad():
                        bn.gamma.uniform_(0.5, 1.5, generator=gen)
                        bn.beta.normal_(0.0, 0.2, generator=gen)
                        bn.moving_mean.normal_(0.0, 0.2, generator=gen)
                        bn.moving_var.uniform_(0.5, 1.5, generator=gen)
        if kind == "train_res":
            s["x"].requires_grad_()
            s["dy"] = _randn(gen, *shape)
            s["wanted"] = [s["x"]] + s["params"][0].parameters()
    return s


# ---------------------------------------------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------------------------------------------

def _run_pipeline(s):
    case = s["case"]
    r = sbnet_amd.reduce_mask(s["mask"], s["bcount"], s["bsize"], s["bstride"], s["boffset"], tol=case["tol"],
                              avgpool=case["avgpool"], sync=case["host_count"])
    p = sbnet_amd.sparse_gather(s["x"], r.bin_counts, r.active_block_indices, s["bsize"], s["bstride"], s["boffset"],
                                transpose=case["transpose"])
    scatter = sbnet_amd.sparse_scatter_var if case["var"] else sbnet_amd.sparse_scatter
    y = scatter(s["q"], r.bin_counts, r.active_block_indices, s["base"], s["out_bsize"], s["bstride"], s["out_boffset"],
                add=case["add"], transpose=case["transpose"])
    count = _active(case)   # rows beyond it are not defined
    return [r.bin_counts, r.active_block_indices[:count], p[:count], y]


def _run_train_ops(s):
    case, ind = s["case"], s["indices"]
    p = sbnet_amd.sparse_gather(s["x"], ind.bin_counts, ind.active_block_indices, s["bsize"], s["bstride"],
                                s["boffset"], transpose=case["transpose"])
    y = sbnet_amd.sparse_scatter(s["q"], ind.bin_counts, ind.active_block_indices, s["x"], s["bsize"], s["bstride"],
                                 s["boffset"], add=case["add"], transpose=case["transpose"])
    dx, dq = torch.autograd.grad([p, y], [s["x"], s["q"]], [s["dp"], s["dy"]])
    return [p, y, dx, dq]


def _run_layers(s):
    case, bp, x = s["case"], s["geometry"], s["x"]
    ind = sparse_conv.convert_mask_to_indices_custom(s["mask"], bp, 0.05, avgpool=True)
    strides = [1, 1, 1, 1]
    data_format = "NCHW" if case["transpose"] else "NHWC"
    if case["kind"] == "train_res":
        bn = [t for b in s["params"][0].bn for t in (b.moving_mean, b.moving_var)]
        y = sparse_conv.sparse_res_block_bottleneck(x, s["params"][0], ind, bp, strides, True, data_format=data_format)
        return [y, *torch.autograd.grad(y, s["wanted"], s["dy"]), *bn]
    with torch.no_grad():
        for i in range(case["depth"]):
            if case["kind"] == "conv":
                x = sparse_conv.sparse_conv2d_custom(x, s["w"][i], ind, bp, strides, use_var=i > 0,
                                                     transpose=case["transpose"])
            else:
                x = sparse_conv.sparse_res_block_bottleneck(x, s["params"][i], ind, bp, strides, False,
                                                            data_format=data_format, use_var=i > 0)
    return x


def run(state):
    kind = state["case"]["kind"]
    if kind == "pipeline":
        return _run_pipeline(state)
    if kind == "overlap":
        return sbnet_amd.sparse_scatter_var(state["q"], state["count"], state["indices"], state["base"], state["bsize"],
                                            state["bstride"], state["boffset"], add=True, atomic=True,
                                            transpose=state["case"]["transpose"])
    if kind == "train_ops":
        return _run_train_ops(state)
    return _run_layers(state)


# ---------------------------------------------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------------------------------------------

def work(case):
    """Expected over the masks; a pixel under several blocks counts once on the tensor's side."""
    kind, C = case["kind"], case["c"]
    plane = 4.0 * case["n"] * case["h"] * case["w"]
    if kind in ("conv", "res", "train_res"):
        bp = _layer_geometry(case)
        # a block is active when a twentieth of it is set: half a block more on each side of a set region
        active = min(1.0, 1.5 * case["density"]) * case["n"] * bp.bcount[0] * bp.bcount[1]
        inside = active * bp.bsize_out[0] * bp.bsize_out[1]   # output pixels under blocks
        halo = active * bp.bsize[0] * bp.bsize[1]
        k, mid, depth = case["k"], case["mid"], case["depth"]
        weights = k * k * C * C if kind == "conv" else 2 * C * mid + k * k * mid * mid
        flops = 2.0 * (inside * k * k * C * C if kind == "conv" else halo * C * mid + inside * (k * k * mid * mid + mid * C))
        if kind == "train_res":   # x, dy in; y, dx out, all whole; twice the products again for the two gradients
            return {"bytes": plane * (4 * C + 1) + 8.0 * weights, "flops": 3.0 * flops}
        first = 2 * plane * C   # the first layer's output is a new tensor
        later = (depth - 1) * 4.0 * C * inside * 2
        return {"bytes": plane + first + later + depth * 4.0 * weights, "flops": depth * flops}
    active = _active(case)
    block = 4.0 * C * case["bh"] * case["bw"]
    covered = 4.0 * C * active * min(case["bh"], case["sh"]) * min(case["bw"], case["sw"])
    if kind == "overlap":
        share = 1.0 - (1.0 - case["density"]) ** (case["bh"] * case["bw"] / float(case["sh"] * case["sw"]))
        return {"bytes": active * block + 2 * plane * C * share, "flops": 0}
    if kind == "train_ops":   # x, q, dp, dy in; p, y, dx, dq out
        return {"bytes": 4 * active * block + 4 * plane * C, "flops": 0}
    out = block if case["out"] == "same" else 4.0 * C * (case["bh"] - 2) * (case["bw"] - 2)
    written = min(covered, active * out)
    scatter = active * out + (written * (2 if case["add"] else 1) if case["var"] else
                              plane * C + plane * C - (0 if case["add"] else written))
    return {"bytes": plane + covered + active * block + scatter, "flops": 0}


def tolerance(case):
    """Copies are exact.  Sums of overlapping blocks differ by the order of at most four float32 terms.  Layers: one
    bottleneck block against itself in float64 is off by 4e-7 (max 2e-6) forward, and by up to 1.3e-6 (max 1.3e-5) in a
    gradient, of the same order for any order of the sums; twice that for an algorithm that transforms the products."""
    return {"pipeline": "exact", "overlap": {"rel": 4e-7, "max": 4e-6}, "train_ops": {"rel": 4e-7, "max": 4e-6},
            "conv": {"rel": 3e-6, "max": 3e-5}, "res": {"rel": 3e-6, "max": 3e-5},
            "train_res": {"rel": 8e-6, "max": 8e-5}}[case["kind"]]
