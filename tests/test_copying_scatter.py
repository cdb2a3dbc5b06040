"""The copying scatter's one-pass kernels against the oracle, by the list, which their workgroups read themselves up to 1536
rows, and by the map that is made of it first for longer ones and some large launches; the gather's gradient by the same kernels."""
import ctypes

import numpy as np
import pytest
import torch

import sbnet_amd
from oracle import sbnet_oracle as orc
from sbnet_amd import _lib

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


NONE, STRIPS, CELLS, REST = range(4)


def route(shape, bs, bst, bo, M, transpose, add, aligned_to=0):
    """How the library goes about a copying scatter: the kernel, whether by the list, the vector width."""
    out = (ctypes.c_int32 * 5)()
    assert _lib.load().sbnet_test_scatter_route((ctypes.c_int32 * 4)(*shape), (ctypes.c_int32 * 6)(*bs, *bst, *bo), M, int(transpose),
                                                int(add), aligned_to, out) == 0
    return tuple(out[:3])


@pytest.mark.parametrize("M", [1, 700, 1536, 1537])
@pytest.mark.parametrize("shape,bs,bst,bo", [
    ((8, 66, 80, 8), (6, 7), (4, 5), (-1, -2)),      # overlap in both directions: 16-byte vectors
    ((8, 66, 80, 6), (6, 4), (4, 4), (-1, 0)),       # in rows only
    ((8, 67, 81, 3), (4, 7), (4, 5), (-2, -3)),      # in columns only; floats of a vector in different pixels
    ((8, 70, 97, 1), (3, 4), (4, 5), (-1, -1)),      # gaps; up to four pixels in a vector, rows that end inside one
    ((8, 70, 97, 18), (3, 4), (4, 6), (2, -1)),
    ((8, 65, 66, 4), (4, 4), (4, 4), (0, 0)),        # planar stack staged in strips
    ((8, 130, 135, 18), (8, 8), (8, 8), (-3, -5)),   # planar stack by cells
    ((8, 140, 135, 130), (4, 5), (6, 7), (0, 0)),    # more channel vectors than a strip that only copies is wide
], ids=lambda v: "x".join(map(str, v)))
def test_copying_scatter_reads_lists_and_maps(shape, bs, bst, bo, M):
    N, H, W, C = shape
    rng = np.random.default_rng(M + C)
    bc = [1 + (H - bo[0] - 1) // bst[0], 1 + (W - bo[1] - 1) // bst[1]]
    cells = np.array([(n, i, j) for n in range(N) for i in range(-1, bc[0] + 1) for j in range(-1, bc[1])], np.int16)
    idx = cells[rng.permutation(len(cells))[:M]]     # some of them reach over the border, some lie outside
    assert len(idx) == M
    idx_d, base = dev(idx), rng.standard_normal(shape).astype(np.float32)
    base_d = dev(base)
    flat = torch.empty(base_d.numel() + 1, device=DEV)
    mis = flat[1:].view(base_d.shape)                # aligned to 4 bytes only
    mis.copy_(base_d)
    overlap = bs[0] > bst[0] or bs[1] > bst[1]
    assert route(shape, bs, bst, bo, M, False, not overlap)[:2] == (STRIPS, M <= 1536)
    planar = route(shape, bs, bst, bo, M, True, not overlap)   # (tiles beside strips by the map: in a test of their own)
    assert planar[:2] in ((STRIPS, M <= 1536), (CELLS, M <= 1536), (REST, 1), (NONE, 0)) and (planar[0] != NONE or M >= 1536)
    for transpose in (False, True):
        stack = rng.standard_normal((M, C, *bs) if transpose else (M, *bs, C)).astype(np.float32)
        stack_d = dev(stack)
        for add in ((False,) if overlap else (False, True)):
            for count in (M, max(1, M - 3)):         # on the host; on the device, with rows past it
                cnt = torch.tensor([count], dtype=torch.int32, device="cpu" if count == M else DEV)
                want = orc.sparse_scatter(stack, [count], idx, base, bs, bst, bo, add=add, transpose=transpose)
                for b in (base_d, mis):
                    y = sbnet_amd.sparse_scatter(stack_d, cnt, idx_d, b, bs, bst, bo, add=add, transpose=transpose)
                    np.testing.assert_array_equal(y.cpu().numpy(), want, err_msg="transpose %s add %s count %d" % (transpose, add, count))


@pytest.mark.parametrize("shape,bs,bo", [((2, 40, 56, 32), (4, 4), (0, 0)), ((2, 50, 41, 24), (13, 15), (0, -1))],
                         ids=["strips", "cells"])
def test_long_lists_that_name_blocks_several_times(shape, bs, bo):
    """Rows that name the same block through the map: the one listed last wins, an add takes all in list order."""
    N, H, W, C = shape
    rng = np.random.default_rng(H)
    bc = [1 + (H - bo[0] - 1) // bs[0], 1 + (W - bo[1] - 1) // bs[1]]
    cells = np.array([(n, i, j) for n in range(N) for i in range(bc[0]) for j in range(bc[1])], np.int16)
    idx = cells[rng.integers(len(cells), size=1600)]
    base = rng.standard_normal(shape).astype(np.float32)
    for transpose in (False, True):
        stack = rng.standard_normal((1600, C, *bs) if transpose else (1600, *bs, C)).astype(np.float32)
        for add in (False, True):
            want = orc.sparse_scatter(stack, [1600], idx, base, bs, bs, bo, add=add, transpose=transpose)
            y = sbnet_amd.sparse_scatter(dev(stack), [1600], dev(idx), dev(base), bs, bs, bo, add=add, transpose=transpose)
            np.testing.assert_array_equal(y.cpu().numpy(), want, err_msg="transpose %s add %s" % (transpose, add))


@pytest.mark.parametrize("shape,bs,bst,bo,M", [
    ((4, 134, 140, 128), (6, 7), (4, 5), (-1, -2), 1600),   # overlap in both directions
    ((4, 150, 150, 126), (8, 5), (5, 5), (-1, 0), 1600),    # in rows only; 8-byte vectors
    ((4, 150, 150, 96), (5, 8), (5, 6), (-2, -3), 2048),    # in columns only
    ((4, 150, 153, 115), (5, 6), (6, 7), (-1, -1), 1900),   # gaps; floats
    ((1, 120, 120, 512), (5, 4), (4, 4), (-1, 0), 600),     # many tiles: a map for a list of few rows
    ((1, 125, 127, 512), (4, 4), (5, 5), (0, -1), 610),
], ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_tiles_and_strips_by_the_map(shape, bs, bst, bo, M):
    N, H, W, C = shape
    rng = np.random.default_rng(C)
    bc = [1 + (H - bo[0] - 1) // bst[0], 1 + (W - bo[1] - 1) // bst[1]]
    cells = np.array([(n, i, j) for n in range(N) for i in range(-1, bc[0] + 1) for j in range(-1, bc[1])], np.int16)
    idx = cells[rng.permutation(len(cells))[:M]]
    assert len(idx) == M
    idx_d, base = dev(idx), rng.standard_normal(shape).astype(np.float32)
    base_d = dev(base)
    mis = torch.empty(base_d.numel() + 1, device=DEV)[1:].view(base_d.shape)   # aligned to 4 bytes only
    mis.copy_(base_d)
    stack = rng.standard_normal((M, C, *bs)).astype(np.float32)
    stack_d = dev(stack)
    overlap = bs[0] > bst[0] or bs[1] > bst[1]
    for add in ((False,) if overlap else (False, True)):
        widths = [route(shape, bs, bst, bo, M, True, add, a) for a in (0, 4)]
        assert widths == [(REST, 0, 4 if C % 4 == 0 else 2 if C % 2 == 0 else 1), (REST, 0, 1)]
        for count in (M, M - 3):
            cnt = torch.tensor([count], dtype=torch.int32, device="cpu" if count == M else DEV)
            want = orc.sparse_scatter(stack, [count], idx, base, bs, bst, bo, add=add, transpose=True)
            for b in (base_d, mis):
                y = sbnet_amd.sparse_scatter(stack_d, cnt, idx_d, b, bs, bst, bo, add=add, transpose=True)
                np.testing.assert_array_equal(y.cpu().numpy(), want, err_msg="add %s count %d" % (add, count))


@pytest.mark.parametrize("shape,bs,bst,bo", [
    ((3, 41, 38, 32), (5, 6), (6, 7), (-1, -2)),       # 16-byte vectors; a list that the workgroups read
    ((3, 41, 38, 6), (5, 6), (5, 7), (-1, 0)),
    ((3, 41, 38, 15), (9, 5), (10, 6), (-3, -2)),
    ((1, 70, 70, 130), (18, 18), (19, 21), (-1, -1)),  # several tiles a block
    ((4, 116, 119, 112), (5, 5), (6, 6), (-2, 0)),     # 1600 rows or more: a map, and chains of rows
    ((4, 116, 119, 110), (5, 5), (6, 6), (-2, 0)),
], ids=lambda v: "x".join(map(str, v)))
def test_repeated_rows_of_planar_blocks_with_gaps(shape, bs, bst, bo):
    """Tiles beside strips that copy the rest: the row listed last wins, an add takes all in list order, exactly."""
    N, H, W, C = shape
    rng = np.random.default_rng(C)
    bc = [1 + (H - bo[0] - 1) // bst[0], 1 + (W - bo[1] - 1) // bst[1]]
    cells = np.array([(n, i, j) for n in range(N) for i in range(-1, bc[0] + 1) for j in range(-1, bc[1])], np.int16)
    long = N * H * W * C > 4e6
    M = 1600 if long else len(cells) // 2
    idx = cells[rng.integers(len(cells), size=M)]
    idx[0] = idx[1] = idx[M // 2] = idx[-1] = cells[len(cells) // 2]
    base = rng.standard_normal(shape).astype(np.float32)
    stack = rng.standard_normal((M, C, *bs)).astype(np.float32)
    flat = torch.empty(base.size + 1, device=DEV)
    mis = flat[1:].view(base.shape)
    mis.copy_(dev(base))
    for add in (False, True):
        assert route(shape, bs, bst, bo, M, True, add)[:2] == route(shape, bs, bst, bo, M, True, add, 4)[:2] == (REST, not long)
        for count in (M, M - 3):
            cnt = torch.tensor([count], dtype=torch.int32, device="cpu" if count == M else DEV)
            want = orc.sparse_scatter(stack, [count], idx, base, bs, bst, bo, add=add, transpose=True)
            for b in (dev(base), mis):
                y = sbnet_amd.sparse_scatter(dev(stack), cnt, dev(idx), b, bs, bst, bo, add=add, transpose=True)
                np.testing.assert_array_equal(y.cpu().numpy(), want, err_msg="add %s count %d" % (add, count))


@pytest.mark.parametrize("M", [1, 1536, 1537])
@pytest.mark.parametrize("shape,bs,bst,bo", [
    ((8, 66, 80, 8), (6, 7), (4, 5), (-1, -2)),       # overlap in both directions
    ((8, 66, 80, 6), (6, 4), (4, 4), (-1, 0)),        # in rows only; 8-byte vectors
    ((8, 67, 81, 3), (4, 7), (4, 5), (-2, -3)),       # in columns only
    ((8, 70, 97, 1), (3, 4), (4, 5), (-1, -1)),       # gaps
    ((8, 140, 135, 132), (4, 5), (6, 7), (0, 0)),     # more channel vectors than a strip of zeros is wide; too large for sums by strips
], ids=lambda v: "x".join(map(str, v)))
@pytest.mark.parametrize("twice", [False, True])
def test_gather_gradient_by_strips(shape, bs, bst, bo, M, twice):
    """The sums in list order, with zeros of either sign, exactly; lists that name blocks twice included up to 1536 rows."""
    from sbnet_amd import ops
    N, H, W, C = shape
    rng = np.random.default_rng(M + C)
    bc = [1 + (H - bo[0] - 1) // bst[0], 1 + (W - bo[1] - 1) // bst[1]]
    cells = np.array([(n, i, j) for n in range(N) for i in range(-1, bc[0] + 1) for j in range(-1, bc[1])], np.int16)
    idx = cells[rng.permutation(len(cells))[:M]]
    if twice:
        idx[-1] = idx[M // 2]
    for transpose in (False, True):
        g = rng.standard_normal((M, C, *bs) if transpose else (M, *bs, C)).astype(np.float32)
        g.reshape(-1)[::5] = -0.0
        want = orc.sparse_scatter(g, [M], idx, np.zeros(shape, np.float32), bs, bst, bo, add=True, atomic=True,
                                  transpose=transpose)
        got = ops.gather_backward(dev(g), [M], dev(idx), shape, list(bs), list(bst), list(bo), transpose).cpu().numpy()
        if twice and M > 1536:     # hardware atomics: five terms below 5 in any order, 2 * 4 * 2^-24 * 25
            np.testing.assert_allclose(got, want, rtol=0, atol=1.2e-5)
        else:
            np.testing.assert_array_equal(got.view(np.int32), want.view(np.int32), err_msg="transpose %s" % transpose)


@pytest.mark.parametrize("shape,bs,bst,bo", [
    ((3, 45, 43, 32), (6, 7), (4, 5), (-1, -2)),       # overlap in both directions
    ((3, 45, 43, 6), (6, 4), (4, 4), (-1, 0)),         # in rows only
    ((3, 45, 43, 15), (4, 7), (4, 5), (-2, -3)),       # in columns only
    ((3, 45, 43, 8), (5, 6), (6, 6), (0, -1)),         # in none
    ((1, 60, 62, 132), (12, 13), (6, 7), (-1, -1)),    # every pixel under four blocks
], ids=lambda v: "x".join(map(str, v)))
@pytest.mark.parametrize("few", [True, False])
def test_gather_gradient_of_lists_with_many_repeats(shape, bs, bst, bo, few):
    """The sums in list order, exactly, with blocks that one, two and more rows name side by side."""
    from sbnet_amd import ops
    N, H, W, C = shape
    rng = np.random.default_rng(C)
    bc = [1 + (H - bo[0] - 1) // bst[0], 1 + (W - bo[1] - 1) // bst[1]]
    cells = np.array([(n, i, j) for n in range(N) for i in range(-1, bc[0] + 1) for j in range(-1, bc[1])], np.int16)
    M = len(cells) * 3 // 4
    idx = cells[rng.permutation(len(cells))[:M]] if few else cells[rng.integers(len(cells), size=M)]
    idx[:3] = idx[-1] = cells[len(cells) // 2]         # one block by four rows, first and last ones among them
    for transpose in (False, True):
        g = rng.standard_normal((M, C, *bs) if transpose else (M, *bs, C)).astype(np.float32)
        g.reshape(-1)[::5] = -0.0
        want = orc.sparse_scatter(g, [M], idx, np.zeros(shape, np.float32), bs, bst, bo, add=True, atomic=True,
                                  transpose=transpose)
        got = ops.gather_backward(dev(g), [M], dev(idx), shape, list(bs), list(bst), list(bo), transpose).cpu().numpy()
        np.testing.assert_array_equal(got.view(np.int32), want.view(np.int32), err_msg="transpose %s" % transpose)
