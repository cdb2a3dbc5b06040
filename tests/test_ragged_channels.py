"""Planar stacks gathered from tensors whose channel counts or addresses make no 16-byte vectors, against the oracle: counts around
the vectors of four and the chunks of 32 channels, blocks over the border."""
import numpy as np
import pytest
import torch

import sbnet_amd
from oracle import sbnet_oracle as orc

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def dev(a, misaligned=False):
    t = torch.from_numpy(np.ascontiguousarray(a)).to(DEV)
    if not misaligned:
        return t
    flat = torch.empty(t.numel() + 1, device=DEV)     # aligned to 4 bytes only
    m = flat[1:].view(t.shape)
    m.copy_(t)
    return m


@pytest.mark.parametrize("C", [1, 2, 3, 4, 5, 6, 7, 18, 31, 32, 33, 34, 35, 129])
@pytest.mark.parametrize("bs,bst", [((2, 2), (2, 2)), ((7, 6), (5, 4)), ((25, 27), (25, 27)), ((25, 27), (23, 27))],
                         ids=lambda v: "x".join(map(str, v)))
def test_ragged_channels(C, bs, bst):
    N, H, W, bo = 2, 53, 60, (-1, -2)
    rng = np.random.default_rng(C + bs[0])
    bc = [1 + (H - bo[0] - 1) // bst[0], 1 + (W - bo[1] - 1) // bst[1]]
    cells = np.array([(n, i, j) for n in range(N) for i in range(bc[0]) for j in range(bc[1])], np.int16)
    for M in {len(cells) * 2 // 5, min(len(cells), 400)}:
        idx = cells[rng.permutation(len(cells))[:M]]
        x = rng.standard_normal((N, H, W, C)).astype(np.float32)
        for mis in (False, True):
            for count in (M, M - 1):                  # on the host; on the device, with a row past it
                cnt = torch.tensor([count], dtype=torch.int32, device="cpu" if count == M else DEV)
                msg = "M %d misaligned %s count %d" % (M, mis, count)
                got = sbnet_amd.sparse_gather(dev(x, mis), cnt, dev(idx), bs, bst, bo, transpose=True)[:count]
                want = orc.sparse_gather(x, [count], idx, bs, bst, bo, transpose=True)[:count]
                np.testing.assert_array_equal(got.cpu().numpy(), want, err_msg=msg)
