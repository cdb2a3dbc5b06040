"""Gradients of SparseGather and SparseScatter as torch.autograd.Functions over the C ABI.

The reference registers them in Python as compositions of its own ops
(sbnet_tensorflow/benchmark/sparse_conv_lib.py:80-147, the same text in
sbnet_ops/tests/test_sparse_blocks.py:36-98); the same compositions are used here, so every
backward pass runs the HIP kernels of the forward ops:

* d SparseGather / dx       = sparse_scatter(grad, ..., zeros_like(x), add=True, atomic=True, transpose),
                              computed by one entry point that writes zeros only where no block lies
* d SparseScatter / dblocks = sparse_gather(grad, ...)
* d SparseScatter / dybase  = grad                       (add=True)
                            = grad * stamp-out mask      (add=False; mask = blocks of zeros scattered over ones),
                              in one pass over grad where at most 2x2 blocks cover a pixel

No gradient flows to the index list, the count or the block parameters, as in the reference.

One deliberate difference: the reference calls the gather of d/dblocks without the op's transpose
attribute (sparse_conv_lib.py:124-130), which returns an [M,R,S,C]-shaped gradient for an
[M,C,R,S]-shaped input.  Here the gather uses the forward op's transpose so that the gradient has
the layout of the input; for transpose=False the two coincide.
"""
import torch

from . import ops


def _count_host(bin_counts):
    """The count is read once in forward and kept as a host integer for backward."""
    return ops._count(bin_counts)


# The gradients by the general wrappers: of the functions below, and of the native ones for what those leave to them.
# sizes: M, the block's size, stride and offset, the shape of the NHWC tensor, transpose (bit 0) and add (bit 1), and for the
# scatter the rows of the stack.

def _geometry(sizes):
    return sizes[0], sizes[1:3], sizes[3:5], sizes[5:7], tuple(sizes[7:11]), bool(sizes[11] & 1)


def gather_gradient(grad, idx, sizes):
    M, bsize, bstride, boffset, x_shape, transpose = _geometry(sizes)
    # the reference scatters onto zeros_like(x) with the copying op; the library builds the same tensor without
    # materialising the zeros first (sbnet_sparse_gather_grad)
    return ops.gather_backward(grad.contiguous(), [M], idx, x_shape, bsize, bstride, boffset, transpose)


def scatter_gradients(grad, idx, sizes, wants_blocks, wants_base):
    M, bsize, bstride, boffset, base_shape, transpose = _geometry(sizes)
    grad = grad.contiguous()
    d_blocks = d_ybase = None
    if wants_blocks:
        d_blocks = ops.gather_forward(grad, [M], idx, bsize, bstride, boffset, transpose)
    if wants_base:
        if sizes[11] & 2:
            d_ybase = grad
        elif not (torch.is_grad_enabled() and grad.requires_grad):
            d_ybase = ops.scatter_base_backward(grad, [M], idx, bsize, bstride, boffset)
        if d_ybase is None:   # a graph of the gradients is asked for, or a geometry that the one pass does not take
            stamp = torch.ones_like(grad)
            C = base_shape[3]
            zeros = torch.zeros((sizes[12], C, *bsize) if transpose else (sizes[12], *bsize, C), dtype=torch.float32,
                                device=grad.device)
            ops.scatter_forward(zeros, [M], idx, stamp, bsize, bstride, boffset, add=False, atomic=False,
                                transpose=transpose, use_var=True)
            d_ybase = grad * stamp
    return d_blocks, d_ybase


def _sizes(M, bsize, bstride, boffset, shape, flags):
    pairs = [int(v) for p in (bsize, bstride, boffset) for v in ops._pair(p)[0]]
    return (M, *pairs, *shape, flags)


class SparseGatherFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, bin_counts, active_block_indices, bsize, bstride, boffset, transpose):
        M = _count_host(bin_counts)
        ctx.sizes = _sizes(M, bsize, bstride, boffset, x.shape, int(transpose))
        ctx.save_for_backward(active_block_indices)
        return ops.gather_forward(x.detach(), [M], active_block_indices, bsize, bstride, boffset, transpose)

    @staticmethod
    def backward(ctx, grad):
        return gather_gradient(grad, ctx.saved_tensors[0], ctx.sizes), None, None, None, None, None, None


class SparseScatterFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, bin_counts, active_block_indices, ybase, bsize, bstride, boffset, add, atomic, transpose):
        M = _count_host(bin_counts)
        ctx.sizes = (*_sizes(M, bsize, bstride, boffset, ybase.shape, int(transpose) | int(add) << 1), x.shape[0] if x.dim() else 0)
        ctx.save_for_backward(active_block_indices)
        return ops.scatter_forward(x.detach(), [M], active_block_indices, ybase.detach(), bsize, bstride, boffset,
                                   add, atomic, transpose, use_var=False)

    @staticmethod
    def backward(ctx, grad):
        d_blocks, d_ybase = scatter_gradients(grad, ctx.saved_tensors[0], ctx.sizes, ctx.needs_input_grad[0],
                                              ctx.needs_input_grad[3])
        return d_blocks, None, None, d_ybase, None, None, None, None, None, None
