"""The sum over many pieces of a short result keeps its order: a grad-filter of one input channel against the same pieces added in
index order (matmul.hip: split_sum_tiles_kernel)."""
import numpy as np
import pytest

from oracle import ops as O
from test_gpu_conv import _describe, _gpu

pytestmark = pytest.mark.gpu


# one piece, fewer than a round of 512, and two rounds; filters of a length that is no multiple of four
@pytest.mark.parametrize("images", [20, 64, 336, 1000])
def test_grad_filter_of_many_pieces(rt, images):
    from tinyflow_amd import gpu_op, ndarray
    rng = np.random.RandomState(images)
    x = rng.normal(0, 1, (images, 1, 28, 28)).astype(np.float32)
    w = rng.normal(0, 1, (6, 1, 5, 5)).astype(np.float32)
    dy = rng.normal(0, 1, (images, 6, 28, 28)).astype(np.float32)
    _, lst = gpu_op.convolution_2d_forward_get_out_shape(x.shape, w.shape, "NCHW", "SAME", 1, 1)
    pieces = int(_describe(lst, 2).split(" | ")[0].split(" s")[1])
    assert pieces == 1 or (pieces > 32 and (pieces > 512) == (images > 64))
    dw = ndarray.empty(w.shape, rt.ctx)
    results = []
    for _ in range(2):
        gpu_op.array_set(dw, np.nan, rt.stream)
        assert gpu_op.convolution_backward_filter(_gpu(x, rt), _gpu(dy, rt), _gpu(w, rt), dw, lst, rt.cudnn, rt.stream) == 0
        results.append(dw.asnumpy())
    assert results[0].tobytes() == results[1].tobytes()
    ref = O.conv2d_backward_filter(x.astype(np.float64), dy.astype(np.float64), w.shape, 2, 2, 1, 1)
    # an fp32 sum of n terms in any order: gamma_n times the sum of the magnitudes
    bound = O.conv2d_backward_filter(np.abs(x).astype(np.float64), np.abs(dy).astype(np.float64), w.shape, 2, 2, 1, 1)
    assert (np.abs(results[0] - ref) <= (images * 784 / pieces + pieces + 8) * 2.0 ** -24 * bound).all()
