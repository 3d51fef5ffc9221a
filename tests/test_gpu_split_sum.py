"""The sum over many pieces of a result adds them in index order (matmul.hip: split_sum_tiles_kernel, split_sum_ordered_kernel)."""
import re

import numpy as np
import pytest

from oracle import ops as O
from test_gpu_conv import _describe, _gpu

pytestmark = pytest.mark.gpu


# one piece, fewer than a round of 512, and two rounds; a filter of a length that is no multiple of four
@pytest.mark.parametrize("images", [20, 64, 336, 1000])
def test_grad_filter_of_many_pieces(rt, images):
    from tinyflow_amd import gpu_op, ndarray
    rng = np.random.RandomState(images)
    x = rng.normal(0, 1, (images, 1, 28, 28)).astype(np.float32)
    w = rng.normal(0, 1, (6, 1, 5, 5)).astype(np.float32)
    dy = rng.normal(0, 1, (images, 6, 28, 28)).astype(np.float32)
    _, lst = gpu_op.convolution_2d_forward_get_out_shape(x.shape, w.shape, "NCHW", "SAME", 1, 1)
    pieces = int(_describe(lst, 2).split(" | ")[0].split(" s")[1])
    assert pieces == 1 if images == 20 else pieces > 128 and (pieces > 512) == (images > 64)
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


# through LDS: one round, two, three, the most values; an element a lane: fewer pieces than values want, too many values, many of both
@pytest.mark.parametrize("case", [(64, 1, 28, 6, 5), (336, 1, 28, 6, 5), (1000, 1, 28, 6, 5), (300, 3, 28, 9, 5), (900, 3, 28, 18, 5),
                                  (100, 7, 40, 19, 3), (16, 5, 56, 13, 7), (64, 23, 28, 27, 5), (100, 9, 28, 33, 5)], ids=str)
def test_pieces_are_added_in_index_order(rt, case):
    """One value in every piece, so that the host knows the pieces, of magnitudes whose float32 sum depends on the order."""
    from tinyflow_amd import gpu_op, ndarray
    images, C, H, K, R = case
    rng = np.random.RandomState(images + C)
    _, lst = gpu_op.convolution_2d_forward_get_out_shape((images, C, H, H), (K, C, R, R), "NCHW", "SAME", 1, 1)
    plan = _describe(lst, 2)
    pieces, stage = int(plan.split(" | ")[0].split(" s")[1]), int(re.search(r"<\d+, \d+, (\d+)", plan).group(1))
    assert "wgrad_pad" in plan and pieces > 32 and K * C * R * R % 4 != 0
    steps = images * H * H
    length = -(-(-(-steps // pieces)) // stage) * stage   # of a piece: whole stages
    assert -(-steps // length) == pieces
    x = np.ldexp(rng.choice([-1.0, 1.0], (images, C, H, H)), rng.randint(-3, 4, (images, C, H, H))).astype(np.float32)
    dy = np.zeros((images, K, H * H), np.float32)
    padded = np.pad(x, ((0, 0), (0, 0), (R // 2, R // 2), (R // 2, R // 2)))
    terms = []
    for at in range(0, steps, length):
        n, pixel = divmod(at, H * H)
        r, c = divmod(pixel, H)
        dy[n, :, pixel] = np.ldexp(rng.uniform(0.5, 1, K), rng.randint(-8, 9, K)).astype(np.float32)
        terms.append(dy[n, :, pixel, None, None, None] * padded[n, :, r:r + R, c:c + R] + np.float32(0))

    def total(terms):
        s = terms[0].copy()
        for t in terms[1:]:
            s += t
        return s
    want = total(terms)
    assert (want != total(terms[::-1])).any()
    dw = ndarray.empty((K, C, R, R), rt.ctx)
    gpu_op.array_set(dw, np.nan, rt.stream)
    assert gpu_op.convolution_backward_filter(_gpu(x, rt), _gpu(dy.reshape(images, K, H, H), rt), _gpu(np.zeros((K, C, R, R), np.float32), rt),
                                              dw, lst, rt.cudnn, rt.stream) == 0
    np.testing.assert_array_equal(dw.asnumpy(), want)

