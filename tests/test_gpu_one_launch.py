"""Column sums and softmax cross entropy whose second pass runs in the launch of the first."""
import numpy as np
import pytest


def _column_sum(x, rows_per_chunk):
    """The order of the additions, in float32: four sums over every fourth row of a chunk, the rest of it on the first, then the chunks."""
    total = np.zeros(x.shape[1], np.float32)
    for a in range(0, len(x), rows_per_chunk):
        chunk = x[a:a + rows_per_chunk]
        whole = len(chunk) // 4 * 4
        s = [np.zeros(x.shape[1], np.float32) for _ in range(4)]
        for i in range(len(chunk)):
            s[i % 4 if i < whole else 0] += chunk[i]
        total += (s[0] + s[1]) + (s[2] + s[3])
    return total


# one chunk; two; a wave of slots and one chunk more; a short last chunk; the most chunks and one row past them; columns that leave
# lanes idle and one past a workgroup's
@pytest.mark.gpu
@pytest.mark.parametrize("rows,cols", [(8, 5), (9, 16), (33, 17), (512, 10), (521, 1), (1000, 84), (2047, 33), (2048, 15), (2049, 15),
                                       (300, 4095)])
def test_column_sums_add_in_the_order_of_two_passes(rt, rows, cols):
    from tinyflow_amd import gpu_op, ndarray
    x = np.random.default_rng(rows).standard_normal((rows, cols), dtype=np.float32)
    gx, out = ndarray.array(x, rt.ctx), ndarray.empty((cols,), rt.ctx)
    gpu_op.array_set(out, 7.0, rt.stream)
    real_in, real_out = gpu_op.reduce_sum_get_real_shape(x.shape, (cols,), "NHWC")
    lst = gpu_op.reduce_sum_get_cudnnlist(real_in, real_out, "NCHW", rt.cudnn)
    assert gpu_op.reduce_sum_new(gx, out, lst, rt.cudnn, rt.stream) == 0
    chunks = min(-(-4 * 256 // -(-cols // 256)), -(-rows // 8))   # four workgroups on each of 256 compute units, or eight rows each
    assert out.asnumpy().tobytes() == _column_sum(x, -(-rows // chunks)).tobytes()


# the first and the last number of rows in one launch and one past it; one to sixteen columns and one past them
@pytest.mark.gpu
@pytest.mark.parametrize("rows", [16, 17, 64, 65, 255, 256, 257])
@pytest.mark.parametrize("cols", [1, 10, 16, 17])
def test_softmax_cross_entropy_against_float64(rt, rows, cols):
    """A row's term is a difference of values of the size of its largest logit, good to a few rounding steps; the mean adds at most
    rows / 16 + 16 in a chain."""
    from tinyflow_amd import gpu_op, ndarray
    rng = np.random.default_rng(rows * 31 + cols)
    x = (rng.standard_normal((rows, cols)) * 4).astype(np.float32)
    t = rng.random((rows, cols), dtype=np.float32)
    out = ndarray.empty((1,), rt.ctx)
    gpu_op.softmax_cross_entropy(ndarray.array(x, rt.ctx), ndarray.array(t, rt.ctx), out, rt.stream)
    x64, t64 = x.astype(np.float64), t.astype(np.float64)
    shifted = x64 - x64.max(axis=1, keepdims=True)
    terms = t64 * (np.log(np.exp(shifted).sum(axis=1, keepdims=True)) - shifted)
    steps = (8 + cols + rows / 16 + 16) * 2.0 ** -24
    bound = steps * (terms + t64 * (1 + np.abs(shifted))).sum() / rows
    assert abs(float(out.asnumpy()[0]) - terms.sum() / rows) <= bound
    x[-1, 0] = np.nan
    gpu_op.softmax_cross_entropy(ndarray.array(x, rt.ctx), ndarray.array(t, rt.ctx), out, rt.stream)
    assert np.isnan(out.asnumpy()[0])


# as many rows as one launch takes, and columns that leave a wave's lanes idle, beside the same with a column of no weight, which two
# launches take
@pytest.mark.gpu
@pytest.mark.parametrize("rows", [17, 63, 64, 65, 130, 255, 256])
@pytest.mark.parametrize("cols", [1, 3, 10, 16])
def test_softmax_cross_entropy_of_one_launch_has_the_bytes_of_two(rt, rows, cols):
    """Logits of -1e30 add the exponential zero and, with labels of zero, nothing to the loss.  Seventeen columns still fall to one lane
    each, so the sums are the same ones."""
    from tinyflow_amd import gpu_op, ndarray
    rng = np.random.default_rng(rows * 17 + cols)
    x = (rng.standard_normal((rows, cols)) * 4).astype(np.float32)
    t = rng.random((rows, cols), dtype=np.float32)
    wide_x, wide_t = np.full((rows, 17), -1e30, np.float32), np.zeros((rows, 17), np.float32)
    wide_x[:, :cols], wide_t[:, :cols] = x, t
    results = []
    for logits, labels in ((x, t), (wide_x, wide_t)):
        out = ndarray.empty((1,), rt.ctx)
        gpu_op.array_set(out, 7.0, rt.stream)
        gpu_op.softmax_cross_entropy(ndarray.array(logits, rt.ctx), ndarray.array(labels, rt.ctx), out, rt.stream)
        results.append(out.asnumpy().tobytes())
    assert results[0] == results[1]
