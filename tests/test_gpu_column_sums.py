"""Column sums whose chunks are folded by one lane per column (at most 16 chunks) or by a workgroup (more)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# one column and a few, column counts around a workgroup's, one to some hundred chunks of rows; sums of small integers are
# exact in any order
@pytest.mark.parametrize("rows,cols", [(1, 5), (33, 3), (63, 64), (64, 65), (130, 257), (1000, 1), (1000, 6), (1000, 10),
                                       (1000, 84), (1001, 120), (999, 16), (4096, 63), (5000, 1030), (40000, 7),
                                       (300, 30011)], ids=str)
def test_column_sums_of_integers_are_exact(rt, rows, cols):
    from tinyflow_amd import gpu_op, ndarray
    x = np.random.default_rng(rows + cols).integers(-9, 10, (rows, cols)).astype(np.float32)
    out = ndarray.empty((cols,), rt.ctx)
    gpu_op.array_set(out, np.nan, rt.stream)
    gpu_op.reduce_sum_axis_zero(ndarray.array(x, rt.ctx), out)
    assert np.array_equal(out.asnumpy(), x.sum(axis=0, dtype=np.float64))


@pytest.mark.parametrize("shape", [(1000, 6, 28, 28), (1000, 16, 10, 10), (64, 6, 5, 7), (7, 130, 3, 3)], ids=str)
def test_bias_gradients_of_integers_are_exact(rt, shape):
    from tinyflow_amd import gpu_op, ndarray
    x = np.random.default_rng(shape[0]).integers(-3, 4, shape).astype(np.float32)
    rows, planes = ndarray.empty(shape[1:], rt.ctx), ndarray.array(x, rt.ctx)
    gpu_op.reduce_sum_axis_zero(planes, rows)
    assert np.array_equal(rows.asnumpy(), x.sum(axis=0, dtype=np.float64))
