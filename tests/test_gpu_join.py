"""A residual sum with the ReLU behind it, and the adjoints' sum with the ReLU's gradient, as one pass each."""
import numpy as np
import pytest

from oracle import ops as O


def _values(n, seed):
    gen = np.random.default_rng(seed)
    a, b = gen.standard_normal((2, n), dtype=np.float32)
    a[::7], b[::7] = 1.5, -1.5       # sums of exactly zero
    a[3::11], b[3::11] = -0.0, -0.0  # and a negative zero
    a[5::13] = np.nan
    b[6::17] = -np.inf
    return a, b


# below and at the size from which sign bits are kept (2^16); a length that is no multiple of four; one workgroup's 4096
# elements with one vector less and more
@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 4, 4092, 4100, 65532, 65536, 65541, 69628, 69636, 3 * 4096 * 97 + 8])
def test_join_writes_the_bytes_of_the_separate_calls(rt, n):
    from tinyflow_amd import gpu_op, ndarray
    ctx, cudnn, stream = rt.ctx, rt.cudnn, rt.stream
    lst = gpu_op.activation_get_cudnnlist((n,), "NCHW", "relu")
    with np.errstate(invalid="ignore"):
        for step in range(3):
            a, b = _values(n, 2 * step)
            c, d = _values(n, 2 * step + 1)
            ga, gb, gc, gd = (ndarray.array(v, ctx) for v in (a, b, c, d))
            total, out, dtotal, dx = (ndarray.empty((n,), ctx) for _ in range(4))
            for arr in (total, out, dtotal, dx):
                gpu_op.array_set(arr, 7.0, stream)
            counts = gpu_op.relu_mask_counts()
            gpu_op.add_activation_forward(ga, gb, total, out, lst, cudnn, stream)
            gpu_op.add_activation_backward(gc, gd, dtotal, total, dx, out, lst, cudnn, stream)
            bits = 1 if step and n >= 65536 and n % 4 == 0 else 0
            assert gpu_op.relu_mask_counts() == (counts[0] + bits, counts[1] + bits)
            want = (a + b, O.relu(a + b), c + d, O.relu_gradient(a + b, c + d))
            for arr, expected in zip((total, out, dtotal, dx), want):
                got, number = arr.asnumpy(), ~np.isnan(expected)
                assert np.array_equal(got, expected, equal_nan=True)
                assert np.array_equal(np.signbit(got)[number], np.signbit(expected)[number])


@pytest.mark.gpu
def test_join_in_place_and_with_foreign_bits(rt):
    """The sum written over the ReLU's input or output, and a backward call whose input is not the array the kept bits
    describe, give what the separate calls give."""
    from tinyflow_amd import gpu_op, ndarray
    ctx, cudnn, stream = rt.ctx, rt.cudnn, rt.stream
    n = 70000
    lst = gpu_op.activation_get_cudnnlist((n,), "NCHW", "relu")
    gen = np.random.default_rng(3)
    a, b, c, d, other = gen.standard_normal((5, n), dtype=np.float32)
    out, dx = ndarray.empty((n,), ctx), ndarray.empty((n,), ctx)
    for _ in range(2):
        ga, gb, gc, gd = (ndarray.array(v, ctx) for v in (a, b, c, d))
        gpu_op.add_activation_forward(ga, gb, ga, out, lst, cudnn, stream)   # the sum over its operand
        assert ga.asnumpy().tobytes() == (a + b).tobytes() and out.asnumpy().tobytes() == O.relu(a + b).tobytes()
        gother = ndarray.array(other, ctx)
        gpu_op.add_activation_backward(gc, gd, gd, gother, dx, out, lst, cudnn, stream)
        assert gd.asnumpy().tobytes() == (c + d).tobytes()
        assert dx.asnumpy().tobytes() == O.relu_gradient(other, c + d).tobytes()
        gd = ndarray.array(d, ctx)
        gpu_op.add_activation_backward(gc, gd, ga, ga, dx, out, lst, cudnn, stream)   # the sum over the ReLU's input
        assert dx.asnumpy().tobytes() == O.relu_gradient(c + d, c + d).tobytes()
        gpu_op.add_activation_forward(gc, gd, out, out, lst, cudnn, stream)   # the ReLU over the sum
        assert out.asnumpy().tobytes() == O.relu(c + d).tobytes()


def test_which_sums_join():
    """A sum joins one ReLU; not where it is fed or applied as a constant, where the ReLU's gradient needs a later
    operand, or where a fused role has it."""
    from tinyflow_amd import autodiff as ad
    from tinyflow_amd.TrainExecute import find_joins
    x, y = ad.Placeholder("x"), ad.Placeholder("y")
    s = x + y
    r = ad.activation_forward_op(s, "NCHW", "relu")
    tanh = ad.activation_forward_op(x + x, "NCHW", "tanh")
    g = y + r
    back = ad.activation_backward_op(s, g, r, "relu", r.cudnnlist)
    shapes = {n: (2, 3) for n in (x, y, s, r, tanh, tanh.inputs[0], g, back)}
    order = [x, y, s, r, tanh.inputs[0], tanh, g, back]
    assert find_joins(order, shapes, set(), {}) == {s: r, g: back}
    assert find_joins(order, shapes, {s}, {}) == {g: back}
    assert find_joins(order, shapes, set(), {s: ("skip",), r: ("add_relu", s, [x, y]),
                                             back: ("mask_from_output", s, [r, g, r])}) == {g: back}
    assert find_joins([x, y, s, r, g, back], {**shapes, y: (1,)}, set(), {}) == {}
    late = ad.activation_forward_op(tanh, "NCHW", "relu")   # the mask's array is computed after the sum
    back2 = ad.activation_backward_op(tanh, g, late, "relu", late.cudnnlist)
    shapes.update({late: (2, 3), back2: (2, 3)})
    order = [x, y, s, r, g, tanh.inputs[0], tanh, late, back2]
    assert find_joins(order, shapes, set(), {}) == {s: r}
