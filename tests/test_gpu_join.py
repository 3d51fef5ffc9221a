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


# per activation: the register kernels of 32, 64 and 128 rows, full and not, and rows past the last of them, which take the two
# calls; columns that do not fill a workgroup.  Spatial: channels that one workgroup holds, and the last one, which it does not
@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["pre_activation", "spatial"])
@pytest.mark.parametrize("shape", [(1, 3, 5, 7), (31, 4, 9, 9), (32, 16, 16, 16), (33, 5, 11, 3), (64, 3, 17, 5),
                                   (65, 2, 8, 8), (128, 3, 6, 7), (129, 3, 6, 7), (130, 2, 33, 35)], ids=str)
def test_batch_norm_with_relu_writes_the_bytes_of_the_separate_calls(rt, shape, mode):
    from tinyflow_amd import gpu_op, ndarray
    ctx, cudnn, stream = rt.ctx, rt.cudnn, rt.stream
    gen = np.random.default_rng(5)
    x, dy = (gen.standard_normal(shape, dtype=np.float32) for _ in range(2))
    x[0, 0] = 2.5
    x[:, 1, 0, 0] = 0.75   # a column of equal values: bn(x) is zero
    dy[0, 0, 0, :2] = [np.nan, -0.0]
    gx, gdy = ndarray.array(x, ctx), ndarray.array(dy, ctx)
    results = []
    for joined in (False, True):
        act = gpu_op.activation_get_cudnnlist(shape, "NCHW", "relu")
        mean_p, var_p, lst = gpu_op.bn_get_cudnnlist(shape, "NCHW", mode)
        out = [ndarray.empty(shape, ctx) for _ in range(4)]
        for step in range(2):
            for arr in out:
                gpu_op.array_set(arr, 7.0, stream)
            bn, relu, drelu, dx = out
            if joined:
                assert gpu_op.bn_and_relu_forward(gx, bn, relu, mode, step, mean_p, var_p, lst, act, cudnn, stream) == 0
                assert gpu_op.bn_and_relu_backward(gx, bn, relu, gdy, drelu, dx, mode, mean_p, var_p, lst, act, cudnn,
                                                   stream) == 0
            else:
                assert gpu_op.bn_forward(gx, bn, mode, step, mean_p, var_p, lst, cudnn, stream) == 0
                gpu_op.activation_forward(bn, relu, "relu", act, cudnn, stream)
                gpu_op.activation_backward(bn, drelu, relu, gdy, "relu", act, cudnn, stream)
                assert gpu_op.bn_backward(gx, drelu, dx, mode, mean_p, var_p, lst, cudnn, stream) == 0
            results.append([arr.asnumpy().tobytes() for arr in out])
    assert results[0] == results[1] == results[2] == results[3]


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


def test_which_batch_norms_join():
    """A batch norm of either mode joins its ReLU, the ReLU's gradient that batch norm's gradient, and not the gradient of
    another batch norm."""
    from tinyflow_amd import autodiff as ad
    from tinyflow_amd.TrainExecute import find_joins
    x, y, dr = ad.Placeholder("x"), ad.Placeholder("y"), ad.Placeholder("dr")
    for mode in ("pre_activation", "spatial"):
        b = ad.bn_forward_op(x, "NCHW", mode)
        r = ad.activation_forward_op(b, "NCHW", "relu")
        a = ad.activation_backward_op(b, dr, r, "relu", r.cudnnlist)
        d = ad.bn_backward_op(x, a, mode, b.Save_p, b.cudnnlist)
        b2 = ad.bn_forward_op(y, "NCHW", mode)
        d2 = ad.bn_backward_op(y, a, mode, b2.Save_p, b2.cudnnlist)
        joins = {b: r, a: d}
        order = [x, y, dr, b, b2, r, a, d, d2]
        shapes = {n: (2, 3, 4, 4) for n in order}
        assert find_joins(order, shapes, set(), {}) == joins
        assert find_joins([x, y, dr, b, b2, r, a, d2], shapes, set(), {}) == {s: t for s, t in joins.items() if s is b}
        assert find_joins(order, shapes, {b}, {}) == {}   # fed: nothing to compute
