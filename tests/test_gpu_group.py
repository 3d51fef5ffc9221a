"""Groups of elementwise nodes (csrc/group.hip): the bytes of the separate calls, what is refused, and which nodes the executor
puts into one launch."""
import numpy as np
import pytest


def _values(shape, seed):
    gen = np.random.default_rng(seed)
    a = gen.standard_normal(shape, dtype=np.float32)
    flat = a.reshape(-1)
    flat[::7], flat[3::11] = 0.0, -0.0
    if flat.size > 20:
        flat[5::13], flat[6::17] = np.nan, -np.inf
    return a


# one element, remainders of a vector and of a workgroup, rows and planes that are and are not multiples of four
@pytest.mark.gpu
@pytest.mark.parametrize("shape,per_channel", [
    ((1, 1), False), ((3, 5), False), ((2, 4), False), ((128, 100), False), ((129, 10), False), ((64, 1030), False),
    ((2, 3, 5, 7), True), ((4, 6, 28, 28), True), ((5, 4, 2, 2), True), ((3, 1, 1, 1), True), ((7, 16, 10, 10), True),
], ids=str)
def test_group_writes_the_bytes_of_the_separate_calls(rt, shape, per_channel):
    from tinyflow_amd import gpu_op as G, ndarray
    ctx, stream = rt.ctx, rt.stream
    x, dy, bias = _values(shape, 1), _values(shape, 2), _values((shape[1],), 3)
    gx, gdy, gb = (ndarray.array(v, ctx) for v in (x, dy, bias))

    def outputs(n):
        arrays = [ndarray.empty(shape, ctx) for _ in range(n)] + [ndarray.empty((1,), ctx)]
        for a in arrays:
            G.array_set(a, 7.0, stream)
        return arrays

    spread, total, relu, scaled, one = outputs(4)
    G.broadcast_to(gb, spread, "NCHW" if per_channel else "NHWC", stream)
    G.matrix_elementwise_add(gx, spread, total, stream)
    G.relu_on_stream(total, relu, stream)
    G.matrix_elementwise_multiply_by_const(relu, -1.7, scaled, stream)
    G.array_set(one, 1.0, stream)
    grad, shifted, product, both, _ = outputs(4)
    G.relu_gradient_on_stream(total, gdy, grad, stream)
    G.matrix_elementwise_add_by_const(grad, 0.0, shifted, stream)
    G.matrix_elementwise_multiply(shifted, gx, product, stream)
    G.matrix_elementwise_add(scaled, product, both, stream)
    want = [a.asnumpy().tobytes() for a in (spread, total, relu, scaled, one, grad, shifted, product, both)]

    for ordered in (0, 1):
        spread, total, relu, scaled, one = outputs(4)
        grad, shifted, product, both, _ = outputs(4)
        for rows in ([(G.GROUP_BROADCAST, 0, gb, None, spread), (G.GROUP_ADD, 0, gx, spread, total),
                      (G.GROUP_RELU, 0, total, None, relu), (G.GROUP_MUL_CONST, -1.7, relu, None, scaled),
                      (G.GROUP_SET, 1.0, None, None, one)],
                     [(G.GROUP_RELU_GRADIENT, 0, total, gdy, grad), (G.GROUP_ADD_CONST, 0.0, grad, None, shifted),
                      (G.GROUP_MUL, 0, shifted, gx, product), (G.GROUP_ADD, 0, scaled, product, both)]):
            G.elementwise_group(_steps(G, rows, per_channel), ordered, stream)
        got = [a.asnumpy().tobytes() for a in (spread, total, relu, scaled, one, grad, shifted, product, both)]
        assert [g == w for g, w in zip(got, want)] == [True] * len(want)


def _alias(start, like):
    """What looks like an array of the shape of `like` at the address of `start`, for calls that refuse it before anything is read."""
    import ctypes
    from types import SimpleNamespace
    from tinyflow_amd.ndarray import DLArray
    view = DLArray.from_buffer_copy(like.handle.contents)
    view.data = start.handle.contents.data
    return SimpleNamespace(handle=ctypes.pointer(view))


def _steps(G, rows, per_channel=False):
    steps = (G.GroupStep * len(rows))()
    for step, (kind, value, a, b, out) in zip(steps, rows):
        step.kind, step.value, step.per_channel, step.out = kind, value, per_channel, out.handle
        if a is not None:
            step.a = a.handle
        if b is not None:
            step.b = b.handle
    return steps


@pytest.mark.gpu
def test_group_refuses_what_it_cannot_order(rt):
    from tinyflow_amd import gpu_op as G, ndarray
    a, b, c = (ndarray.array(np.full((4, 8), v, np.float32), rt.ctx) for v in (1, 2, 3))
    short = ndarray.array(np.ones((4, 4), np.float32), rt.ctx)
    turned, four = ndarray.array(np.ones((8, 4), np.float32), rt.ctx), ndarray.array(np.ones(4, np.float32), rt.ctx)
    one = ndarray.array(np.ones(1, np.float32), rt.ctx)
    long_at_one = _alias(one, a)   # longer than the step's result at the same address
    add = G.GROUP_ADD_CONST
    for rows in ([(G.GROUP_SET, 1.0, None, None, one), (add, 1.0, a, None, b), (add, 1.0, long_at_one, None, c)],
                 [(add, 1.0, a, None, b), (G.GROUP_SET, 1.0, None, None, one), (G.GROUP_MUL, 0.0, a, long_at_one, c)],
                 [(add, 1.0, a, None, b), (add, 1.0, c, None, b)],          # written twice
                 [(add, 1.0, a, None, b), (add, 1.0, c, None, a)],          # a later step writes what an earlier one read
                 [(add, 1.0, a, None, a)],                                  # in place
                 [(add, 1.0, a, None, b), (add, 1.0, short, None, c)],      # lengths
                 [(add, 1.0, turned, None, b)], [(G.GROUP_RELU_GRADIENT, 0.0, a, turned, b)],   # shapes of one length
                 [(G.GROUP_BROADCAST, 0.0, four, None, b)], [(G.GROUP_BROADCAST, 0.0, short, None, b)],   # not the trailing dims
                 [(99, 1.0, a, None, b)], [(G.GROUP_ADD, 0.0, a, None, b)],
                 [(add, 1.0, a, None, b)] * 7):
        with pytest.raises(RuntimeError):
            G.elementwise_group(_steps(G, rows), 0, rt.stream)
    assert (a.asnumpy() == 1).all() and (b.asnumpy() == 2).all() and (c.asnumpy() == 3).all()


@pytest.mark.gpu
@pytest.mark.parametrize("net,head,optimizer", [("mlp", "softmax_xent", "sgd"), ("lenet5", "softmax_xent", "sgd"),
                                                ("lenet5", "cross", "adam")])
def test_steps_with_groups_have_the_bytes_of_steps_without(rt, monkeypatch, net, head, optimizer):
    from tinyflow_amd import TrainExecute, TrainExecuteAdam, models
    results = []
    for grouped in (True, False):
        if not grouped:
            monkeypatch.setattr(TrainExecute, "find_groups", lambda *a: {})
        rng = np.random.RandomState(11)
        model = getattr(models, net)(rng, batch=96, head=head)
        X, y = models.synthetic_batch(rng, model.input_shape, model.n_class, "uniform")
        module = TrainExecuteAdam if optimizer == "adam" else TrainExecute
        executor = module.TrainExecutor(model.loss, 1e-3)
        executor.init_Variable(dict(model.variables))
        for _ in range(3):
            out = executor.run({model.X: X, model.y_: y})
        results.append([o.asnumpy().tobytes() for o in out]
                       + [executor.value_of(n).asnumpy().tobytes() for n in executor.topo_order
                          if n in executor.node_to_arr_map])
        executor.close()
    assert results[0] == results[1]


def test_which_nodes_form_a_group():
    from tinyflow_amd import autodiff as ad
    from tinyflow_amd.TrainExecute import find_groups, find_joins
    x, b, dy = ad.Placeholder("x"), ad.Variable("b"), ad.Placeholder("dy")
    spread = ad.broadcastto_op(b, x)
    s = x + spread
    r = ad.activation_forward_op(s, "NCHW", "relu")
    t = ad.activation_forward_op(r, "NCHW", "tanh")       # no step of a group
    back = ad.activation_backward_op(s, t, r, "relu", r.cudnnlist)
    ones = ad.oneslike_op(back)
    order = [x, b, dy, spread, s, r, t, back, ones]
    shapes = {n: (8, 12) for n in order}
    shapes[b], shapes[ones] = (12,), (1,)
    fed = {x, b, dy}
    joins = find_joins(order, shapes, fed, {})
    assert find_groups(order, shapes, fed, {}, {}) == {spread: [spread, s, r, ones]}
    # the sum has a fed operand and joins nothing; where it joined, the group would take both, and leave both without the operand
    assert find_groups(order, shapes, fed, {}, {s: r}) == {spread: [spread, s, r, ones]}
    assert find_groups(order, shapes, fed | {spread}, {}, {s: r}) == {} and joins == {}
    # the gradient waits for its upstream, which comes behind the ReLU
    back2 = ad.activation_backward_op(s, dy, r, "relu", r.cudnnlist)
    shifted = back2 + 2.0
    order = [x, b, dy, spread, s, r, t, back2, shifted]
    shapes.update({back2: (8, 12), shifted: (8, 12)})
    assert find_groups(order, shapes, fed, {}, {}) == {spread: [spread, s, r, back2, shifted]}
    assert find_groups(order, shapes, fed, {s: ("skip",), r: ("add_relu", s, [x, spread])}, {}) == {back2: [back2, shifted]}
    shapes.update({n: (2 ** 12, 2 ** 12) for n in (spread, s, r, back2, shifted)})
    assert find_groups(order, shapes, fed, {}, {}) == {}   # too long


def test_nodes_of_unequal_shapes_are_left_to_their_own_calls():
    """An adjoint of as many elements in another shape: ``ReluGradient`` refuses it, the activation's backward pass takes it."""
    from tinyflow_amd import autodiff as ad
    from tinyflow_amd.TrainExecute import find_groups
    x, dy = ad.Placeholder("x"), ad.Placeholder("dy")
    for gradient in (lambda: ad.relu_gradient_op(x, dy), lambda: ad.activation_backward_op(x, dy, x, "relu", [None])):
        g = gradient()
        shifted = g + 2.0
        doubled = shifted * 2.0
        order = [x, dy, g, shifted, doubled]
        for shape, expected in (((8, 12), {g: [g, shifted, doubled]}), ((12, 8), {shifted: [shifted, doubled]})):
            shapes = {n: (8, 12) for n in order}
            shapes[dy] = shape
            assert find_groups(order, shapes, {x, dy}, {}, {}) == expected


@pytest.mark.gpu
def test_a_steps_constants_are_those_of_their_nodes_now(rt):
    """A program may set ``const_attr`` between two steps, as it may where the node has a launch of its own."""
    from tinyflow_amd import autodiff as ad, gpu_op
    from tinyflow_amd.TrainExecute import TrainExecutor, find_groups
    x, w, y_ = ad.Placeholder("x"), ad.Variable("w"), ad.Placeholder("y_")
    h = ad.matmul_op(x, w)
    scaled = h * 2.0
    shifted = scaled + 0.5
    rng = np.random.RandomState(5)
    X, W = rng.normal(0, 1, (6, 5)).astype(np.float32), rng.normal(0, 1, (5, 4)).astype(np.float32)
    Y = np.eye(4, dtype=np.float32)[rng.randint(0, 4, 6)]
    executor = TrainExecutor(ad.softmaxcrossentropy_op(shifted, y_), 0.0)
    executor.init_Variable({w: W})
    for factor, term in ((2.0, 0.5), (-3.0, 0.25)):
        scaled.const_attr, shifted.const_attr = factor, term
        executor.run({x: X, y_: Y})
        groups = find_groups(executor.topo_order, executor.node_to_shape_map, {x, w, y_}, {}, {})
        assert any(scaled in g and shifted in g for g in groups.values())
        got = executor.value_of(h).asnumpy()
        assert (executor.value_of(shifted).asnumpy() == got * np.float32(factor) + np.float32(term)).all()
    executor.close()


def test_a_groups_call_keeps_its_arrays():
    """They live as long as the plan, whatever becomes of the executor's map of them, as those of other plan entries do."""
    import weakref
    from types import SimpleNamespace
    from tinyflow_amd import autodiff as ad, ndarray
    from tinyflow_amd.TrainExecute import _group_compute

    class Array(SimpleNamespace):
        pass
    x = ad.Placeholder("x")
    shifted = x + 1.0
    doubled = shifted * 2.0
    shapes = {n: (3, 4) for n in (x, shifted, doubled)}
    arrays = {n: Array(handle=ndarray.DLArrayHandle(ndarray.DLArray())) for n in shapes}
    alive = [weakref.ref(a) for a in arrays.values()]
    compute = _group_compute([shifted, doubled], shapes, arrays)
    arrays.clear()
    assert all(a() is not None for a in alive)
    del compute
    assert all(a() is None for a in alive)
