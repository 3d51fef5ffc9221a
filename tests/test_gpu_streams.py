"""Programs of several streams: the library recycles scratch and arrays between them and lets an executor's update stand
between what other streams enqueued before and after it.

Every result has to be the one that the same calls give when the host waits in between.  ``_busy`` puts some milliseconds
of products on a stream, so that whatever is not ordered behind them runs before them."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


class _Stream(object):
    def __init__(self):
        from tinyflow_amd import gpu_op
        self.cell = gpu_op.create_cudaStream()
        self.cublas = gpu_op.create_cublasHandle(self.cell)

    def close(self):
        from tinyflow_amd import gpu_op
        gpu_op.destroy_cublasHandle(self.cublas)
        gpu_op.destroy_cudaStream(self.cell)


@pytest.fixture
def streams(rt):
    pair = (_Stream(), _Stream())
    yield pair
    for s in pair:
        s.close()


def _array(rt, values):
    from tinyflow_amd import ndarray
    return ndarray.array(np.asarray(values, np.float32), ctx=rt.ctx)


def _empty(rt, shape):
    from tinyflow_amd import ndarray
    return ndarray.empty(shape, rt.ctx)


@pytest.fixture(scope="module")
def ballast(rt):
    return [_array(rt, np.full((4096, 4096), 1e-3)) for _ in range(2)] + [_empty(rt, (4096, 4096))]


def _busy(ballast, stream, products=12):
    from tinyflow_amd import gpu_op
    a, b, c = ballast
    for _ in range(products):
        gpu_op.matrix_multiply(a, False, b, False, c, stream.cublas, stream.cell)


def _product(rt, stream, a, b, out):
    """A product whose reduction is cut up: it takes scratch."""
    from tinyflow_amd import gpu_op
    gpu_op.matrix_multiply(a, False, b, False, out, stream.cublas, stream.cell)
    return out


def _executors(optimizer, n=2):
    from tinyflow_amd import TrainExecute, TrainExecuteAdam, models
    made = []
    for seed in range(n):
        rng = np.random.RandomState(seed)
        model = models.resnet(rng, [1, 1, 1, 1], 16, image=64, n_class=10, bn_mode="pre_activation", width=16)
        module = TrainExecuteAdam if optimizer == "adam" else TrainExecute
        ex = module.TrainExecutor(model.loss, 1e-4)
        ex.init_Variable(dict(model.variables))
        X, y = models.synthetic_batch(rng, (16, 3, 64, 64), 10, "normal")
        ex.run({model.X: X, model.y_: y})
        made.append(ex)
    return made


@pytest.mark.parametrize("optimizer", ["sgd", "adam"])
def test_executors_in_turn_without_feeds(rt, ballast, optimizer):
    """Resident steps: nothing is copied, so no feed orders the streams.  Both executors take the same scratch."""
    from tinyflow_amd import ndarray

    def train(waiting):
        executors = _executors(optimizer)
        losses = []
        for _ in range(5):
            for ex in executors:
                if not waiting:
                    _busy(ballast, _of(ex), 2)
                loss = ex.run({})[0]
                if waiting:
                    loss.asnumpy()
        for ex in executors:
            losses += [a.asnumpy() for a in ex.run({})]
            ex.close()
        return losses

    for a, b in zip(train(False), train(True)):
        assert a.tobytes() == b.tobytes()


def _of(ex):
    s = _Stream.__new__(_Stream)
    s.cell, s.cublas = ex.cudaStream, ex.cublasHandle
    return s


@pytest.mark.parametrize("optimizer", ["sgd", "adam"])
def test_operators_on_another_stream_around_a_step(rt, streams, ballast, optimizer):
    """A reader on another stream after the step sees the updated parameters, one before it those from before (the SGD
    update waits for it; Adam's does not, there the host has to); a product there takes the scratch that the step has just
    given back."""
    from tinyflow_amd import gpu_op
    mine, _ = streams
    ex, = _executors(optimizer, 1)
    weight = ex.value_of(ex.Variable_node_list[-1])
    before, after, old = (_empty(rt, weight.shape) for _ in range(3))
    rng = np.random.RandomState(5)
    a, b = _array(rt, rng.normal(0, 1, (64, 20000))), _array(rt, rng.normal(0, 1, (20000, 64)))
    wanted = _product(rt, mine, a, b, _empty(rt, (64, 64))).asnumpy()
    for _ in range(3):
        old_values = weight.asnumpy()
        _busy(ballast, mine)                       # the reader of the old values is late
        gpu_op.matrix_elementwise_multiply_by_const(weight, 1.0, before, mine.cell)
        if optimizer == "adam":
            before.asnumpy()
        _busy(ballast, _of(ex))                    # the step is late
        ex.run({})
        gpu_op.matrix_elementwise_multiply_by_const(weight, 1.0, after, mine.cell)
        got = _product(rt, mine, a, b, _empty(rt, (64, 64))).asnumpy()
        assert got.tobytes() == wanted.tobytes()
        assert before.asnumpy().tobytes() == old_values.tobytes()
        assert after.asnumpy().tobytes() == weight.asnumpy().tobytes()
        assert weight.asnumpy().tobytes() != old_values.tobytes()
    ex.close()


def test_relu_of_an_executor_stands_between_the_streams(rt, streams, ballast):
    """The ReLU nodes' entry points, which ran on the default stream: behind what other streams hold and in front of
    what they launch next."""
    from tinyflow_amd import gpu_op
    one, two = streams
    x, g, y, dx, seen, dseen = (_empty(rt, (1000,)) for _ in range(6))
    source = np.random.RandomState(1).normal(0, 1, 1000).astype(np.float32)
    src = _array(rt, source)
    for sign in (1.0, -1.0, 1.0):
        _busy(ballast, two)
        gpu_op.matrix_elementwise_multiply_by_const(src, sign, x, two.cell)
        gpu_op.matrix_elementwise_multiply_by_const(src, 3.0 * sign, g, two.cell)
        gpu_op.relu_on_stream(x, y, one.cell)
        gpu_op.relu_gradient_on_stream(x, g, dx, one.cell)
        gpu_op.matrix_elementwise_multiply_by_const(y, 1.0, seen, two.cell)
        gpu_op.matrix_elementwise_multiply_by_const(dx, 1.0, dseen, two.cell)
        want = sign * source
        np.testing.assert_array_equal(seen.asnumpy(), np.maximum(want, 0))
        np.testing.assert_array_equal(dseen.asnumpy(), np.where(want > 0, np.float32(3) * want, np.float32(0)))


@pytest.mark.parametrize("budget", [0, 2 << 30], ids=["pool", "budget"])
def test_scratch_goes_from_one_stream_to_the_other(rt, streams, ballast, budget):
    """The same products on two streams in turn, the first late: the second takes the scratch that the first has given
    back and not yet used."""
    from tinyflow_amd import gpu_op
    rng = np.random.RandomState(2)
    host = [(rng.normal(0, 1, (64, 20000)), rng.normal(0, 1, (20000, 64))) for _ in streams]

    def products():
        pairs = [(_array(rt, a), _array(rt, b)) for a, b in host]
        outs = [[_empty(rt, (64, 64)) for _ in range(6)] for _ in streams]
        wanted = [_product(rt, s, a, b, _empty(rt, (64, 64))).asnumpy() for s, (a, b) in zip(streams, pairs)]
        _busy(ballast, streams[0])
        for step in range(6):
            for s, (a, b), out in zip(streams, pairs, outs):
                _product(rt, s, a, b, out[step])
        return wanted, [[o.asnumpy() for o in out] for out in outs]

    gpu_op.set_device_memory_limit(budget)
    try:
        for want, out in zip(*products()):
            assert all(o.tobytes() == want.tobytes() for o in out)
    finally:
        gpu_op.set_device_memory_limit(0)


def test_an_arrays_storage_goes_from_one_stream_to_the_other(rt, streams, ballast):
    """An array is freed while a late kernel of one stream still has to read it; the next array of that size is written
    on the other stream."""
    from tinyflow_amd import gpu_op
    one, two = streams
    n = 7_340_033   # of no other test: the pool prefers the block that fits best, so it is the one just freed
    values = np.random.RandomState(3).normal(0, 1, n).astype(np.float32)
    for _ in range(3):
        source, kept = _array(rt, values), _empty(rt, (n,))
        address = source.handle.contents.data
        _busy(ballast, one)
        gpu_op.matrix_elementwise_multiply_by_const(source, 1.0, kept, one.cell)
        del source
        fresh = _empty(rt, (n,))
        assert fresh.handle.contents.data == address    # the case that this is about
        gpu_op.array_set(fresh, 7.0, two.cell)
        assert kept.asnumpy().tobytes() == values.tobytes()
        assert (fresh.asnumpy() == 7.0).all()
        del kept, fresh


def test_threads_with_a_stream_each(rt, streams):
    """Each thread's products keep their bits while the other's take and give back scratch of the same size."""
    rng = np.random.RandomState(4)
    pairs = [(_array(rt, rng.normal(0, 1, (64, 20000))), _array(rt, rng.normal(0, 1, (20000, 64)))) for _ in streams]
    wanted = [_product(rt, s, a, b, _empty(rt, (64, 64))).asnumpy() for s, (a, b) in zip(streams, pairs)]
    outs = [[_empty(rt, (64, 64)) for _ in range(150)] for _ in streams]
    failures = []

    def work(s, pair, out):
        try:
            for o in out:
                _product(rt, s, pair[0], pair[1], o)
        except Exception as e:   # shown by the main thread
            failures.append(e)

    threads = [threading.Thread(target=work, args=(s, p, o)) for s, p, o in zip(streams, pairs, outs)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failures
    for want, out in zip(wanted, outs):
        assert all(o.asnumpy().tobytes() == want.tobytes() for o in out)
