"""Feeding a step from host memory (csrc/feed.hip): every step sees the batch it was given, whatever the caller does with
the host arrays afterwards and however far the host is ahead of the GPU."""
import gc

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ballast(rt):
    from tinyflow_amd import ndarray
    return [ndarray.array(np.full((4096, 4096), 1e-3, np.float32), ctx=rt.ctx) for _ in range(2)] + [
        ndarray.empty((4096, 4096), rt.ctx)]


def _busy(rt, ballast, products):
    """Two thirds of a millisecond each on the stream."""
    from tinyflow_amd import gpu_op
    a, b, c = ballast
    for _ in range(products):
        gpu_op.matrix_multiply(a, False, b, False, c, rt.cublas, rt.stream)


# one element, no multiple of four, the largest feed that a kernel reads from pinned memory (1 MiB) and the next one, more
# than one chunk of the copy stream (4 MiB), several arrays, more than eight of them, arrays that straddle chunks
@pytest.mark.parametrize("busy", [False, True], ids=["idle", "busy"])
@pytest.mark.parametrize("sizes", [[1], [5, 3], [262144], [262145], [2500003], [1 << 21, 7, 4097], [3] * 19,
                                   [300000] * 11], ids=lambda s: "x".join(str(n) for n in s[:3]) + "...%d" % len(s))
def test_arrays_arrive_in_order(rt, ballast, sizes, busy):
    """Seven feeds in a row.  On a stream that is busy for longer than the host needs for all of them, the large ones go
    over the copy stream while it still works, two at a time; on an idle one they are plain copies."""
    from tinyflow_amd import gpu_op, ndarray
    rng = np.random.RandomState(len(sizes))
    targets = [ndarray.empty((n,), rt.ctx) for n in sizes]
    batches = [[rng.uniform(-1, 1, n).astype(np.float32) for n in sizes] for _ in range(7)]
    copies = [[ndarray.empty((n,), rt.ctx) for n in sizes] for _ in batches]
    hosts = [np.empty(n, np.float32) for n in sizes]
    ndarray.reserve_feed(targets, rt.stream)
    before = ndarray.feed_counts()
    for batch, kept in zip(batches, copies):
        for h, values in zip(hosts, batch):   # the same host arrays, overwritten right after the call before
            h[:] = values
        if busy:
            _busy(rt, ballast, 15)   # 10 ms, right in front of the feed; the host is at most two feeds ahead
        ndarray.feed(list(zip(targets, hosts)), rt.stream)
        for h in hosts:
            h[:] = np.nan
        for t, k in zip(targets, kept):
            gpu_op.matrix_elementwise_multiply_by_const(t, 1.0, k, rt.stream)
        if not busy:
            copies[0][0].asnumpy()
    direct, overlapped, synchronous = (a - b for a, b in zip(ndarray.feed_counts(), before))
    if sum(-(-n // 64) * 64 for n in sizes) <= 1 << 18:   # every array starts at a multiple of 256 bytes
        assert (direct, overlapped, synchronous) == (7, 0, 0)
    else:
        assert (direct, overlapped, synchronous) == ((0, 7, 0) if busy else (0, 0, 7))
    for batch, kept in zip(batches, copies):
        for a, b in zip(batch, kept):
            np.testing.assert_array_equal(a, b.asnumpy())


def test_what_is_refused(rt):
    from tinyflow_amd import ndarray
    target = ndarray.empty((4, 5), rt.ctx)
    with pytest.raises(ValueError):
        ndarray.feed([(target, np.zeros((5, 4), np.float32))], rt.stream)
    with pytest.raises(TypeError):
        ndarray.feed([(target, "not an array")], rt.stream)
    ndarray.feed([(target, np.arange(20).reshape(4, 5).tolist())], rt.stream)   # converted, as a synchronous copy would
    np.testing.assert_array_equal(target.asnumpy(), np.arange(20, dtype=np.float32).reshape(4, 5))
    ndarray.feed([], rt.stream)   # nothing to feed
    ndarray.feed([(target, np.ones((4, 5), np.float64).T.copy().T)], rt.stream)   # another type and order
    np.testing.assert_array_equal(target.asnumpy(), np.ones((4, 5), np.float32))


def test_a_feed_waits_for_the_other_streams(rt, ballast):
    """A late kernel of another stream still reads the array that is fed."""
    from tinyflow_amd import gpu_op, ndarray
    stream = gpu_op.create_cudaStream()
    for n in (1000, 2500003):
        target, kept, fed = (ndarray.empty((n,), rt.ctx) for _ in range(3))
        old, new = np.arange(n, dtype=np.float32), -np.arange(n, dtype=np.float32)
        target._sync_copyfrom(old)
        _busy(rt, ballast, 15)
        gpu_op.matrix_elementwise_multiply_by_const(target, 1.0, kept, rt.stream)
        ndarray.feed([(target, new)], stream)
        gpu_op.matrix_elementwise_multiply_by_const(target, 1.0, fed, stream)
        np.testing.assert_array_equal(kept.asnumpy(), old)
        np.testing.assert_array_equal(fed.asnumpy(), new)
    gpu_op.destroy_cudaStream(stream)


@pytest.mark.parametrize("batch", [64, 600], ids=str)   # a feed of 0.2 MB and one of 1.9 MB
def test_steps_equal_those_of_synchronous_feeds(batch):
    """Several executors in turn, batches that change every step; with a device-memory budget the feeds are synchronous."""
    from tinyflow_amd import gpu_op, models
    from tinyflow_amd.TrainExecute import TrainExecutor

    def train(synchronous):
        if synchronous:
            gpu_op.set_device_memory_limit(8 << 30)
        try:
            executors = []
            for seed in (1, 2):
                model = models.lenet5(np.random.RandomState(seed), batch=batch)
                ex = TrainExecutor(model.loss, 1e-4)
                ex.init_Variable(dict(model.variables))
                executors.append((model, ex))
            losses = []
            rng = np.random.RandomState(9)
            X = np.empty(executors[0][0].input_shape, np.float32)
            y = np.zeros((batch, 10), np.float32)
            for step in range(6):
                X[:] = rng.uniform(0, 1, X.shape)
                y[:] = 0
                y[np.arange(batch), rng.randint(0, 10, batch)] = 1
                for model, ex in executors:
                    out = ex.run({model.X: X, model.y_: y})
                    if step in (0, 3, 5):
                        losses.append(out[0].asnumpy())
            weights = [a.asnumpy() for _, ex in executors for a in ex.run({executors[0][0].X: X, executors[0][0].y_: y}
                       if ex is executors[0][1] else {executors[1][0].X: X, executors[1][0].y_: y})[1:]]
            for _, ex in executors:
                ex.close()
            return losses + weights
        finally:
            if synchronous:
                gpu_op.set_device_memory_limit(0)

    for a, b in zip(train(False), train(True)):
        assert a.tobytes() == b.tobytes()


def _held(rt):
    from tinyflow_amd import gpu_op
    return gpu_op.device_memory_stats()[1]


@pytest.mark.parametrize("why", ["no room", "a budget"])
def test_the_buffers_of_feeds_are_given_back(rt, why):
    """Device memory that feeds hold between steps is there for whoever finds no room, and for a budget.  An array of
    4 TiB fits no device, so asking for it is a device without room."""
    from tinyflow_amd import gpu_op, ndarray
    stream = gpu_op.create_cudaStream()
    n = 3000017
    target, kept = ndarray.empty((n,), rt.ctx), ndarray.empty((n,), rt.ctx)
    gc.collect()   # arrays of other tests
    before = _held(rt)
    ndarray.reserve_feed([target], stream)
    assert _held(rt) >= before + 2 * 4 * n
    if why == "no room":
        assert isinstance(ndarray.empty((1 << 40,), rt.ctx), int)
    else:
        gpu_op.set_device_memory_limit(4 << 30)
        gpu_op.set_device_memory_limit(0)
    assert _held(rt) == before
    for step in range(3):   # feeds arrive without it, and take it again only where nobody had to go without
        values = np.full(n, step + 0.5, np.float32)
        values[step] = -1
        ndarray.reserve_feed([target], stream)
        ndarray.feed([(target, values)], stream)
        gpu_op.matrix_elementwise_multiply_by_const(target, 1.0, kept, stream)
        assert kept.asnumpy().tobytes() == values.tobytes()
    if why == "no room":
        assert _held(rt) == before
    else:
        assert _held(rt) >= before + 2 * 4 * n
    gpu_op.destroy_cudaStream(stream)
    assert _held(rt) == before
