"""Spatial batch norm of a channel that fits one workgroup: both passes in one launch, alone and with the ReLU."""
import numpy as np
import pytest


# one to four register slots a lane; one to sixteen chunks; images left over in the last chunk; one lane and one full slot;
# 16-byte and single accesses; and the first sizes past the limit, which two passes take; short rows of many images on both sides of
# the number of images, the size and the length from which on two passes take them
@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(1, 3, 1, 1), (1, 2, 32, 32), (3, 1100, 5, 5), (5, 300, 9, 9), (8, 256, 10, 10),
                                   (4, 256, 56, 56), (8, 128, 20, 20), (2, 90, 31, 33), (7, 600, 16, 16), (16, 16, 8, 8),
                                   (17, 64, 6, 6), (16, 64, 32, 32), (16, 64, 32, 36), (4, 300, 15, 17), (4, 300, 16, 17),
                                   (31, 8500, 1, 3), (32, 8500, 1, 3), (32, 8191, 1, 3), (32, 2000, 4, 4)],
                         ids=str)
def test_against_float64_and_its_joint_form(rt, shape):
    """A lane adds at most 16 values (64 past the limit) in float32 before float64 takes over, which bounds each sum by that
    many rounding steps of the sum of magnitudes; the steps behind add one each."""
    from tinyflow_amd import gpu_op, ndarray
    rng = np.random.default_rng(3)
    x = (rng.standard_normal(shape) * 2 + 0.5).astype(np.float32)
    dy = rng.standard_normal(shape, dtype=np.float32)
    x[:, -1] = 1.25   # no variance: bn(x) is zero, and not above it
    mean_p, var_p, lst = gpu_op.bn_get_cudnnlist(shape, "NCHW", "spatial")
    act = gpu_op.activation_get_cudnnlist(shape, "NCHW", "relu")
    gx, gdy = ndarray.array(x, rt.ctx), ndarray.array(dy, rt.ctx)
    y, dx, y2, relu, drelu, dx2, dx3 = (ndarray.empty(shape, rt.ctx) for _ in range(7))
    for out in (y, dx, y2, relu, drelu, dx2, dx3):
        gpu_op.array_set(out, 7.0, rt.stream)

    def forward():
        assert gpu_op.bn_forward(gx, y, "spatial", 0, mean_p, var_p, lst, rt.cudnn, rt.stream) == 0
    forward()
    assert gpu_op.bn_backward(gx, gdy, dx, "spatial", mean_p, var_p, lst, rt.cudnn, rt.stream) == 0
    assert gpu_op.bn_and_relu_forward(gx, y2, relu, "spatial", 0, mean_p, var_p, lst, act, rt.cudnn, rt.stream) == 0
    assert gpu_op.bn_and_relu_backward(gx, y2, relu, gdy, drelu, dx2, "spatial", mean_p, var_p, lst, act, rt.cudnn,
                                       rt.stream) == 0
    # the joint form has the bytes of the calls that it stands for
    got = y.asnumpy()
    assert y2.asnumpy().tobytes() == got.tobytes() and relu.asnumpy().tobytes() == np.where(got < 0, 0, got).tobytes()
    want_drelu = np.where(got > 0, dy, np.float32(0))
    assert drelu.asnumpy().tobytes() == want_drelu.tobytes()
    forward()
    assert gpu_op.bn_backward(gx, drelu, dx3, "spatial", mean_p, var_p, lst, rt.cudnn, rt.stream) == 0
    assert dx2.asnumpy().tobytes() == dx3.asnumpy().tobytes()

    axes, m, u = (0, 2, 3), x[:, 0].size, 2.0 ** -24

    def over(a):
        return a.sum(axis=axes, keepdims=True)
    x64, g = x.astype(np.float64), dy.astype(np.float64)
    mean, var = x64.mean(axis=axes, keepdims=True), x64.var(axis=axes, keepdims=True) + float(np.float32(1e-5))
    istd, t = 1 / np.sqrt(var), np.abs(x64 - x64[:1, :, :1, :1])
    xhat = (x64 - mean) * istd
    steps = (64 + 3) * u
    rel_istd = steps * (over(t * t) / m + 2 * (over(t) / m) ** 2) / var / 2 + 2 * u
    e_xhat = istd * (steps * over(t) / m + 2 * u * np.abs(mean) + u * np.abs(x64 - mean)) + np.abs(xhat) * (rel_istd + 2 * u)
    assert np.all(np.abs(got - xhat) <= e_xhat)
    for masked, result in ((g, dx), (want_drelu.astype(np.float64), dx2)):
        s1, s2 = over(masked), over(masked * xhat)
        e1 = steps * over(np.abs(masked))
        e2 = steps * over(np.abs(masked * xhat)) + over(np.abs(masked) * e_xhat)
        ref = istd * (masked - s1 / m - xhat * s2 / m)
        bound = istd * (8 * u * (np.abs(masked) + np.abs(s1) / m + np.abs(xhat * s2) / m) +
                        (e1 + np.abs(xhat) * e2 + e_xhat * np.abs(s2)) / m) + rel_istd * np.abs(ref)
        assert np.all(np.abs(result.asnumpy() - ref) <= bound)


@pytest.mark.gpu
@pytest.mark.parametrize("shape,launches", [((32, 8500, 1, 3), 2), ((512, 2048, 1, 1), 2), ((31, 8500, 1, 3), 1), ((32, 8191, 1, 3), 1),
                                            ((32, 2000, 4, 4), 1), ((8, 256, 10, 10), 1)], ids=str)
def test_which_channels_take_one_launch(rt, shape, launches):
    """Two launches keep partial sums, which a forward call that finds no room reports beside the statistics."""
    from tinyflow_amd import gpu_op, ndarray
    gx = ndarray.array(np.ones(shape, np.float32), rt.ctx)
    gy = ndarray.empty(shape, rt.ctx)
    mean_p, var_p, lst = gpu_op.bn_get_cudnnlist(shape, "NCHW", "spatial")
    gpu_op.set_device_memory_limit(max(1, gpu_op.device_memory_stats()[1]))   # nothing more can be allocated
    try:
        wanted = gpu_op.bn_forward(gx, gy, "spatial", 0, mean_p, var_p, lst, rt.cudnn, rt.stream)
    finally:
        gpu_op.set_device_memory_limit(0)
    statistics = 2 * 4 * shape[1]
    assert wanted >= statistics and (wanted >= statistics + shape[1] * (2 * 8 + 4)) == (launches == 2), wanted


def _results(rt, x, dy, offset):
    """y, both statistics, dx and the joint calls' outputs, of arrays that start `offset` elements into an allocation."""
    import ctypes
    from types import SimpleNamespace
    from tinyflow_amd import gpu_op, ndarray
    shape, keep = x.shape, []

    def array(values=None):
        room = ndarray.array(np.full(x.size + offset, 7.0, np.float32), rt.ctx)
        like = ndarray.empty(shape, rt.ctx) if values is None else ndarray.array(values, rt.ctx)
        view = ndarray.DLArray.from_buffer_copy(like.handle.contents)
        view.data = room.handle.contents.data + 4 * offset
        keep.extend((room, like, view))
        inner = ndarray.NDArray(ctypes.pointer(view))
        inner.is_freed = True   # its storage is the room's
        if values is not None:
            gpu_op.matrix_elementwise_add_by_const(like, 0.0, inner, rt.stream)
        return inner
    mean_p, var_p, lst = gpu_op.bn_get_cudnnlist(shape, "NCHW", "spatial")
    act = gpu_op.activation_get_cudnnlist(shape, "NCHW", "relu")
    gx, gdy = array(x), array(dy)
    y, dx, y2, relu, drelu, dx2 = (array() for _ in range(6))
    assert gpu_op.bn_forward(gx, y, "spatial", 0, mean_p, var_p, lst, rt.cudnn, rt.stream) == 0
    statistics = []
    for cell in (mean_p, var_p):
        view = ndarray.DLArray(ctypes.cast(cell, ctypes.POINTER(ctypes.c_void_p))[0], rt.ctx, 1, (ctypes.c_int64 * 1)(shape[1]))
        array_of = ndarray.NDArray(ctypes.pointer(view))
        array_of.is_freed = True
        statistics.append(array_of.asnumpy())
    assert gpu_op.bn_backward(gx, gdy, dx, "spatial", mean_p, var_p, lst, rt.cudnn, rt.stream) == 0
    assert gpu_op.bn_and_relu_forward(gx, y2, relu, "spatial", 0, mean_p, var_p, lst, act, rt.cudnn, rt.stream) == 0
    assert gpu_op.bn_and_relu_backward(gx, y2, relu, gdy, drelu, dx2, "spatial", mean_p, var_p, lst, act, rt.cudnn, rt.stream) == 0
    return [a.asnumpy() for a in (y, dx, y2, relu, drelu, dx2)] + statistics


# slots of a lane's chunk and rounds of chunks: 1 in one to four rounds, 2 in one and two, 3, 4; the last chunk short; rows by
# 16 bytes, by elements, and by elements because of where they lie
@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(8, 256, 10, 10), (16, 16, 8, 8), (17, 64, 6, 6), (16, 64, 32, 32), (8, 64, 40, 40), (2, 90, 31, 33),
                                   (3, 1100, 28, 28), (3, 1100, 15, 17), (4, 256, 45, 40), (4, 256, 56, 56), (5, 300, 9, 9), (1, 3, 1, 1)], ids=str)
@pytest.mark.parametrize("offset", [0, 1])
def test_one_launch_has_the_bytes_of_two_passes(rt, monkeypatch, shape, offset):
    rng = np.random.default_rng(shape[1] + offset)
    x = (rng.standard_normal(shape) * 3 - 1).astype(np.float32)
    dy = rng.standard_normal(shape, dtype=np.float32)
    got = _results(rt, x, dy, offset)
    monkeypatch.setenv("TINYFLOW_SPATIAL_ONE_LAUNCH", "0")
    want = _results(rt, x, dy, offset)
    assert [a.tobytes() == b.tobytes() for a, b in zip(got, want)] == [True] * len(want)
