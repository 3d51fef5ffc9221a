"""Transformed inputs so large that their stores go past the caches (csrc/conv.hip, launch_wino_input)."""
import numpy as np
import pytest

import parity
from oracle import ops as O
from test_gpu_conv import _gpu


# 36 values a tile, 2 940 tiles and 512 channels are 217 MB, and so are 256 channels with grad-filter's form: rows of whole and of half vectors
# and of neither, on the side of the input and of the output gradient
@pytest.mark.gpu
@pytest.mark.parametrize("case", [(15, 512, 56, 56, 16), (15, 16, 56, 56, 256), (15, 512, 55, 54, 16), (15, 16, 55, 54, 256),
                                  (15, 512, 54, 55, 16), (15, 16, 54, 55, 256)], ids=str)
def test_large_transformed_inputs(rt, monkeypatch, case):
    """Additions of random sign put an error of 2^-24 * sqrt(terms) on a sum, 2.7 times that in this domain at full length; the transforms
    themselves were measured at 2e-6 of the output.  A value out of place is an error of the size of the output."""
    from tinyflow_amd import gpu_op, ndarray
    monkeypatch.setenv("TINYFLOW_WINOGRAD", "4")
    N, C, H, W, K = case
    rng = np.random.RandomState(parity.stable_seed(case))
    x, w, dy = (rng.normal(0, 1, s).astype(np.float32) for s in ((N, C, H, W), (K, C, 3, 3), (N, K, H, W)))
    gx, gw, gdy = _gpu(x, rt), _gpu(w, rt), _gpu(dy, rt)
    y, dx, dw = (ndarray.empty(s, rt.ctx) for s in (dy.shape, x.shape, w.shape))
    _, lst = gpu_op.convolution_2d_forward_get_out_shape(x.shape, w.shape, "NCHW", "SAME", 1, 1)
    steps = []
    for _ in range(3):   # the later steps of a descriptor share the passes over x and dy: the bytes of the first
        for out in (y, dx, dw):
            gpu_op.array_set(out, 7.0, rt.stream)
        assert gpu_op.convolution_2d_forward(gx, gw, y, lst, rt.cudnn, rt.stream) == 0
        assert gpu_op.convolution_backward_data(gx, gdy, gw, dx, lst, rt.cudnn, rt.stream) == 0
        assert gpu_op.convolution_backward_filter(gx, gdy, gw, dw, lst, rt.cudnn, rt.stream) == 0
        steps.append([o.asnumpy().tobytes() for o in (y, dx, dw)])
    assert steps[0] == steps[1] == steps[2]
    ends = [0, N - 1]
    w64, x64, dy64 = w.astype(np.float64), x.astype(np.float64), dy.astype(np.float64)
    for got, ref, terms in ((y.asnumpy()[ends], O.conv2d_forward(x64[ends], w64, 1, 1, 1, 1), 9 * C),
                            (dx.asnumpy()[ends], O.conv2d_backward_data(dy64[ends], w64, x[ends].shape, 1, 1, 1, 1), 9 * K),
                            (dw.asnumpy(), O.conv2d_backward_filter(x64, dy64, w.shape, 1, 1, 1, 1), N * H * W)):
        error = np.linalg.norm(got - ref) / np.linalg.norm(ref)
        assert error <= 2.7 * 2.0 ** -24 * np.sqrt(terms) + 4e-6, error
