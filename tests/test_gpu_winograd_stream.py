"""Transformed inputs so large that their stores go past the caches (csrc/conv.hip, launch_wino_input)."""
import numpy as np
import pytest

import parity
from test_gpu_conv import _check_conv_case, _gpu


# 36 values a tile, 256 channels and 3 136 tiles are 116 MB, and twice that with grad-filter's form: rows of whole and of half vectors
# and of neither, on the side of the input and of the output gradient; 2 940 tiles, whose planes' rows start inside a line, go past
# the caches for products on slices alone
@pytest.mark.gpu
@pytest.mark.parametrize("engine", ["0", "1"])
@pytest.mark.parametrize("case", [(16, 256, 56, 56, 16), (16, 16, 56, 56, 256), (16, 256, 55, 54, 16), (16, 16, 55, 54, 256),
                                  (16, 256, 54, 55, 16), (16, 16, 54, 55, 256), (15, 256, 56, 56, 16), (15, 16, 54, 55, 256)], ids=str)
def test_large_transformed_inputs(rt, monkeypatch, case, engine):
    from tinyflow_amd import gpu_op, ndarray
    monkeypatch.setenv("TINYFLOW_WINOGRAD", "4")
    monkeypatch.setenv("TINYFLOW_SPLIT", engine)
    N, C, H, W, K = case
    _check_conv_case(rt, (N, C, H, W, K, 3, 3, "SAME", 1, 1))
    # the later steps of a descriptor share the passes over x and dy: the bytes of the first
    rng = np.random.RandomState(parity.stable_seed(case))
    x, w, dy = (rng.normal(0, 1, s).astype(np.float32) for s in ((N, C, H, W), (K, C, 3, 3), (N, K, H, W)))
    gx, gw, gdy = _gpu(x, rt), _gpu(w, rt), _gpu(dy, rt)
    y, dx, dw = (ndarray.empty(s, rt.ctx) for s in (dy.shape, x.shape, w.shape))
    _, lst = gpu_op.convolution_2d_forward_get_out_shape(x.shape, w.shape, "NCHW", "SAME", 1, 1)
    steps = []
    for _ in range(3):
        for out in (y, dx, dw):
            gpu_op.array_set(out, 7.0, rt.stream)
        assert gpu_op.convolution_2d_forward(gx, gw, y, lst, rt.cudnn, rt.stream) == 0
        assert gpu_op.convolution_backward_data(gx, gdy, gw, dx, lst, rt.cudnn, rt.stream) == 0
        assert gpu_op.convolution_backward_filter(gx, gdy, gw, dw, lst, rt.cudnn, rt.stream) == 0
        steps.append([o.asnumpy().tobytes() for o in (y, dx, dw)])
    assert steps[0] == steps[1] == steps[2]
