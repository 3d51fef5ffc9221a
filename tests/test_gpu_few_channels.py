"""Convolutions with a handful of output channels on the vector units (csrc/conv_few.h): the tile engine's bits.

The engine's matrix instruction is a chain of fused multiply-adds in the order of the reduction; a product of the same
operands through DLGpuMatrixMultiply, whose reduction is not a multiple of four, runs that chain on it."""
import numpy as np
import pytest

from test_gpu_conv import _check_conv_case, _describe, _gpu

pytestmark = pytest.mark.gpu

# (N, C, H, W, K, R, S, padding, u, v): every size of the kernel (4, 6, 8 channels; 3, 5, 7 taps), whole planes in one
# workgroup (several images, the last group not full), planes in spans, strides, tap rows unlike columns, channels in
# more than one LDS fill, one output channel
CASES = [
    (1000, 6, 14, 14, 16, 5, 5, "VALID", 1, 1),   # grad-data: 6 channels of 196 pixels
    (1030, 1, 28, 28, 6, 5, 5, "SAME", 1, 1),     # forward: 6 channels in spans; grad-data: 1 channel
    (520, 3, 11, 10, 5, 3, 3, "SAME", 2, 2),      # two images a workgroup
    (511, 7, 7, 9, 8, 3, 3, "VALID", 1, 1),       # four, an odd number of images
    (40, 5, 61, 59, 4, 7, 7, "VALID", 1, 1),
    (70, 3, 33, 130, 7, 3, 7, "SAME", 1, 2),
    (260, 8, 20, 20, 60, 3, 3, "SAME", 1, 1),     # grad-data with 60 source channels, reduction of 540: the engine's
    (260, 8, 20, 20, 50, 3, 3, "SAME", 1, 1),     # 50 source channels: several fills
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(str(v) for v in c))
def test_against_the_oracle(rt, monkeypatch, case):
    monkeypatch.setenv("TINYFLOW_WINOGRAD", "0")
    _check_conv_case(rt, case)


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(str(v) for v in c))
def test_bits_of_the_tile_engine(rt, monkeypatch, case):
    """Forward against the product of the filter with the gathered patches on the engine, image by image."""
    from tinyflow_amd import gpu_op, ndarray
    from oracle import ops as O
    monkeypatch.setenv("TINYFLOW_WINOGRAD", "0")
    N, C, H, W, K, R, S, padding, u, v = case
    out_shape, lst = gpu_op.convolution_2d_forward_get_out_shape((N, C, H, W), (K, C, R, S), "NCHW", padding, u, v)
    described = _describe(lst, 0)
    if "gemm_kernel<%d, %d, false>" % (4 if K <= 4 else 6 if K <= 6 else 8, S) not in described or " s1 " not in described:
        pytest.skip("forward of this layer runs on the engine")
    rng = np.random.RandomState(3)
    x = rng.normal(0, 1, (N, C, H, W)).astype(np.float32)
    w = rng.normal(0, 0.3, (K, C, R, S)).astype(np.float32)
    y = ndarray.empty(out_shape, rt.ctx)
    assert gpu_op.convolution_2d_forward(_gpu(x, rt), _gpu(w, rt), y, lst, rt.cudnn, rt.stream) == 0
    y = y.asnumpy()
    ph, pw = O.conv_pad(R, padding), O.conv_pad(S, padding)
    xp = np.pad(x, ((0, 0), (0, 0), (ph, ph), (pw, pw)))
    P, Q = out_shape[2:]
    for n in (0, N // 2, N - 1):
        patches = np.empty((C, R, S, P, Q), np.float32)
        for r in range(R):
            for s in range(S):
                patches[:, r, s] = xp[n, :, r:r + u * (P - 1) + 1:u, s:s + v * (Q - 1) + 1:v]
        c = ndarray.empty((K, P * Q), rt.ctx)
        gpu_op.matrix_multiply(_gpu(w.reshape(K, -1), rt), False, _gpu(patches.reshape(C * R * S, P * Q), rt), False, c,
                               rt.cublas, rt.stream)
        assert c.asnumpy().tobytes() == y[n].reshape(K, -1).tobytes()


def test_which_kernel_runs(rt):
    from tinyflow_amd import gpu_op

    def kernels(case):
        N, C, H, W, K, R, S, padding, u, v = case
        _, lst = gpu_op.convolution_2d_forward_get_out_shape((N, C, H, W), (K, C, R, S), "NCHW", padding, u, v)
        return [_describe(lst, which).split(" | ")[1] for which in (0, 1)]
    assert kernels((1000, 1, 28, 28, 6, 5, 5, "SAME", 1, 1)) == ["gemm_kernel<6, 5, false>", "gemm_kernel<4, 5, true>"]
    assert kernels((1000, 6, 14, 14, 16, 5, 5, "VALID", 1, 1))[1] == "gemm_kernel<6, 5, true>"
    for case in ((1000, 6, 14, 14, 9, 5, 5, "VALID", 1, 1),       # nine output channels
                 (1000, 4, 14, 14, 6, 5, 5, "VALID", 1, 1),       # a reduction of a multiple of four
                 (64, 3, 14, 14, 6, 5, 5, "VALID", 1, 1),         # fewer workgroups than CUs
                 (1000, 23, 14, 14, 6, 5, 5, "VALID", 1, 1)):     # a reduction of more than 512
        assert kernels(case)[0].count("<") > 1, case
