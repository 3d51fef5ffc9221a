"""Convolutions with a handful of output channels on the vector units (csrc/conv_few.h): the tile engine's bits.

The engine's matrix instruction is a chain of fused multiply-adds in the order of the reduction.
TINYFLOW_FEW_CHANNELS=0 leaves the same layers to the engine, and a product of the same operands through
DLGpuMatrixMultiply, whose reduction is not a multiple of four, runs that chain on it."""
import numpy as np
import pytest

from test_gpu_conv import _check_conv_case, _describe, _gpu

pytestmark = pytest.mark.gpu

# (N, C, H, W, K, R, S, padding, u, v), whether forward and grad-data run on these kernels: every size of them (4, 6, 8
# channels; 3, 5, 7 taps), planes in spans, whole planes of several images in one workgroup with the last group not full,
# strides, tap rows unlike columns, channels in more than one LDS fill, one output channel, folded pieces
CASES = [
    ((1000, 6, 14, 14, 16, 5, 5, "VALID", 1, 1), (False, True)),   # 6 channels of 196 pixels
    ((1030, 1, 28, 28, 6, 5, 5, "SAME", 1, 1), (True, True)),      # 6 channels in spans; 1 channel
    ((520, 3, 11, 10, 5, 3, 3, "SAME", 2, 2), (False, False)),     # too few workgroups
    ((511, 7, 7, 9, 8, 3, 3, "VALID", 1, 1), (False, False)),
    ((2203, 3, 11, 10, 5, 3, 3, "SAME", 2, 2), (True, False)),     # eight images a workgroup, three in the last
    ((1801, 7, 7, 9, 8, 3, 3, "VALID", 1, 1), (True, True)),       # seven and four images a workgroup
    ((4099, 1, 7, 7, 3, 7, 7, "SAME", 1, 1), (True, True)),        # five; more taps than pixels inside
    ((1301, 8, 10, 12, 31, 3, 3, "SAME", 1, 1), (False, True)),    # two, with 31 channels in several fills
    ((2500, 8, 9, 9, 50, 3, 3, "SAME", 1, 1), (False, True)),      # three, with pieces in the last columns
    ((40, 5, 61, 59, 4, 7, 7, "VALID", 1, 1), (True, True)),
    ((70, 3, 33, 130, 7, 3, 7, "SAME", 1, 2), (True, False)),
    ((260, 8, 20, 20, 60, 3, 3, "SAME", 1, 1), (False, False)),    # 60 source channels, reduction of 540: the engine's
    ((260, 8, 20, 20, 50, 3, 3, "SAME", 1, 1), (False, True)),     # 50 source channels: several fills, and pieces
]


@pytest.mark.parametrize("case", [c[0] for c in CASES], ids=lambda c: "x".join(str(v) for v in c))
def test_against_the_oracle(rt, monkeypatch, case):
    monkeypatch.setenv("TINYFLOW_WINOGRAD", "0")
    _check_conv_case(rt, case)


def _few(described):
    """The kernel's symbol has numbers only, the engine's names its loaders."""
    return described.split(" | ")[1].count("<") == 1


@pytest.mark.parametrize("case,few", CASES, ids=str)
def test_bits_of_the_tile_engine(rt, monkeypatch, case, few):
    from tinyflow_amd import gpu_op, ndarray
    monkeypatch.setenv("TINYFLOW_WINOGRAD", "0")
    N, C, H, W, K, R, S, padding, u, v = case
    out_shape, lst = gpu_op.convolution_2d_forward_get_out_shape((N, C, H, W), (K, C, R, S), "NCHW", padding, u, v)
    assert tuple(_few(_describe(lst, which)) for which in (0, 1)) == few
    rng = np.random.RandomState(3)
    x, w, dy = (rng.normal(0, s, shape).astype(np.float32)
                for s, shape in ((1, (N, C, H, W)), (0.3, (K, C, R, S)), (1, out_shape)))
    xd, wd, dyd = _gpu(x, rt), _gpu(w, rt), _gpu(dy, rt)
    results = []
    for switch in ("1", "0"):
        monkeypatch.setenv("TINYFLOW_FEW_CHANNELS", switch)
        y, dx = ndarray.empty(out_shape, rt.ctx), ndarray.empty(x.shape, rt.ctx)
        assert gpu_op.convolution_2d_forward(xd, wd, y, lst, rt.cudnn, rt.stream) == 0
        assert gpu_op.convolution_backward_data(xd, dyd, wd, dx, lst, rt.cudnn, rt.stream) == 0
        results.append((y.asnumpy(), dx.asnumpy()))
    assert not any(_few(_describe(lst, which)) for which in (0, 1))
    for few_bits, engine_bits in zip(*results):
        assert few_bits.tobytes() == engine_bits.tobytes()


@pytest.mark.parametrize("case", [c for c, few in CASES if few[0] and c[0] < 2000], ids=str)
def test_forward_is_the_product_with_the_patches(rt, monkeypatch, case):
    """The product of the filter with the gathered patches on the engine, image by image."""
    from tinyflow_amd import gpu_op, ndarray
    from oracle import ops as O
    monkeypatch.setenv("TINYFLOW_WINOGRAD", "0")
    N, C, H, W, K, R, S, padding, u, v = case
    out_shape, lst = gpu_op.convolution_2d_forward_get_out_shape((N, C, H, W), (K, C, R, S), "NCHW", padding, u, v)
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
