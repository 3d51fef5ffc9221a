"""What the permission for bf16 slices (DLGpuConvolutionAllowSlices) changes in the plans of 3x3 / stride-1 layers, from the plans
alone (csrc/conv.hip: choose_direct, consider_winograd)."""
import pytest

from test_gpu_conv import _describe


@pytest.fixture(autouse=True)
def _planner_decides(monkeypatch):
    for name in ("TINYFLOW_SPLIT", "TINYFLOW_WINOGRAD", "TINYFLOW_WINOGRAD_MAX_TILE"):
        monkeypatch.delenv(name, raising=False)


def _plans(n, c, h, w, k, padding="SAME"):
    """The plans of forward, grad-data and grad-filter without and with the permission."""
    from tinyflow_amd import gpu_op
    plans = []
    for allow in (False, True):
        _, lst = gpu_op.convolution_2d_forward_get_out_shape((n, c, h, w), (k, c, 3, 3), "NCHW", padding, 1, 1)
        gpu_op.convolution_allow_slices(lst, allow)
        plans.append([_describe(lst, which) for which in range(3)])
    return plans


# outside the transformed domain: one and many pieces, aligned and ragged channels
@pytest.mark.parametrize("layer", [(4, 64, 6, 6, 64), (4, 24, 6, 6, 200), (32, 45, 2, 2, 27), (6, 64, 28, 28, 128), (16, 32, 56, 56, 32)],
                         ids=str)
def test_direct_grad_filter_keeps_its_engine(layer):
    without, with_permission = _plans(*layer)
    assert "winograd" not in without[2] and with_permission[2] == without[2]


# ragged channels, many images of small maps, one image of large ones
@pytest.mark.parametrize("layer", [(5, 96, 40, 40, 72), (32, 96, 14, 14, 72), (60, 240, 7, 7, 92), (1, 64, 102, 102, 96), (5, 320, 22, 22, 96)],
                         ids=str)
def test_permission_takes_no_grad_data_out_of_the_transformed_domain(layer):
    without, with_permission = _plans(*layer)
    assert "winograd" in without[1] and "winograd" in with_permission[1], with_permission
