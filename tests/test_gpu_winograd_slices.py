"""Transformed-domain products of 3x3 / stride-1 layers on bf16 slices (csrc/conv.hip, csrc/gemm_split.h): every tile and loader
pair against the oracle, the error against float64 beside the fp32 engine's, and who is given them."""
import numpy as np
import pytest

import parity
from oracle import ops as O
from test_gpu_conv import WINOGRAD_CASES, _check_conv_case, _describe, _gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("force", ["2", "4"])
@pytest.mark.parametrize("case", [c[0] for c in WINOGRAD_CASES] + [
    (9, 160, 30, 34, 136, 3, 3, "SAME", 1, 1),     # 128 x 128 tiles with a remainder both ways
    (8, 320, 16, 16, 96, 3, 3, "VALID", 1, 1),
    (40, 72, 13, 13, 200, 3, 3, "SAME", 1, 1),     # grad-filter in pieces
], ids=str)
def test_products_on_slices(rt, monkeypatch, case, force):
    from tinyflow_amd import gpu_op
    monkeypatch.setenv("TINYFLOW_WINOGRAD", force)
    monkeypatch.setenv("TINYFLOW_SPLIT", "1")
    N, C, H, W, K, R, S, padding, u, v = case
    _, lst = gpu_op.convolution_2d_forward_get_out_shape((N, C, H, W), (K, C, R, S), "NCHW", padding, u, v)
    for which in range(3):
        described = _describe(lst, which)
        if "winograd" in described:
            assert "Split" in described, described
    _check_conv_case(rt, case)


@pytest.mark.parametrize("case", [(4, 256, 28, 28, 256), (2, 512, 14, 14, 512), (8, 64, 56, 56, 64)], ids=str)
def test_error_is_not_above_the_fp32_engines(rt, monkeypatch, case):
    """The transforms are the same and so is their rounding, which is most of it: 1.01 is what two roundings of the same size may
    differ by over 10^4 and more elements; what the products add is smaller on slices."""
    from tinyflow_amd import gpu_op, ndarray
    N, C, H, W, K = case
    rng = np.random.RandomState(parity.stable_seed(case))
    x = np.maximum(rng.normal(0, 1, (N, C, H, W)), 0).astype(np.float32)
    w = rng.normal(0, np.sqrt(2.0 / (C * 9)), (K, C, 3, 3)).astype(np.float32)
    dy = rng.normal(0, 1, (N, K, H, W)).astype(np.float32)
    x64, w64, dy64 = (a.astype(np.float64) for a in (x, w, dy))
    refs = (O.conv2d_forward(x64, w64, 1, 1, 1, 1), O.conv2d_backward_data(dy64, w64, x.shape, 1, 1, 1, 1),
            O.conv2d_backward_filter(x64, dy64, w.shape, 1, 1, 1, 1))
    gx, gw, gdy = _gpu(x, rt), _gpu(w, rt), _gpu(dy, rt)
    outs = [ndarray.empty(r.shape, rt.ctx) for r in refs]
    monkeypatch.setenv("TINYFLOW_WINOGRAD", "4")
    errors = []
    for engine in ("0", "1"):
        monkeypatch.setenv("TINYFLOW_SPLIT", engine)
        _, lst = gpu_op.convolution_2d_forward_get_out_shape(x.shape, w.shape, "NCHW", "SAME", 1, 1)
        assert gpu_op.convolution_2d_forward(gx, gw, outs[0], lst, rt.cudnn, rt.stream) == 0
        assert gpu_op.convolution_backward_data(gx, gdy, gw, outs[1], lst, rt.cudnn, rt.stream) == 0
        assert gpu_op.convolution_backward_filter(gx, gdy, gw, outs[2], lst, rt.cudnn, rt.stream) == 0
        errors.append([np.linalg.norm(o.asnumpy().astype(np.float64) - r) / np.linalg.norm(r) for o, r in zip(outs, refs)])
    print(case, errors)
    assert all(s <= 1.01 * f for f, s in zip(*errors)), errors


def test_executors_give_permission_for_sgd_without_batch_norm_alone(rt):
    from tinyflow_amd import autodiff as ad, models, TrainExecute, TrainExecuteAdam
    for module, norms, allowed in ((TrainExecute, False, True), (TrainExecuteAdam, False, False), (TrainExecute, True, False)):
        rng = np.random.RandomState(3)
        X, y = models.synthetic_batch(rng, (4, 3, 64, 64), 10, "normal")
        if norms:
            model = models.resnet(rng, (1, 1, 1, 1), batch=4, image=64, n_class=10, bn_mode="spatial")
        else:
            model = models.vgg16(rng, batch=4, image=64, n_class=10, fc_width=32)
        executor = module.TrainExecutor(model.loss, 1e-4)
        executor.init_Variable(dict(model.variables))
        executor.run({model.X: X, model.y_: y})
        plans = [_describe(n.cudnnlist[0], w) for n in executor.topo_order if isinstance(n.op, ad.Convolution2DForwardOp)
                 and executor.node_to_shape_map[n.inputs[1]][2] == 3 for w in range(3)]
        assert any("Split" in p for p in plans) == allowed, plans
        executor.close()


def _calls(rt, case, spoil):
    """Outputs of the three calls of a layer in the transformed domain, and the time of its product-heavy calls, with `spoil` applied to x, w
    and dy before."""
    import time
    from tinyflow_amd import gpu_op, ndarray
    N, C, H, W, K = case
    rng = np.random.RandomState(parity.stable_seed(case))
    x = np.maximum(rng.normal(0, 1, (N, C, H, W)), 0).astype(np.float32)
    w = rng.normal(0, np.sqrt(2.0 / (C * 9)), (K, C, 3, 3)).astype(np.float32)
    dy = rng.normal(0, 1, (N, K, H, W)).astype(np.float32)
    spoil(x, w, dy)
    gx, gw, gdy = _gpu(x, rt), _gpu(w, rt), _gpu(dy, rt)
    outs = [ndarray.empty(a.shape, rt.ctx) for a in (dy, x, w)]
    _, lst = gpu_op.convolution_2d_forward_get_out_shape(x.shape, w.shape, "NCHW", "SAME", 1, 1)

    def step():
        assert gpu_op.convolution_2d_forward(gx, gw, outs[0], lst, rt.cudnn, rt.stream) == 0
        assert gpu_op.convolution_backward_data(gx, gdy, gw, outs[1], lst, rt.cudnn, rt.stream) == 0
        assert gpu_op.convolution_backward_filter(gx, gdy, gw, outs[2], lst, rt.cudnn, rt.stream) == 0
    step()
    values = [o.asnumpy() for o in outs]
    best = 1e9
    for _ in range(5):
        start = time.perf_counter()
        for _ in range(20):
            step()
        outs[2].asnumpy()
        best = min(best, time.perf_counter() - start)
    return values, best


# the first and the last stage of a reduction, one value and all of them, of every operand
@pytest.mark.parametrize("what", ["x first inf", "x last nan", "w first nan", "w last -inf", "dy first inf", "dy last nan", "all nan"])
def test_values_that_are_not_finite(rt, monkeypatch, what):
    """What is finite on the fp32 engine is finite on slices, and within the rounding of two fp32 sums of it."""
    def spoil(x, w, dy):
        if what == "all nan":
            for a in (x, w, dy):
                a[...] = np.nan
            return
        name, place, value = what.split(" ")
        {"x": x, "w": w, "dy": dy}[name][0, 0 if place == "first" else -1, 1, 1] = float(value)
    monkeypatch.setenv("TINYFLOW_WINOGRAD", "4")
    results = []
    for engine in ("0", "1"):
        monkeypatch.setenv("TINYFLOW_SPLIT", engine)
        results.append(_calls(rt, (2, 136, 20, 20, 72), spoil)[0])
    for fp32, slices, terms in zip(*results, (136 * 9, 72 * 9, 800)):
        finite = np.isfinite(fp32)
        assert (np.isfinite(slices) == finite).all()
        if finite.any():
            # sums of random signs: 2^-24 sqrt(terms) of their size apart, 2.7 times that in this domain, and the transforms' rounding
            assert (np.abs(fp32 - slices)[finite] <= 6 * (2.7 * 2.0 ** -24 * np.sqrt(terms) + 4e-6) * np.abs(fp32[finite]).std()).all()


def test_steps_on_nan_take_about_the_fp32_engines_time(rt, monkeypatch):
    """Nothing of the slices' work is done for a tile whose first operands show that the fp32 pass will compute it: with it the three
    calls took twice the fp32 engine's time, without it they take 1.2 times."""
    monkeypatch.setenv("TINYFLOW_WINOGRAD", "4")

    def spoil(x, w, dy):
        for a in (x, w, dy):
            a[...] = np.nan
    times = []
    for engine in ("0", "1"):
        monkeypatch.setenv("TINYFLOW_SPLIT", engine)
        times.append(_calls(rt, (32, 512, 28, 28, 512), spoil)[1])
    print(times)
    assert times[1] <= 1.6 * times[0], times
