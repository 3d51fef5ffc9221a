"""The contractions on bf16 slices (csrc/gemm_split.h) against float64 and against the fp32 engine.

TINYFLOW_SPLIT=1 forces the engine wherever it has loaders, so that small cases reach every loader; 0 is the fp32
engine.  Bounds: an element of a product is off by at most gamma = (K + 8) 2^-24 times the sum of its terms'
magnitudes (one rounding per reduction step, the omitted slices 2^-24 at most and the last addition), the classical bound of
an fp32 sum in any order."""
import math

import numpy as np
import pytest

from oracle import ops as O
import parity
from test_gpu_conv import CONV_CASES, STRIDED_CASES, _check_conv_case, _describe, _gpu

pytestmark = pytest.mark.gpu


@pytest.fixture
def split(monkeypatch):
    monkeypatch.setenv("TINYFLOW_SPLIT", "1")
    monkeypatch.setenv("TINYFLOW_WINOGRAD", "0")


@pytest.mark.parametrize("case", CONV_CASES + [c[0] for c in STRIDED_CASES], ids=lambda c: "x".join(str(v) for v in c))
def test_convolutions_on_the_split_engine(rt, split, case):
    _check_conv_case(rt, case)


# (N, C, H, W, K, R, S, padding, u, v), which, loaders that the plan has to name: every loader pair, on the 128 x 128
# tile where the size asks for it
LOADER_CASES = [
    ((16, 256, 28, 28, 512, 1, 1, "VALID", 1, 1), 0, "gemm_kernel<128, 128, 16, SplitAcross4<128, 16, false, false>, SplitAlong4<128, 16>"),
    ((16, 256, 28, 28, 512, 1, 1, "VALID", 1, 1), 1, "gemm_kernel<128, 128, 16, SplitAlong4<128, 16>, SplitAlong4<128, 16>, StoreNCHW"),
    ((16, 256, 28, 28, 512, 1, 1, "VALID", 1, 1), 2, "SplitAcross4<128, 16, false, true>, SplitAcross4<128, 16, false, true>"),
    ((16, 262, 7, 7, 512, 1, 1, "VALID", 1, 1), 0, "SplitAcross4<64, 32, true, false>, SplitGatherAlong<64, 32, 0>"),
    ((16, 264, 7, 7, 512, 1, 1, "VALID", 1, 1), 2, "true, true>, SplitAcross4<"),
    ((16, 128, 56, 56, 512, 1, 1, "VALID", 2, 2), 1, "StoreScatter"),
    ((8, 128, 32, 32, 140, 1, 1, "VALID", 2, 2), 2, "SplitGatherAcross<64, 32, 3>"),
    ((8, 64, 19, 18, 72, 3, 3, "VALID", 1, 1), 2, "SplitGatherAcross<64, 32, 2>"),
    ((4, 64, 14, 14, 72, 1, 1, "VALID", 2, 2), 2, "true, true>, SplitGatherAcross<64, 32, 0>"),   # 49 outputs: ragged dy
    ((9, 64, 6, 6, 72, 1, 1, "VALID", 2, 2), 2, "SplitDyAcross<64, 32>, SplitGatherAcross<64, 32, 0>"),  # 9 outputs
    ((20, 50, 61, 59, 70, 5, 5, "VALID", 2, 2), 1, "PhasedFilter<SplitAlong4<"),
]


@pytest.mark.parametrize("case,which,loaders", LOADER_CASES, ids=str)
def test_loaders_at_the_sizes_that_use_them(rt, split, case, which, loaders):
    from tinyflow_amd import gpu_op
    N, C, H, W, K, R, S, padding, u, v = case
    _, lst = gpu_op.convolution_2d_forward_get_out_shape((N, C, H, W), (K, C, R, S), "NCHW", padding, u, v)
    assert loaders in _describe(lst, which), _describe(lst, which)
    _check_conv_case(rt, case)


def _product(rt, a, ta, b, tb):
    from tinyflow_amd import gpu_op, ndarray
    c = ndarray.empty((a.shape[0], b.shape[1]), rt.ctx)
    gpu_op.array_set(c, np.nan, rt.stream)
    gpu_op.matrix_multiply(_gpu(np.ascontiguousarray(a.T) if ta else a, rt), ta,
                           _gpu(np.ascontiguousarray(b.T) if tb else b, rt), tb, c, rt.cublas, rt.stream)
    return c.asnumpy().astype(np.float64)


@pytest.mark.parametrize("m,k,n", [
    (1, 1, 1), (2, 3, 5), (64, 32, 64), (65, 33, 63), (128, 16, 128), (129, 47, 130), (130, 1023, 70),  # remainders
    (300, 258, 257), (257, 4097, 263),     # split along the reduction
    (1000, 1537, 777), (2049, 261, 2050),  # both tiles, pieces, a partial last round
], ids=str)
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)], ids=str)
def test_products(rt, split, m, k, n, ta, tb):
    rng = np.random.RandomState(parity.stable_seed((m, k, n)))
    a = rng.normal(0, 1, (m, k)).astype(np.float32)
    b = rng.normal(0, 1, (k, n)).astype(np.float32)
    got = _product(rt, a, ta, b, tb)
    ref = a.astype(np.float64) @ b.astype(np.float64)
    bound = (k + 8) * 2.0 ** -24 * (np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64))
    assert (np.abs(got - ref) <= bound).all()


@pytest.mark.parametrize("scale_a,scale_b", [(1.0, 1.0), (1e-30, 1e25), (3e15, 2e18), (1e-18, 1e-18)], ids=str)
def test_products_are_no_further_from_float64_than_the_fp32_engine(rt, monkeypatch, scale_a, scale_b):
    """Signed and one-signed data, long and short reductions: root mean square error not above the fp32 engine's."""
    rng = np.random.RandomState(3)
    for m, k, n in [(320, 264, 512), (288, 4608, 320), (512, 1000, 384)]:
        for positive in (False, True):
            a = rng.normal(0, 1, (m, k))
            a = (np.maximum(a, 0) * scale_a).astype(np.float32)
            b = (rng.normal(0, 1, (k, n)) if not positive else rng.uniform(0.5, 1.5, (k, n)))
            b = (b * scale_b).astype(np.float32)
            ref = a.astype(np.float64) @ b.astype(np.float64)
            err = []
            for engine in ("0", "1"):
                monkeypatch.setenv("TINYFLOW_SPLIT", engine)
                err.append(np.linalg.norm(_product(rt, a, False, b, False) - ref))
            assert err[1] <= err[0], (m, k, n, positive, err)


# 1 + 2^-8 - 2^-17 - 2^-23: the middle slice all but 2^-8 and the last 2^-17 of it, so the products that are left out, all of
# one sign, are 0.97 of 2^-24 of the whole
WORST = 1 + 2.0 ** -8 - 2.0 ** -17 - 2.0 ** -23


@pytest.mark.parametrize("k", [1, 16, 24, 100, 264, 4096])
def test_the_largest_omission_stays_within_roundings(rt, split, monkeypatch, k):
    """Equal operands: the omissions add up to 2^-24 of the result, beside the final rounding (2^-24) and those of the
    sums, where the fp32 engine's chain of equal summands adds up to more."""
    a, b = np.full((70, k), WORST, np.float32), np.full((k, 70), WORST, np.float32)
    ref = k * float(np.float32(WORST)) ** 2
    err = []
    for engine in ("0", "1"):
        monkeypatch.setenv("TINYFLOW_SPLIT", engine)
        err.append(np.abs(_product(rt, a, False, b, False) - ref).max() / ref)
    assert err[1] <= max(err[0], 2.0 ** -23), err


@pytest.mark.parametrize("k", [24, 264, 1024])
@pytest.mark.parametrize("signed", [False, True])
def test_slices_of_extreme_rests_are_no_further_from_float64(rt, monkeypatch, k, signed):
    """Every element has the rests of WORST behind eight leading bits of its own."""
    rng = np.random.RandomState(7)
    a = rng.randint(128, 256, (320, k)) / 128.0 + (WORST - 1)
    b = rng.randint(128, 256, (k, 320)) / 128.0 + (WORST - 1)
    if signed:
        b *= rng.choice([-1, 1], b.shape)
    a, b = a.astype(np.float32), b.astype(np.float32)
    ref = a.astype(np.float64) @ b.astype(np.float64)
    err = []
    for engine in ("0", "1"):
        monkeypatch.setenv("TINYFLOW_SPLIT", engine)
        err.append(np.linalg.norm(_product(rt, a, False, b, False) - ref))
    assert err[1] <= err[0], err


@pytest.mark.parametrize("scale_a,scale_b", [
    (1e-33, 1.0), (1e-35, 1.0), (1e-37, 1.0), (1e-40, 1.0), (1e-44, 1.0),     # down to one bit of a subnormal number
    (1e-36, 1e30), (1e-37, 1e37), (1e-40, 1e30), (1e-44, 1e37),               # tiny operands of ordinary results
    (1e-19, 1e-19), (1e-20, 1e-20), (1e-22, 1e-22),                           # results below the normal numbers
    (1.0, 1e24), (1e30, 1.0), (1e-38, 3e31), (1e12, 1e12), (1e18, 1e18),      # around the scaled range's upper end and past it
], ids=str)
@pytest.mark.parametrize("swapped", [False, True], ids=["a", "b"])
def test_operands_of_any_size_keep_their_bits(rt, monkeypatch, scale_a, scale_b, swapped):
    """The error is not above the fp32 engine's whatever the exponents are; tiles of ordinary numbers beside tiny ones, rows
    of zeros and single tiny elements do not matter."""
    rng = np.random.RandomState(6)
    m, k, n = 320, 264, 288
    a, b = rng.normal(0, 1, (m, k)) * scale_a, rng.normal(0, 1, (k, n)) * scale_b
    ordinary, tiny = np.arange(0, 128), np.arange(128, m)
    if scale_a < 1:
        a[ordinary] *= min(1.0, 1.0 / scale_b) / scale_a
        a[40, 261] = scale_a
    a[2::9] = 0.0
    a, b = a.astype(np.float32), b.astype(np.float32)
    ref = a.astype(np.float64) @ b.astype(np.float64)
    err = []
    for engine in ("0", "1"):
        monkeypatch.setenv("TINYFLOW_SPLIT", engine)
        got = _product(rt, b.T.copy(), False, a.T.copy(), False).T if swapped else _product(rt, a, False, b, False)
        np.testing.assert_array_equal(got[2::9], 0.0)
        err.append([np.linalg.norm((got - ref)[rows]) for rows in (ordinary, tiny)])
    assert err[1][0] <= err[0][0] and err[1][1] <= err[0][1], err


def test_what_bf16_cannot_hold_is_computed_in_fp32(rt, monkeypatch):
    """Infinities, NaN, values above the largest bf16 and sums that overflow part way: tiles that meet one have the
    fp32 engine's results, elements of other tiles are not touched by them."""
    rng = np.random.RandomState(4)
    m, k, n = 300, 320, 290
    a = rng.normal(0, 1, (m, k)).astype(np.float32)
    b = rng.uniform(0.25, 0.75, (k, n)).astype(np.float32)   # no zeros: infinity times zero has no sign to compare
    a[3, 5] = np.inf
    a[70, 6] = -np.inf
    a[71, 7] = np.nan
    a[140, 8] = np.float32(3.4e38)          # above the largest bf16
    a[140, 9] = -np.float32(3.4e38)
    a[200, :] = np.float32(1e37)            # overflows
    out = []
    for engine in ("0", "1"):
        monkeypatch.setenv("TINYFLOW_SPLIT", engine)
        out.append(_product(rt, a, False, b, False))
    for rows in (3, 70, 71, 200):
        np.testing.assert_array_equal(out[0][rows], out[1][rows])
    assert np.isposinf(out[1][3]).all() and np.isneginf(out[1][70]).all() and np.isnan(out[1][71]).all()
    assert np.isposinf(out[1][200]).all()
    finite = [r for r in range(m) if r not in (3, 70, 71, 140, 200)]
    ref = a[finite].astype(np.float64) @ b.astype(np.float64)
    np.testing.assert_allclose(out[1][finite], ref, rtol=0, atol=(k + 8) * 2.0 ** -24 * float(np.abs(a[finite]).sum(1).max()))
    big = a[140].astype(np.float64) @ b.astype(np.float64)
    assert (np.abs(out[1][140] - big) <= (k + 8) * 2.0 ** -24 * (np.abs(a[140]).astype(np.float64) @ b.astype(np.float64))).all()


def test_repeated_calls_have_the_same_bits(rt, split):
    rng = np.random.RandomState(5)
    a = rng.normal(0, 1, (1000, 1537)).astype(np.float32)
    b = rng.normal(0, 1, (1537, 777)).astype(np.float32)
    first = _product(rt, a, False, b, False)
    for _ in range(3):
        assert first.tobytes() == _product(rt, a, False, b, False).tobytes()
