"""GPU parity: 17..64 f16 rows with all of K in one workgroup (gemm_rows.hip), against the oracle."""
import ctypes as C
import zlib

import numpy as np
import pytest

import torchlette_amd as T
from oracle import quant_oracle as O
from torchlette_amd import _lib as L
from helpers import fmt_name, make_weight, make_x, rel_l2
from test_gpu_gemv import run_linear

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def be():
    return T.getBackend()


@pytest.mark.parametrize("m", [17, 32, 33, 48, 49, 64])
@pytest.mark.parametrize("fmt,g,n,k", [
    ("int4-grouped", 32, 100, 128),    # one step: seven waves have none; the last columns off the tile and off four
    ("int4-grouped", 32, 1030, 2304),  # 18 steps: an odd number for some waves
    ("int8-grouped", 64, 131, 1152),   # 9 steps
    ("int8-grouped", 256, 96, 2048),
    ("int8-row", 0, 515, 1920),
])
def test_rows_match_the_oracle(be, fmt, g, n, k, m):
    rng = np.random.default_rng(zlib.crc32(repr((fmt, g, n, k, m)).encode()))
    packed, scales, deq = make_weight(fmt, n, k, g, rng)
    x, bias = make_x(m, k, "f16", rng), rng.standard_normal(n).astype(np.float32)
    want = O.linear(x.astype(np.float32), deq, bias, "silu", threads=8)
    ran = []
    for cols in (1, 2, 3, 4):
        try:
            got = run_linear(be, fmt, packed, scales, n, k, g, x, "f32", bias=bias, act="silu", fused=True,
                             config=L.KernelConfig.of(L.VARIANT_GEMV_MFMA, 8, 0, 0, 0, cols))
        except L.TlhipError as e:
            assert "not applicable" in str(e)  # more registers than a lane has
            continue
        ran.append(cols)
        assert rel_l2(got, want) <= 2e-6, cols  # exact products, f32 sums: order noise only
    assert ran == widths(fmt, m)


def widths(fmt, m):
    """Blocks of 16 columns whose instance a lane's registers hold, at 32, 48 and 64 rows."""
    return [1, 2, 3, 4][:{2: 4, 3: 4 if fmt == "int4-grouped" else 3, 4: 3 if fmt == "int4-grouped" else 2}[(m + 15) // 16]]


@pytest.mark.parametrize("m", [17, 40, 64])
@pytest.mark.parametrize("fmt,g,n,k,ydt,alpha", [
    ("int4-grouped", 32, 132, 1152, "f16", 1.0),   # whole vectors of four columns
    ("int4-grouped", 32, 131, 1152, "f16", -0.75),  # the last columns one by one
    ("int8-grouped", 128, 164, 640, "f16", 0.5),
    ("int8-grouped", 64, 165, 640, "f32", 1.0),
    ("int8-row", 0, 196, 896, "f32", 1.0),
    ("int8-row", 0, 197, 896, "f16", 1.5),
])
def test_stores_residual_and_alpha(be, fmt, g, n, k, ydt, alpha, m):
    """f16 and f32 stores by four columns and one by one, behind a bias, a residual that is the output
    itself and alpha.  Bounds: the products are exact, the sums of f32 round like those above; an f16
    store rounds once to 2^-11 of the value, or half of the smallest f16."""
    rng = np.random.default_rng(zlib.crc32(repr((fmt, g, n, k, m)).encode()))
    packed, scales, deq = make_weight(fmt, n, k, g, rng)
    x, bias = make_x(m, k, "f16", rng), rng.standard_normal(n).astype(np.float32)
    other = make_x(m, n, ydt, rng)
    w = be.createQuantizedWeight(packed, scales, n, k, T.resolveWeightFormat(fmt_name(fmt, g), "f32"))
    qw, xt, bt = be._qweight(w, False), be.ops.tensorFromArray(x, [m, k], "f16"), be.ops.tensorFromArray(bias, [n], "f32")
    xs, d = x.astype(np.float64), deq.astype(np.float64)
    want = alpha * (xs @ d.T) + bias + other
    magnitudes = abs(alpha) * (np.abs(xs) @ np.abs(d).T) + np.abs(bias) + np.abs(other)
    for cols in widths(fmt, m):
        y = be.ops.tensorFromArray(other, [m, n], ydt)
        ep = be.makeEpilogueChain([("bias", bt), ("binary", "add", y)])
        cfg = L.KernelConfig.of(L.VARIANT_GEMV_MFMA, 8, 0, 0, 0, cols)
        L.call("tlhip_matmul_quantized_config", C.byref(qw), xt.ptr, L.F16, m, y.ptr, L.F16 if ydt == "f16" else L.F32, alpha,
               C.byref(ep), C.byref(cfg), None)
        got = y.numpy()
        y.destroy()
        bound = 2.0**-21 * magnitudes
        if ydt == "f16":
            bound = bound + 2.0**-11 * (np.abs(want) + bound) + 2.0**-25
        assert np.all(np.abs(got.astype(np.float64) - want) <= bound), cols


@pytest.mark.parametrize("fmt,g", [("int4-grouped", 32), ("int8-grouped", 64), ("int8-row", 0)])
@pytest.mark.parametrize("m", [20, 48, 61])
def test_values_that_are_not_finite_stay_in_their_row(be, fmt, g, m):
    """An infinity and a NaN of one row, in a step of K that no whole round of waves has."""
    n, k = 80, 1152
    rng = np.random.default_rng(m)
    packed, scales, deq = make_weight(fmt, n, k, g, rng)
    x = make_x(m, k, "f16", rng)
    x[2, 1130], x[m - 1, 3] = np.inf, np.nan
    with np.errstate(invalid="ignore"):
        want = x.astype(np.float64) @ deq.astype(np.float64).T  # an infinity times a zero weight is NaN
    for cols in widths(fmt, m):
        got = run_linear(be, fmt, packed, scales, n, k, g, x, "f32", config=L.KernelConfig.of(L.VARIANT_GEMV_MFMA, 8, 0, 0, 0, cols))
        finite = [r for r in range(m) if r not in (2, m - 1)]
        assert rel_l2(got[finite], want[finite]) <= 2e-6, cols
        assert np.all(np.isnan(got[m - 1])) and np.array_equal(got[2], want[2].astype(np.float32), equal_nan=True), cols


def test_the_width_is_not_read_with_the_other_forms_fields(be):
    fmt, g, n, k, m = "int4-grouped", 32, 512, 2048, 40
    rng = np.random.default_rng(7)
    packed, scales, _ = make_weight(fmt, n, k, g, rng)
    x = make_x(m, k, "f16", rng)
    plain, with_width = (run_linear(be, fmt, packed, scales, n, k, g, x, "f32", config=L.KernelConfig.of(L.VARIANT_GEMV_MFMA, 8, 2, 8, 2, p4))
                         for p4 in (0, 2))
    assert np.array_equal(plain.view(np.uint32), with_width.view(np.uint32))
