"""GPU parity: 2..5 f32 rows on the VALU in one launch (gemv_some.hip), against 64-bit sums of the oracle's weights."""
import zlib

import numpy as np
import pytest

import torchlette_amd as T
from torchlette_amd import _lib as L
from helpers import fmt_name, make_weight, make_x

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def be():
    return T.getBackend()


def some(lanes, cols):
    return L.KernelConfig.of(L.VARIANT_GEMV, lanes, 1, 8, 1, cols, 4)


@pytest.mark.parametrize("m", [2, 3, 4, 5])
@pytest.mark.parametrize("fmt,g,n,k,lanes", [
    ("int4-grouped", 32, 101, 64, 16),      # eight lanes of one wave have all of K
    ("int4-grouped", 32, 260, 1024, 16),    # a whole range
    ("int4-grouped", 32, 131, 2112, 64),    # five waves, the last with eight lanes
    ("int4-grouped", 64, 77, 8192, 64),     # two pieces of K a wave
    ("int8-grouped", 64, 96, 1920, 32),
    ("int8-grouped", 128, 100, 5376, 64),   # the second pieces: a part of them past the end
    ("int8-grouped", 1024, 33, 2048, 32),
    ("int8-row", 0, 66, 1056, 32),
    ("int8-row", 0, 9, 4096, 64),
])
def test_a_few_f32_rows(be, fmt, g, n, k, lanes, m):
    rng = np.random.default_rng(zlib.crc32(repr((fmt, g, n, k, m)).encode()))
    packed, scales, deq = make_weight(fmt, n, k, g, rng)
    w = be.createQuantizedWeight(packed, scales, n, k, T.resolveWeightFormat(fmt_name(fmt, g), "f32"))
    x = make_x(m, k, "f32", rng, std=0.5)
    bias, other = rng.standard_normal(n).astype(np.float32), rng.standard_normal((m, n)).astype(np.float32)
    xt, bt, ot = be.ops.tensorFromArray(x, [m, k], "f32"), be.ops.tensorFromArray(bias, [n], "f32"), be.ops.tensorFromArray(other, [m, n], "f32")
    ep = be.makeEpilogueChain([("bias", bt), ("binary", "add", ot)])
    want = x.astype(np.float64) @ deq.astype(np.float64).T + bias + other
    magnitudes = np.abs(x).astype(np.float64) @ np.abs(deq).astype(np.float64).T + np.abs(bias) + np.abs(other)
    for cols in (1, 5, 12, 37, 64):  # one column; a branch a column; some of two, three and four turns
        got = be._matmulQuantizedB(xt, be.ops.transpose(w), ep, some(lanes, cols)).numpy()
        # two roundings in the oracle's weight; here 8 products a lane, two pieces, and ten levels of sums
        assert np.all(np.abs(got - want) <= 21 * 2.0**-24 * magnitudes), cols


def test_what_is_not_finite_stays_in_its_row(be):
    rng = np.random.default_rng(5)
    n, k, m = 131, 2304, 4
    packed, scales, deq = make_weight("int8-grouped", n, k, 64, rng)
    w = be.createQuantizedWeight(packed, scales, n, k, T.resolveWeightFormat("int8-64", "f32"))
    x = make_x(m, k, "f32", rng, std=0.5)
    x[1, 700], x[3, k - 1] = np.inf, np.nan
    got = be._matmulQuantizedB(be.ops.tensorFromArray(x, [m, k], "f32"), be.ops.transpose(w), None, some(64, 9)).numpy()
    with np.errstate(invalid="ignore"):
        want = x.astype(np.float64) @ deq.astype(np.float64).T
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
    ok = np.isfinite(want)
    assert np.all(np.abs(got[ok] - want[ok]) <= 21 * 2.0**-24 * (np.abs(x[[0, 2]]).astype(np.float64) @ np.abs(deq).astype(np.float64).T).ravel())


def test_the_form_rejects_what_it_does_not_cover(be):
    rng = np.random.default_rng(6)
    for m, k, cfg in ((6, 2048, some(32, 8)), (1, 2048, some(32, 8)), (3, 2304, some(32, 8)), (3, 8256, some(64, 8)), (3, 2048, some(32, 65)),
                      (3, 2048, some(32, 0)), (3, 2048, some(8, 8)), (3, 2112, some(64, 8))):  # (33 groups of 64)
        packed, scales, _ = make_weight("int8-grouped", 64, k, 64, rng)
        w = be.createQuantizedWeight(packed, scales, 64, k, T.resolveWeightFormat("int8-64", "f32"))
        with pytest.raises(L.TlhipError, match="not applicable"):
            be._matmulQuantizedB(be.ops.tensorFromArray(make_x(m, k, "f32", rng), [m, k], "f32"), be.ops.transpose(w), None, cfg)
