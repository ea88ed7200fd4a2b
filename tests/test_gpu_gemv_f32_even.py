"""GPU parity: 2..16 f32 rows with all of K in one workgroup and an even share of the columns (gemv_f32.hip)."""
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


def product(be, fmt, g, n, k, x, cols, rng):
    packed, scales, deq = make_weight(fmt, n, k, g, rng)
    w = be.createQuantizedWeight(packed, scales, n, k, T.resolveWeightFormat(fmt_name(fmt, g), "f32"))
    xt = be.ops.tensorFromArray(x, list(x.shape), "f32")
    got = [be._matmulQuantizedB(xt, be.ops.transpose(w), None, L.KernelConfig.of(L.VARIANT_GEMV_F32, 8, 1, c)).numpy() for c in cols]
    return got, deq


@pytest.mark.parametrize("m", [2, 4, 5, 8, 9, 12, 16])
@pytest.mark.parametrize("fmt,g,n,k", [
    ("int4-grouped", 32, 101, 128),    # one step: seven waves have none
    ("int4-grouped", 32, 260, 2432),   # 19 steps: two and three a wave
    ("int4-grouped", 32, 36, 16384),   # sixteen steps a wave: the scales in two loads
    ("int8-grouped", 64, 131, 1152),
    ("int8-grouped", 128, 100, 2176),  # 17 steps, a scale each
    ("int8-grouped", 256, 96, 16384),  # a scale for two steps, four loads of them
    ("int8-row", 0, 515, 1920),
])
def test_an_even_share_of_the_columns(be, fmt, g, n, k, m):
    rng = np.random.default_rng(zlib.crc32(repr((fmt, g, n, k, m)).encode()))
    x = make_x(m, k, "f32", rng, std=0.5)
    cols = (3, 20, 36, 48) + ((50, 64) if m <= 10 else ())  # a block, even shares of two to four, full ones
    got, deq = product(be, fmt, g, n, k, x, cols, rng)
    want = x.astype(np.float64) @ deq.astype(np.float64).T
    magnitudes = np.abs(x).astype(np.float64) @ np.abs(deq).astype(np.float64).T
    for c, y in zip(cols, got):
        assert np.all(np.abs(y - want) <= 2.0**-21 * magnitudes), c  # a chain of at most 2048 in f32, as the K slices


def test_what_is_not_finite_stays_in_its_row(be):
    rng = np.random.default_rng(5)
    x = make_x(5, 1152, "f32", rng, std=0.5)
    x[1, 700], x[2, 3], x[4, 1151] = np.inf, -np.inf, np.nan
    got, deq = product(be, "int8-grouped", 64, 131, 1152, x, (36,), rng)
    with np.errstate(invalid="ignore"):
        want = x.astype(np.float64) @ deq.astype(np.float64).T
    assert np.array_equal(np.isnan(got[0]), np.isnan(want)) and np.array_equal(np.isinf(got[0]), np.isinf(want))
    ok = np.isfinite(want)
    assert np.all(got[0][~ok & ~np.isnan(want)] == want[~ok & ~np.isnan(want)])
    assert np.allclose(got[0][ok], want[ok], rtol=1e-4, atol=1e-4)  # 1152 products of about 0.5 x 0.02


def test_the_form_rejects_what_it_does_not_cover(be):
    rng = np.random.default_rng(6)
    for m, k, cfg in ((5, 1152, (8, 1, 65)), (12, 1152, (8, 1, 50)), (5, 1152, (8, 1, -1)), (5, 1152, (8, 0, 36)), (5, 1152, (4, 1, 36)), (5, 1088, (8, 1, 36))):
        packed, scales, _ = make_weight("int8-grouped", 64, k, 64, rng)
        w = be.createQuantizedWeight(packed, scales, 64, k, T.resolveWeightFormat("int8-64", "f32"))
        with pytest.raises(L.TlhipError, match="config not applicable"):
            be._matmulQuantizedB(be.ops.tensorFromArray(make_x(m, k, "f32", rng), [m, k], "f32"), be.ops.transpose(w), None, L.KernelConfig.of(L.VARIANT_GEMV_F32, *cfg))
