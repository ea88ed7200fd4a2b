"""GPU parity: values that are not finite, where lanes lie past a row's end (they work on its last chunk again and must not add it)."""
import zlib

import numpy as np
import pytest

import torchlette_amd as T
from torchlette_amd import _lib as L
from helpers import fmt_name, make_weight, make_x
from test_gpu_gemv import run_linear

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def be():
    return T.getBackend()


def same_kind(got, want):
    got, want = np.asarray(got, np.float64).ravel(), np.asarray(want, np.float64).ravel()
    return np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(got[np.isinf(want)], want[np.isinf(want)]) and not np.isinf(got[np.isfinite(want)]).any()


def product(x, deq):
    with np.errstate(invalid="ignore"):
        return x.astype(np.float64) @ deq.astype(np.float64).T


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("xdt", ["f16", "f32"])
@pytest.mark.parametrize("fmt,g,n,k", [
    ("int4-grouped", 32, 67, 1312),    # 41 chunks
    ("int8-grouped", 64, 130, 5248),   # 328
    ("int8-row", 0, 70, 6128),         # 383
])
def test_one_row_with_its_last_chunk_not_finite(be, fmt, g, n, k, xdt, value):
    rng = np.random.default_rng(zlib.crc32(repr((fmt, k, xdt)).encode()))
    packed, scales, deq = make_weight(fmt, n, k, g, rng)
    x = make_x(1, k, xdt, rng)
    x[0, k - 3] = value
    want = product(x, deq)
    ran = 0
    for lpr, waves, kw, resident in [(16, 4, 1, 4), (32, 8, 2, 2), (64, 4, 1, 2), (64, 8, 8, 1)]:
        try:
            got = run_linear(be, fmt, packed, scales, n, k, g, x, "f32", config=L.KernelConfig.of(L.VARIANT_GEMV, lpr, 1, waves, kw, resident, 3))
        except L.TlhipError as e:
            assert "more chunks per lane" in str(e)
            continue
        ran += 1
        assert same_kind(got, want), (lpr, kw)
    assert ran >= 2


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("xdt", ["f16", "f32"])
@pytest.mark.parametrize("fmt,g,n,k", [
    ("int4-grouped", 32, 67, 1312),
    ("int8-grouped", 64, 130, 5248),
    ("int8-row", 0, 70, 6128),
])
def test_one_to_five_rows_with_a_last_chunk_not_finite(be, fmt, g, n, k, xdt, value):
    """The kernel whose lanes hold several chunks of several rows at a time, and its 4 x 4 x 4 form."""
    rng = np.random.default_rng(zlib.crc32(repr((fmt, k, xdt)).encode()))
    packed, scales, deq = make_weight(fmt, n, k, g, rng)
    for m in (1, 2, 3, 5):
        x = make_x(m, k, xdt, rng)
        x[m // 2, k - 3] = value
        want = product(x, deq)
        configs = [(16, 1, 4, 1, 2, 0), (32, 2, 8, 2, 2, 0), (64, 1, 4, 4, 8, 0), (64, 4, 8, 1, 2, 0)]
        if fmt == "int4-grouped" and xdt == "f16" and m <= 4:
            configs += [(16, 1, 4, 1, 2, 1), (16, 1, 8, 2, 8, 1)]
        for c in configs:
            got = run_linear(be, fmt, packed, scales, n, k, g, x, "f32", config=L.KernelConfig.of(L.VARIANT_GEMV, *c))
            assert same_kind(got, want), (m, c)
