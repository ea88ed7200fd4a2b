"""GPU parity: 17..64 f16 rows with all of K in one workgroup (gemm_rows.hip), against the oracle."""
import zlib

import numpy as np
import pytest

import torchlette_amd as T
from oracle import quant_oracle as O
from torchlette_amd import _lib as L
from helpers import make_weight, make_x, rel_l2
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
    ran = 0
    for cols in (1, 2, 3, 4):
        try:
            got = run_linear(be, fmt, packed, scales, n, k, g, x, "f32", bias=bias, act="silu", fused=True,
                             config=L.KernelConfig.of(L.VARIANT_GEMV_MFMA, 8, 0, 0, 0, cols))
        except L.TlhipError as e:
            assert cols > 2 and "not applicable" in str(e)  # more registers than a lane has
            continue
        ran += 1
        assert rel_l2(got, want) <= 2e-6, cols  # exact products, f32 sums: order noise only
    assert ran >= 2


def test_the_width_is_not_read_with_the_other_forms_fields(be):
    fmt, g, n, k, m = "int4-grouped", 32, 512, 2048, 40
    rng = np.random.default_rng(7)
    packed, scales, _ = make_weight(fmt, n, k, g, rng)
    x = make_x(m, k, "f16", rng)
    plain, with_width = (run_linear(be, fmt, packed, scales, n, k, g, x, "f32", config=L.KernelConfig.of(L.VARIANT_GEMV_MFMA, 8, 2, 8, 2, p4))
                         for p4 in (0, 2))
    assert np.array_equal(plain.view(np.uint32), with_width.view(np.uint32))
