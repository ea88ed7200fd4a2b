"""GPU parity: one row whose lanes hold five chunks each, an instance of its own (K = 5120 and 9728 of int8), against the oracle."""
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


@pytest.mark.parametrize("xdt", ["f16", "f32"])
@pytest.mark.parametrize("fmt,g,n,k,lanes,kw", [
    ("int8-grouped", 64, 67, 5120, 64, 1),    # five chunks a lane, none past the end
    ("int8-row", 0, 130, 9728, 64, 2),        # 608 chunks on 128 lanes: the last 32 without a fifth
    ("int8-grouped", 128, 33, 1152, 16, 1),   # 72 chunks on 16
    ("int4-grouped", 32, 131, 9728, 64, 1),   # 304 on 64 (f32 rows: no such instance)
])
def test_five_chunks_a_lane(be, fmt, g, n, k, lanes, kw, xdt):
    rng = np.random.default_rng(zlib.crc32(repr((fmt, n, k, xdt)).encode()))
    packed, scales, deq = make_weight(fmt, n, k, g, rng)
    x = make_x(1, k, xdt, rng)
    cfg = L.KernelConfig.of(L.VARIANT_GEMV, lanes, 1, 4, kw, 2, 3)
    if fmt == "int4-grouped" and xdt == "f32":
        with pytest.raises(L.TlhipError, match="more chunks per lane"):
            run_linear(be, fmt, packed, scales, n, k, g, x, "f32", config=cfg)
        return
    got = run_linear(be, fmt, packed, scales, n, k, g, x, "f32", config=cfg)
    assert rel_l2(got, O.linear(x.astype(np.float32), deq, threads=8)) <= 2e-6  # exact products, f32 sums: order noise only
