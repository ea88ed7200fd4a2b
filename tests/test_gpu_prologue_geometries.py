"""GPU parity: the geometries that one and two rows with a prologue take by their sizes, against the oracle."""
import zlib

import numpy as np
import pytest

import torchlette_amd as T
from oracle import quant_oracle as O
from torchlette_amd import _lib as L
from helpers import f16_round, fmt_name, make_weight, make_x, rel_l2

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def be():
    return T.getBackend()


@pytest.mark.parametrize("fmt,g,n,k,m", [
    ("int4-grouped", 32, 1029, 3072, 2),     # 64 lanes to a row
    ("int4-grouped", 32, 2050, 3104, 2),     # 32, with a prologue of either kind
    ("int4-grouped", 32, 2050, 9728, 2),     # the 4x4x4 form behind a gated multiply
    ("int4-grouped", 32, 4099, 3072, 2),     # ... and behind an RMSNorm too
    ("int8-grouped", 64, 1030, 8192, 2),
    ("int8-row", 0, 2049, 2064, 2),
    ("int8-grouped", 64, 2048, 12288, 1),    # behind an RMSNorm the VALU kernel
    ("int8-row", 0, 3075, 12304, 1),         # behind a gated multiply
])
def test_rows_with_a_prologue(be, fmt, g, n, k, m):
    rng = np.random.default_rng(zlib.crc32(repr((fmt, n, k, m)).encode()))
    packed, scales, deq = make_weight(fmt, n, k, g, rng)
    w = be.createQuantizedWeight(packed, scales, n, k, T.resolveWeightFormat(fmt_name(fmt, g), "f16"))
    x, up = make_x(m, k, "f16", rng, std=0.5), make_x(m, k, "f16", rng, std=0.5)
    nw = (1.0 + 0.1 * rng.standard_normal(k)).astype(np.float32)
    xt, ut, nt = be.ops.tensorFromArray(x, [m, k], "f16"), be.ops.tensorFromArray(up, [m, k], "f16"), be.ops.tensorFromArray(nw, [k], "f32")
    xf, uf = x.astype(np.float32), up.astype(np.float32)
    # activations rounded to f16 once on either side, a neighbour's rounding now and then, and the output's
    got = be.linearAfterRMSNorm(xt, nt, 1e-6, w).numpy().astype(np.float32)
    assert rel_l2(got, O.linear(f16_round(O.rmsnorm(xf, nw, 1e-6)).astype(np.float32), deq, threads=8)) <= 1e-3
    got = be.linearAfterGatedMul(xt, ut, "silu", w).numpy().astype(np.float32)
    assert rel_l2(got, O.linear(f16_round(O.gated(xf, uf, "silu")).astype(np.float32), deq, threads=8)) <= 1e-3
