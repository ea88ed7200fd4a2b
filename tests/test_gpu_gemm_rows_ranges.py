"""GPU parity of the 17..64 row kernel (gemm_rows.hip) where its waves' ranges of K and the patch of their scales
can go wrong, against the oracle."""
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


@pytest.mark.parametrize("m", [17, 48, 64])
@pytest.mark.parametrize("fmt,g,n,k", [
    ("int4-grouped", 32, 52, 1024),    # a step a wave
    ("int4-grouped", 32, 100, 7168),   # seven steps: at 64 rows and three blocks the scales come in two parts
    ("int4-grouped", 32, 49, 17408),   # 17 steps: in two parts or three everywhere
    ("int8-grouped", 64, 50, 16512),   # 129 steps: sixteen a wave but one of seventeen
    ("int8-grouped", 512, 36, 18432),  # 18 steps, a scale for four
    ("int8-row", 0, 51, 17408),
])
def test_ranges_and_their_scales(be, fmt, g, n, k, m):
    rng = np.random.default_rng(zlib.crc32(repr((fmt, g, n, k, m)).encode()))
    packed, scales, deq = make_weight(fmt, n, k, g, rng)
    x = make_x(m, k, "f16", rng)
    want = O.linear(x.astype(np.float32), deq, threads=8)
    most = {17: 4, 48: 4 if fmt == "int4-grouped" else 3, 64: 3 if fmt == "int4-grouped" else 2}[m]
    for cols in range(1, most + 1):
        got = run_linear(be, fmt, packed, scales, n, k, g, x, "f32", fused=True, config=L.KernelConfig.of(L.VARIANT_GEMV_MFMA, 8, 0, 0, 0, cols))
        assert rel_l2(got, want) <= 2e-6, cols  # exact products, f32 sums of at most 2304 a wave: order noise only


@pytest.mark.parametrize("m", [17, 33, 40, 64])
@pytest.mark.parametrize("fmt,g,n,k", [("int4-grouped", 32, 52, 1152), ("int8-grouped", 64, 49, 640), ("int8-row", 0, 36, 17408)])
def test_a_share_of_the_rows(be, fmt, g, n, k, m):
    """One or two tiles of rows a workgroup: a last share of one row, of eight, of a whole tile; bias, residual and store at the rows' places."""
    rng = np.random.default_rng(zlib.crc32(repr((fmt, g, n, k, m)).encode()))
    packed, scales, deq = make_weight(fmt, n, k, g, rng)
    x, bias, other = make_x(m, k, "f16", rng), rng.standard_normal(n).astype(np.float32), rng.standard_normal((m, n)).astype(np.float32)
    w = be.createQuantizedWeight(packed, scales, n, k, T.resolveWeightFormat(fmt_name(fmt, g), "f32"))
    qw, xt, bt = be._qweight(w, False), be.ops.tensorFromArray(x, [m, k], "f16"), be.ops.tensorFromArray(bias, [n], "f32")
    want = O.linear(x.astype(np.float32), deq, bias, threads=8) + other
    for tiles in (1, 2):
        y = be.ops.tensorFromArray(other, [m, n], "f32")  # the residual is the output itself
        ep, cfg = be.makeEpilogueChain([("bias", bt), ("binary", "add", y)]), L.KernelConfig.of(L.VARIANT_GEMV_MFMA, 8, 0, 0, 0, 1, 0, tiles)
        args = (C.byref(qw), xt.ptr, L.F16, m, y.ptr, L.F32, 1.0, C.byref(ep), C.byref(cfg), None)
        if tiles >= (m + 15) // 16:
            with pytest.raises(L.TlhipError, match="not applicable"):
                L.call("tlhip_matmul_quantized_config", *args)
            continue
        L.call("tlhip_matmul_quantized_config", *args)
        assert rel_l2(y.numpy(), want) <= 2e-6, tiles  # exact products, f32 sums: order noise only
