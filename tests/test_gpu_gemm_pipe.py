"""GPU parity of the eight-wave tiled GEMM (tiled_direct with tile K 64) at the sizes where it
can go wrong: one row and column more and less than a tile, one, two, three and five steps
of 64 k (its buffers rotate over two and three), N that forbids 16-byte pieces of a row, the
whole chain, K slices.

Tolerances: the grouped formats round q * s once to f16 (2^-11 relative, uniform: rel-L2 about
2.8e-4 on each weight, so on the sum too), an f16 output once more: <= 1e-3 as for the other
prefill kernels.  int8 per row multiplies exact integers and sums in f32: <= 5e-6."""
import numpy as np
import pytest

import torchlette_amd as T
from oracle import quant_oracle as O
from torchlette_amd import _lib as L
from helpers import f16_round, fmt_name, make_weight, make_x, rel_l2

pytestmark = pytest.mark.gpu

TILES = [(256, 256, 2, 4), (256, 192, 2, 4), (256, 128, 4, 2), (128, 128, 2, 4), (64, 128, 2, 4)]
FORMATS = [("int4-grouped", 32), ("int4-grouped", 64), ("int8-grouped", 64), ("int8-grouped", 128), ("int8-row", 0)]


@pytest.fixture(scope="module")
def be():
    return T.getBackend()


@pytest.mark.parametrize("fmt,g", FORMATS)
@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("dm,dn,k,ks", [(0, 0, 128, 0), (1, 8, 64, 0), (-1, -8, 192, 0), (17, 1, 320, 0), (3, -3, 128, 0), (5, 16, 512, 4), (5, 3, 512, 2)])
def test_tile_edges(be, fmt, g, tile, dm, dn, k, ks):
    if g and k % g:
        pytest.skip("not whole groups")
    m, n = tile[0] + dm, tile[1] + dn
    rng = np.random.default_rng(m * 131 + n * 7 + k + g)
    packed, scales, deq = make_weight(fmt, n, k, g, rng)
    w = be.createQuantizedWeight(packed, scales, n, k, T.resolveWeightFormat(fmt_name(fmt, g), "f32"))
    x = make_x(m, k, "f16", rng, std=0.5)
    bias, other = f16_round(rng.standard_normal(n) * 0.1), f16_round(rng.standard_normal((m, n)))
    xt = be.ops.tensorFromArray(x, [m, k], "f16")
    bt = be.ops.tensorFromArray(bias.astype(np.float16), [n], "f16")
    ot = be.ops.tensorFromArray(other.astype(np.float32), [m, n], "f32")
    cfg = L.KernelConfig.of(3, tile[0], tile[1], 64, tile[2], tile[3], ks)
    ep = be.makeEpilogueChain([("bias", bt), ("unary", "silu"), ("binary", "add", ot)])
    got = be._matmulQuantizedB(xt, be.ops.transpose(w), ep, cfg).numpy()
    want = (O.linear(x.astype(np.float32), deq, bias.astype(np.float32), "silu", threads=8) + other).astype(np.float32)
    tol = 5e-6 if fmt == "int8-row" else 1e-3
    for r0 in range(0, m, 64):       # by blocks: one wrong piece of a tile cannot hide
        for c0 in range(0, n, 64):
            assert rel_l2(got[r0:r0 + 64, c0:c0 + 64], want[r0:r0 + 64, c0:c0 + 64]) <= tol, (r0, c0)
    again = be._matmulQuantizedB(xt, be.ops.transpose(w), ep, cfg).numpy()
    assert np.array_equal(got, again)
    for t in (xt, bt, ot, w):
        t.destroy()
