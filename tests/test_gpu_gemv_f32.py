"""GPU parity of the f32-activation matrix-core GEMV (variant 6) at the sizes where it can go
wrong: rows around its 16-row operand tiles (three pieces a row), columns around its 128, a K
that ends inside a block, slices of unequal length, values that are not finite.

Tolerance: products are exact, so what is left is f32 rounding: two in the oracle's dequantised
weight, and in the sums (blocks of 32 or 64 k, then their scaled sums, slices, bias, add).  Each
rounds by at most 2^-24 of a partial sum, which the sum of the terms' magnitudes bounds, so a row
is held to 2e-6 of its norm and, where a row is one element that its terms may cancel in, that
element to 2^-21 (eight roundings) of the sum of their magnitudes."""
import numpy as np
import pytest

import torchlette_amd as T
from oracle import quant_oracle as O
from torchlette_amd import _lib as L
from helpers import fmt_name, make_weight, make_x, rel_l2

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def be():
    return T.getBackend()


def product(be, fmt, g, n, k, x, slices, rng):
    packed, scales, deq = make_weight(fmt, n, k, g, rng)
    w = be.createQuantizedWeight(packed, scales, n, k, T.resolveWeightFormat(fmt_name(fmt, g), "f32"))
    m = x.shape[0]
    xt = be.ops.tensorFromArray(x, [m, k], "f32")
    bias, other = rng.standard_normal(n).astype(np.float32), rng.standard_normal((m, n)).astype(np.float32)
    bt, ot = be.ops.tensorFromArray(bias, [n], "f32"), be.ops.tensorFromArray(other, [m, n], "f32")
    cfg = L.KernelConfig.of(L.VARIANT_GEMV_F32, slices) if slices else None
    ep = be.makeEpilogueChain([("bias", bt), ("binary", "add", ot)])
    got = [be._matmulQuantizedB(xt, be.ops.transpose(w), ep, cfg).numpy() for _ in range(2)]
    assert np.array_equal(got[0], got[1], equal_nan=True)
    for t in (xt, bt, ot, w):
        t.destroy()
    with np.errstate(invalid="ignore", over="ignore"):
        magnitudes = np.abs(x).astype(np.float64) @ np.abs(deq).astype(np.float64).T + np.abs(bias) + np.abs(other)
        return got[0], x.astype(np.float64) @ deq.astype(np.float64).T + bias + other, magnitudes


@pytest.mark.parametrize("fmt,g", [("int4-grouped", 32), ("int4-grouped", 64), ("int8-grouped", 64), ("int8-grouped", 128), ("int8-row", 0)])
@pytest.mark.parametrize("m", [1, 2, 5, 6, 10, 11, 16])
@pytest.mark.parametrize("n,k,slices", [(128, 128, 1), (129, 640, 1), (127, 640, 3), (300, 1152, 5), (1, 384, 2)])
def test_edges(be, fmt, g, m, n, k, slices):
    k += {"int8-row": 16, "int4-grouped": 32 if g == 32 else 0}.get(fmt, 0)  # K ends inside a block
    rng = np.random.default_rng(m * 1000 + n + k + g)
    got, want, magnitudes = product(be, fmt, g, n, k, make_x(m, k, "f32", rng, std=0.5), slices, rng)
    assert np.all(np.abs(got - want) <= 2.0**-21 * magnitudes)
    for r in range(m if n > 1 else 0):
        assert rel_l2(got[r], want[r]) <= 2e-6, r


@pytest.mark.parametrize("slices", [0, 3])  # the default, all of K in one workgroup; and K slices
def test_default_route_and_values_that_are_not_finite(be, slices):
    n, k, m = 1024, 2304, 5
    rng = np.random.default_rng(3)
    x = make_x(m, k, "f32", rng, std=0.5)
    x[1] *= np.float32(1e-30)
    x[2, 7], x[3, 9] = np.inf, np.nan
    got, want, magnitudes = product(be, "int8-grouped", 64, n, k, x, slices, rng)
    for r in (0, 1, 4):
        assert rel_l2(got[r], want[r]) <= 2e-6, r
    assert np.array_equal(np.isnan(got[2]), np.isnan(want[2])) and np.array_equal(np.sign(got[2]), np.sign(want[2]), equal_nan=True)
    assert np.all(np.isinf(got[2]) | np.isnan(got[2])) and np.all(np.isnan(got[3]))


@pytest.mark.parametrize("fmt,g", [("int4-grouped", 32), ("int8-grouped", 64), ("int8-row", 0)])
def test_subnormal_activations(be, fmt, g):
    """Rows around the smallest normal f32 and far below it.  The matrix cores keep subnormal bf16
    values, so a piece loses only what lies under their last bit, 2^-133: that much of each value,
    times the integer it meets, beside the sums' own rounding; and f32 sums round to 2^-149."""
    n, k, m = 256, 640, 5
    rng = np.random.default_rng(11)
    x = make_x(m, k, "f32", rng, std=0.5)
    for r, e in enumerate((-118, -124, -127, -130, -135)):
        x[r] = np.ldexp(x[r], e)
    packed, scales, deq = make_weight(fmt, n, k, g, rng)
    w = be.createQuantizedWeight(packed, scales, n, k, T.resolveWeightFormat(fmt_name(fmt, g), "f32"))
    xt = be.ops.tensorFromArray(x, [m, k], "f32")
    got = be._matmulQuantizedB(xt, be.ops.transpose(w), None, L.KernelConfig.of(L.VARIANT_GEMV_F32, 2)).numpy().astype(np.float64)
    d = np.abs(deq.astype(np.float64))
    want, magnitudes = x.astype(np.float64) @ deq.astype(np.float64).T, np.abs(x).astype(np.float64) @ d.T
    assert np.any(want[4] != 0)
    assert np.all(np.abs(got - want) <= 2.0**-21 * magnitudes + 2.0**-133 * d.sum(1) + 2.0**-145)


@pytest.mark.parametrize("fmt,g", [("int4-grouped", 32), ("int8-grouped", 64), ("int8-grouped", 256), ("int8-row", 0)])
@pytest.mark.parametrize("m", [1, 2, 5, 6, 10, 11, 16])
@pytest.mark.parametrize("n,k", [(1, 256), (131, 1280), (300, 2304)])  # one column; ten and eighteen steps on eight waves
def test_all_of_k_in_one_workgroup(be, fmt, g, m, n, k):
    rng = np.random.default_rng(m * 1000 + n + k + g)
    packed, scales, deq = make_weight(fmt, n, k, g, rng)
    w = be.createQuantizedWeight(packed, scales, n, k, T.resolveWeightFormat(fmt_name(fmt, g), "f32"))
    x = make_x(m, k, "f32", rng, std=0.5)
    bias, other = rng.standard_normal(n).astype(np.float32), rng.standard_normal((m, n)).astype(np.float32)
    xt, bt, ot = be.ops.tensorFromArray(x, [m, k], "f32"), be.ops.tensorFromArray(bias, [n], "f32"), be.ops.tensorFromArray(other, [m, n], "f32")
    ep = be.makeEpilogueChain([("bias", bt), ("binary", "add", ot)])
    want = x.astype(np.float64) @ deq.astype(np.float64).T + bias + other
    magnitudes = np.abs(x).astype(np.float64) @ np.abs(deq).astype(np.float64).T + np.abs(bias) + np.abs(other)
    for cols in (1, 2, 4) if m <= 10 else (1, 2):
        got = be._matmulQuantizedB(xt, be.ops.transpose(w), ep, L.KernelConfig.of(L.VARIANT_GEMV_F32, 8, cols)).numpy()
        assert np.all(np.abs(got - want) <= 2.0**-21 * magnitudes), cols  # the bound of the K slices above
