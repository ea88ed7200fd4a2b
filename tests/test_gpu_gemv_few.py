"""GPU parity: 2..16 f16 rows with all of K in one workgroup (gemv_few.hip), against the oracle."""
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

# blocks of columns, columns: full, an even share that leaves lanes idle, the smallest
GEOMETRIES = [(1, 16), (1, 4), (2, 20), (3, 48), (4, 52), (6, 96)]


@pytest.fixture(scope="module")
def be():
    return T.getBackend()


def few(nb, cols):
    return L.KernelConfig.of(L.VARIANT_GEMV_MFMA, 8, 0, cols, 0, nb)


@pytest.mark.parametrize("m", [2, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("fmt,g,n,k", [
    ("int4-grouped", 32, 101, 128),    # one step: seven waves have none; columns off four and off the workgroup
    ("int4-grouped", 32, 260, 2432),   # 19 steps: two and three a wave
    ("int4-grouped", 32, 36, 16384),   # sixteen steps a wave: the scales in two loads
    ("int8-grouped", 64, 131, 1152),
    ("int8-grouped", 128, 100, 2176),  # 17 steps, a scale each
    ("int8-grouped", 256, 96, 4864),   # a scale for two steps
    ("int8-row", 0, 515, 1920),
])
def test_few_rows_match_the_oracle(be, fmt, g, n, k, m):
    rng = np.random.default_rng(zlib.crc32(repr((fmt, g, n, k, m)).encode()))
    packed, scales, deq = make_weight(fmt, n, k, g, rng)
    x, bias = make_x(m, k, "f16", rng), rng.standard_normal(n).astype(np.float32)
    want = O.linear(x.astype(np.float32), deq, bias, "silu", threads=8)
    for nb, cols in GEOMETRIES:
        got = run_linear(be, fmt, packed, scales, n, k, g, x, "f32", bias=bias, act="silu", fused=True, config=few(nb, cols))
        assert rel_l2(got, want) <= 2e-6, (nb, cols)  # exact products, f32 sums: order noise only


def test_few_rows_form_rejects_what_it_does_not_cover(be):
    rng = np.random.default_rng(6)
    packed, scales, _ = make_weight("int8-row", 64, 1024, 0, rng)
    odd = make_weight("int8-row", 64, 1040, 0, rng)
    for m, k, cfg in ((17, 1024, (8, 0, 16, 0, 1)), (4, 1024, (8, 0, 18, 0, 2)), (4, 1024, (8, 0, 20, 0, 1)), (4, 1024, (8, 0, 16, 0, 2, 1)),
                      (4, 1024, (8, 0, 16, 0, 3)), (4, 1024, (8, 0, 80, 0, 5)), (4, 1024, (4, 0, 16, 0, 1)), (4, 1040, (8, 0, 16, 0, 1))):
        p, s = (packed, scales) if k == 1024 else odd[:2]
        with pytest.raises(L.TlhipError, match="config not applicable"):
            run_linear(be, "int8-row", p, s, 64, k, 0, make_x(m, k, "f16", rng), "f32", config=L.KernelConfig.of(L.VARIANT_GEMV_MFMA, *cfg))


@pytest.mark.parametrize("m,ydt", [(3, "f16"), (11, "f32")])
def test_a_group_with_residuals(be, m, ydt):
    """Three problems on the same rows in one launch; residuals of both types, chains of two steps."""
    rng = np.random.default_rng(m)
    k, ns = 1280, (300, 61, 1111)
    x = make_x(m, k, "f16", rng)
    xt = be.ops.tensorFromArray(x, [m, k], "f16")
    probs, keep, wants = (L.GemvProblem * 3)(), [], []
    for i, n in enumerate(ns):
        packed, scales, deq = make_weight("int8-grouped", n, k, 64, rng)
        w = be.createQuantizedWeight(packed, scales, n, k, T.resolveWeightFormat("int8-64", ydt))
        rdt = "f16" if i == 1 else "f32"
        res = make_x(m, n, rdt, rng)
        rt, out = be.ops.tensorFromArray(res, [m, n], rdt), be._alloc([m, n], ydt)
        ep = L.Epilogue()
        ep.n_ops = 2
        ep.ops[0] = L.EpilogueOp(L.EPI_UNARY, L.UNARY["relu"], None, 0, 0)
        ep.ops[1] = L.EpilogueOp(L.EPI_BINARY, L.BINARY["mul" if i else "sub"], rt.ptr, L.F16 if i == 1 else L.F32, m)
        probs[i].w, probs[i].x, probs[i].y, probs[i].epilogue = be._qweight(w, transposed=False), xt.ptr, out.ptr, C.pointer(ep)
        keep += [w, rt, ep]
        lin = np.maximum(O.linear(x.astype(np.float32), deq), 0)
        wants.append((out, lin * res.astype(np.float32) if i else lin - res))
    L.call("tlhip_gemv_grouped_rows", probs, 3, L.F16, m, L.F16 if ydt == "f16" else L.F32, 1.0, be.stream)
    for out, want in wants:
        assert rel_l2(out.numpy(), want) <= (4e-4 if ydt == "f16" else 2e-6)  # f16: one rounding, 2.8e-4 at most


@pytest.mark.parametrize("m", [2, 7, 16])
@pytest.mark.parametrize("fmt,g,ff,hidden", [("int4-grouped", 32, 1104, 1024), ("int8-row", 0, 832, 2048), ("int8-grouped", 128, 3072, 1152)])
def test_gate_and_up_in_one_launch(be, fmt, g, ff, hidden, m):
    """tlhip_mlp_decode: h is the product of both projections rounded to f16, as two launches and a
    multiply leave it."""
    rng = np.random.default_rng(zlib.crc32(repr((fmt, ff, hidden, m)).encode()))
    ws, names = [], [fmt_name(fmt, g)] * 2 + ["int8-row"]
    for n, k in ((ff, hidden), (ff, hidden), (96, ff)):
        packed, scales, deq = make_weight(*((fmt, n, k, g) if n == ff else ("int8-row", n, k, 0)), rng)
        ws.append((packed, scales, deq, n, k))
    tensors = [be.createQuantizedWeight(p, s, n, k, T.resolveWeightFormat(nm, "f32")) for (p, s, _, n, k), nm in zip(ws, names)]
    x = make_x(m, hidden, "f16", rng, std=0.3)
    xt, h, y = be.ops.tensorFromArray(x, [m, hidden], "f16"), be._alloc([m, ff], "f16"), be._alloc([m, 96], "f32")
    q = [be._qweight(w, transposed=False) for w in tensors]
    L.call("tlhip_mlp_decode", C.byref(q[0]), C.byref(q[1]), C.byref(q[2]), L.UNARY["silu"], xt.ptr, L.F16, m, h.ptr, y.ptr, L.F32, None,
           be.stream)
    xf = x.astype(np.float32)
    f16 = lambda a: a.astype(np.float16).astype(np.float32)  # noqa: E731
    want = O.gated(f16(O.linear(xf, ws[0][2])), f16(O.linear(xf, ws[1][2])), "silu")
    got = h.numpy().astype(np.float32)
    assert rel_l2(got, want) <= 4e-4  # one rounding to f16 (2.8e-4), and a projection on the other side of one now and then
    assert rel_l2(y.numpy(), O.linear(got, ws[2][2])) <= 2e-6
