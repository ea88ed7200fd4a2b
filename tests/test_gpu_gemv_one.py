"""GPU parity: one activation row in the one-row form of the VALU kernel (gemv_one.hip), against the oracle."""
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

# lanes per row, waves, waves that share a row, workgroups per CU
GEOMETRIES = [(16, 4, 1, 4), (32, 8, 2, 2), (64, 4, 1, 2), (64, 8, 8, 1)]


@pytest.fixture(scope="module")
def be():
    return T.getBackend()


@pytest.mark.parametrize("xdt", ["f16", "f32"])
@pytest.mark.parametrize("fmt,g,n,k", [
    ("int4-grouped", 32, 1, 32),        # one row of one chunk: every other lane past its end
    ("int4-grouped", 64, 67, 1536),     # three chunks a lane on 16 lanes; rows off the workgroup
    ("int4-grouped", 32, 131, 12288),   # six a lane on 64; activations staged in several rounds
    ("int8-grouped", 64, 5, 64),
    ("int8-grouped", 128, 130, 5248),   # 328 chunks: a part of the lanes past the row's end
    ("int8-row", 0, 33, 48),
    ("int8-row", 0, 70, 6128),          # 383 chunks
    ("int8-grouped", 64, 24581, 64),    # more rows than are resident: four rounds on 16 lanes, the last with few
])
def test_one_row_matches_the_oracle(be, fmt, g, n, k, xdt):
    rng = np.random.default_rng(zlib.crc32(repr((fmt, g, n, k, xdt)).encode()))
    packed, scales, deq = make_weight(fmt, n, k, g, rng)
    x, bias = make_x(1, k, xdt, rng), rng.standard_normal(n).astype(np.float32)
    want = O.linear(x.astype(np.float32), deq, bias, "silu", threads=8)
    plain = O.linear(x.astype(np.float32), deq, bias, threads=8)
    ran = 0
    for lpr, waves, kw, resident in GEOMETRIES + [(16, 4, 1, 2)]:
        cfg = L.KernelConfig.of(L.VARIANT_GEMV, lpr, 1, waves, kw, resident, 3)
        try:
            got = run_linear(be, fmt, packed, scales, n, k, g, x, "f32", bias=bias, act="silu", fused=True, config=cfg)
        except L.TlhipError as e:
            assert "more chunks per lane" in str(e)
            continue
        ran += 1
        assert rel_l2(got, want) <= 2e-6, (lpr, kw)  # exact products, f32 sums: order noise only
        # a bias and nothing else, which comes with the weights
        got = run_linear(be, fmt, packed, scales, n, k, g, x, "f32", bias=bias, fused=True, config=cfg)
        assert rel_l2(got, plain) <= 2e-6, (lpr, kw)
    assert ran >= 1


def test_one_row_form_rejects_what_it_does_not_cover(be):
    rng = np.random.default_rng(5)
    packed, scales, _ = make_weight("int8-row", 64, 1024, 0, rng)
    for m, cfg in ((2, (64, 1, 4, 1, 4, 3)), (1, (8, 1, 4, 1, 4, 3)), (1, (64, 2, 4, 1, 4, 3)), (1, (64, 1, 2, 1, 4, 3)),
                   (1, (64, 1, 4, 8, 4, 3)), (1, (64, 1, 8, 1, 8, 3)), (1, (64, 1, 4, 1, 0, 3))):
        with pytest.raises(L.TlhipError, match="config not applicable"):
            run_linear(be, "int8-row", packed, scales, 64, 1024, 0, make_x(m, 1024, "f16", rng), "f32", config=L.KernelConfig.of(0, *cfg))


def test_a_group_whose_problems_have_their_own_rows(be):
    """Problems of one K on different activation rows, residuals of both types, one launch."""
    rng = np.random.default_rng(11)
    k, ns = 1024, (300, 64, 1111)
    probs, keep, wants = (L.GemvProblem * 3)(), [], []
    for i, n in enumerate(ns):
        packed, scales, deq = make_weight("int8-grouped", n, k, 64, rng)
        w = be.createQuantizedWeight(packed, scales, n, k, T.resolveWeightFormat("int8-64", "f32"))
        x = make_x(1, k, "f16", rng)
        res = make_x(1, n, "f16" if i == 1 else "f32", rng)
        xt, rt = be.ops.tensorFromArray(x, [1, k], "f16"), be.ops.tensorFromArray(res, [1, n], "f16" if i == 1 else "f32")
        out = be._alloc([1, n], "f32")
        ep = L.Epilogue()
        ep.n_ops = 2
        ep.ops[0] = L.EpilogueOp(L.EPI_UNARY, L.UNARY["relu"], None, 0, 0)
        ep.ops[1] = L.EpilogueOp(L.EPI_BINARY, L.BINARY["mul" if i else "sub"], rt.ptr, L.F16 if i == 1 else L.F32, 1)
        probs[i].w, probs[i].x, probs[i].y, probs[i].epilogue = be._qweight(w, transposed=False), xt.ptr, out.ptr, C.pointer(ep)
        keep += [w, xt, rt, ep]
        lin = np.maximum(O.linear(x.astype(np.float32), deq), 0)
        wants.append((out, lin * res.astype(np.float32) if i else lin - res))
    L.call("tlhip_gemv_grouped", probs, 3, L.F16, L.F32, 1.0, be.stream)
    for out, want in wants:
        assert rel_l2(out.numpy(), want) <= 2e-6


@pytest.mark.parametrize("fmt,g,ff,hidden", [("int4-grouped", 32, 1104, 1024), ("int8-row", 0, 832, 2048), ("int8-grouped", 64, 3072, 4096)])
def test_gate_and_up_in_one_launch(be, fmt, g, ff, hidden):
    """tlhip_mlp_decode at one row: h is the product of both projections rounded to f16, as two
    launches and a multiply leave it."""
    rng = np.random.default_rng(zlib.crc32(repr((fmt, ff, hidden)).encode()))
    ws, names = [], [fmt_name(fmt, g)] * 2 + ["int8-row"]
    for n, k in ((ff, hidden), (ff, hidden), (96, ff)):
        packed, scales, deq = make_weight(*((fmt, n, k, g) if n == ff else ("int8-row", n, k, 0)), rng)
        ws.append((packed, scales, deq, n, k))
    gate, up, down = (be.createQuantizedWeight(p, s, n, k, T.resolveWeightFormat(nm, "f32")) for (p, s, _, n, k), nm in zip(ws, names))
    x = make_x(1, hidden, "f16", rng, std=0.3)
    xt, h, y = be.ops.tensorFromArray(x, [1, hidden], "f16"), be._alloc([1, ff], "f16"), be._alloc([1, 96], "f32")
    q = [be._qweight(w, transposed=False) for w in (gate, up, down)]
    L.call("tlhip_mlp_decode", C.byref(q[0]), C.byref(q[1]), C.byref(q[2]), L.UNARY["gelu_tanh"], xt.ptr, L.F16, 1, h.ptr, y.ptr, L.F32, None,
           be.stream)
    xf = x.astype(np.float32)
    f16 = lambda a: a.astype(np.float16).astype(np.float32)  # noqa: E731
    want = O.gated(f16(O.linear(xf, ws[0][2])), f16(O.linear(xf, ws[1][2])), "gelu_tanh")
    got = h.numpy().astype(np.float32)
    assert rel_l2(got, want) <= 4e-4  # one rounding to f16 (2.8e-4), and a projection on the other side of one now and then
    assert rel_l2(y.numpy(), O.linear(got, ws[2][2])) <= 2e-6
