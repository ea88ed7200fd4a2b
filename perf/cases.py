"""The work that a program built on this library has it do, as cases that can be timed.

A case is a dict of plain values.  Its ``path`` is one of

``linear``  one Linear on a packed weight through ``tlhip_matmul_quantized``: a prompt
            (prefill), a short prompt, a single small call.
``decode``  one decode step through the Linears of ``layers`` decoder layers: RMSNorm ->
            q, k, v -> o + residual -> RMSNorm -> act(gate) * up -> down + residual.
            (Attention itself is not part of the library: o reads the q rows.)  With
            ``graph`` the step is captured once and replayed, as a serving loop does; one
            row with f16 activations takes the fused-prologue entry points there.
``head``    an LM head and the top-k of every row of its logits.
``load``    quantize-at-load of a weight that is in device memory, and its explicit
            dequantisation.

Buffers are the caller's, as at the C ABI; calls go to the library's own stream.
"""
import ctypes as C
import math

import torch

import torchlette_amd as T
from torchlette_amd import _lib as L

F16, F32 = L.F16, L.F32
TORCH = {"f16": torch.float16, "f32": torch.float32}
CODE = {"f16": F16, "f32": F32}
FORMATS = {"int4-32": (L.FMT_INT4_GROUPED, 32), "int8-64": (L.FMT_INT8_GROUPED, 64),
           "int8-128": (L.FMT_INT8_GROUPED, 128), "int8-row": (L.FMT_INT8_ROW, 0)}
EPS = 1e-6


def listed():
    return [
        # a small call: one row through a 3 MB down projection in the frontend's own types; launch and host path
        dict(name="linear 1x1024x3072 int8-64", path="linear", fmt="int8-64", n=1024, k=3072, m=1, x="f32",
             bias=True, act="none", residual=False),
        # one token of a 0.6B model, replayed from a graph: 112 launches of 1-3 MB each
        dict(name="token 0.6B graph", path="decode", fmt="int4-32", layers=28, hidden=1024, q=2048, kv=1024, ffn=3072,
             m=1, x="f16", act="silu", graph=True),
        # single-stream decode on an 8B model, issued call by call (four of its layers)
        dict(name="decode 8B m1", path="decode", fmt="int4-32", layers=4, hidden=4096, q=4096, kv=1024, ffn=12288, m=1,
             x="f16", act="silu", graph=False),
        # the same model serving a batch of 16
        dict(name="decode 8B m16", path="decode", fmt="int4-32", layers=4, hidden=4096, q=4096, kv=1024, ffn=12288, m=16,
             x="f16", act="silu", graph=False),
        # the frontend's own default types: f32 activations on int8 groups of 64, five rows
        dict(name="decode 2B f32 m5", path="decode", fmt="int8-64", layers=4, hidden=2304, q=2048, kv=1024, ffn=9216,
             m=5, x="f32", act="gelu_tanh", graph=False),
        # a speculative-decoding check or a large batch: more rows than decode, fewer than prefill
        dict(name="verify 8B m48", path="decode", fmt="int4-32", layers=4, hidden=4096, q=4096, kv=1024, ffn=12288, m=48,
             x="f16", act="silu", graph=False),
        # prompts through the gate projection of an 8B model with its fused epilogue
        dict(name="prefill 512 int4", path="linear", fmt="int4-32", n=12288, k=4096, m=512, x="f16", bias=True,
             act="silu", residual=False),
        dict(name="prefill 2048 int4", path="linear", fmt="int4-32", n=12288, k=4096, m=2048, x="f16", bias=True,
             act="gelu_tanh", residual=False),
        # a short prompt of no round length, f32 activations, a down projection in the reference's format
        dict(name="prefill 333 f32 int8-64", path="linear", fmt="int8-64", n=2304, k=9216, m=333, x="f32", bias=True,
             act="none", residual=False),
        # the largest: a batch of long prompts
        dict(name="prefill 8192 int8-64", path="linear", fmt="int8-64", n=12288, k=4096, m=8192, x="f16", bias=False,
             act="none", residual=False),
        # a 256 000-word LM head for eight sequences, and the 64 candidates of each for the sampler
        dict(name="head 256000x2304 m8", path="head", fmt="int8-row", n=256000, k=2304, m=8, x="f16", topk=64),
        # quantize-at-load and the explicit dequantisation of one large weight
        dict(name="load 12288x4096", path="load", fmt="int8-64", n=12288, k=4096),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _k(rng, lo, hi, fmt):
    """A K that `fmt` takes: whole groups; half of the draws are whole multiples of 128."""
    step = 128 if (fmt == "int8-128" or rng.random() < 0.5) else {"int4-32": 32, "int8-64": 64, "int8-row": 16}[fmt]
    return max(step, _log(rng, lo, hi) // step * step)


def draw(rng):
    path = rng.choices(["linear", "decode", "head", "load"], [6, 4, 1, 1])[0]
    fmt = rng.choice(list(FORMATS))
    if path == "linear":
        n = _log(rng, 1024, 16384)
        if rng.random() < 0.75:
            n = max(64, n // 64 * 64)
        k = _k(rng, 1024, 12288, fmt)
        most = 8192 * 12288 * 4096 // (n * k)
        return dict(path=path, fmt=fmt, n=n, k=k, m=_log(rng, 1, max(1, min(8192, most))),
                    x=rng.choice(["f16", "f16", "f16", "f32"]), bias=rng.random() < 0.5,
                    act=rng.choice(["none", "silu", "gelu_tanh", "relu"]), residual=rng.random() < 0.25)
    if path == "decode":
        hidden = _log(rng, 768, 4096) // 128 * 128
        x = rng.choice(["f16", "f16", "f16", "f32"])
        ffn = int(hidden * rng.uniform(2.5, 4.0)) // 128 * 128
        q = int(hidden * rng.choice([0.75, 1, 1, 2])) // 128 * 128
        m = rng.choice([1, 1, 2, 3, 4, 6, 8, 12, 16, _log(rng, 17, 128)])
        return dict(path=path, fmt=fmt, layers=rng.randint(3, 6), hidden=hidden, q=q, kv=rng.choice([512, 1024]), ffn=ffn,
                    m=m, x=x, act=rng.choice(["silu", "gelu_tanh"]), graph=rng.random() < 0.4)
    if path == "head":
        return dict(path=path, fmt=fmt, n=_log(rng, 32000, 260000), k=_k(rng, 1024, 4096, fmt),
                    m=rng.choice([1, 1, 2, 4, 7, 8, 16]), x="f16", topk=rng.choice([1, 20, 50, 64, 100]))
    return dict(path=path, fmt=rng.choice(["int8-64", "int8-128"]), n=_log(rng, 256, 16384), k=_log(rng, 4, 96) * 128)


# ---------------------------------------------------------------------------- inputs

def _weight(gen, fmt, n, k):
    """A packed weight of trained-like values: normal integers, standard deviation 0.02."""
    code, group = FORMATS[fmt]
    cuda = dict(device="cuda", generator=gen)
    if fmt == "int4-32":
        q = (torch.randn(n, k, **cuda) * 2.5).round_().clamp_(-8, 7).to(torch.int32).bitwise_and_(15)
        lo, hi = q[:, 0::2].to(torch.uint8), q[:, 1::2].to(torch.uint8)
        packed = lo | (hi << 4)
        std = 2.5
    else:
        packed = (torch.randn(n, k, **cuda) * 35.0).round_().clamp_(-127, 127).to(torch.int8)
        std = 35.0 if fmt == "int8-row" else 35.0 / 127.0
    per = torch.rand(n, **cuda) if fmt == "int8-row" else torch.rand(n, k // group, **cuda)
    scales = (0.02 / std) * (0.7 + 0.6 * per)
    if fmt != "int8-row":
        scales = scales.to(torch.float16)
    packed, scales = packed.contiguous(), scales.contiguous()
    return packed, scales, L.QWeight(code, group, n, k, packed.data_ptr(), scales.data_ptr())


def _epilogue(*ops):
    ep = L.Epilogue()
    ep.n_ops = len(ops)
    for i, op in enumerate(ops):
        if op[0] == "bias":
            ep.ops[i] = L.EpilogueOp(L.EPI_BIAS, 0, op[1].data_ptr(), CODE["f16" if op[1].dtype == torch.float16 else "f32"], 1)
        elif op[0] == "unary":
            ep.ops[i] = L.EpilogueOp(L.EPI_UNARY, L.UNARY[op[1]], None, 0, 0)
        else:  # ("add" or "mul", a tensor [m, n])
            ep.ops[i] = L.EpilogueOp(L.EPI_BINARY, L.BINARY[op[0]], op[1].data_ptr(),
                                     CODE["f16" if op[1].dtype == torch.float16 else "f32"], op[1].shape[0])
    return ep


class _Graph:
    """A captured step; its handle goes with it."""

    def __init__(self, enqueue):
        self.handle = C.c_void_p()
        L.call("tlhip_graph_begin_capture", None)
        enqueue()
        L.call("tlhip_graph_end_capture", None, C.byref(self.handle))

    def launch(self):
        L.call("tlhip_graph_launch", self.handle, None)

    def __del__(self):
        if self.handle:
            L.call("tlhip_graph_destroy", self.handle)


class _State:
    """What the program keeps: `keep` holds every buffer, `calls` the prepared calls of a pass."""

    def __init__(self):
        T.getBackend(0)
        self.keep, self.calls, self.out, self.graph = [], [], None, None

    def tensor(self, *shape, dtype):
        t = torch.empty(*shape, dtype=dtype, device="cuda")
        self.keep.append(t)
        return t

    def call(self, name, *args):
        self.keep.append(args)
        self.calls.append((getattr(L.load(), name), args))


def _linear(s, gen, c):
    n, k, m, x = c["n"], c["k"], c["m"], c["x"]
    packed, scales, qw = _weight(gen, c["fmt"], n, k)
    xs = torch.randn(m, k, device="cuda", generator=gen).mul_(0.5).to(TORCH[x])
    y = s.tensor(m, n, dtype=TORCH[x])
    ops = []
    if c["bias"]:
        ops.append(("bias", torch.randn(n, device="cuda", generator=gen).mul_(0.1).to(TORCH[x])))
    if c["act"] != "none":
        ops.append(("unary", c["act"]))
    if c["residual"]:
        ops.append(("add", torch.randn(m, n, device="cuda", generator=gen).to(TORCH[x])))
    ep = _epilogue(*ops)
    s.keep += [packed, scales, qw, xs, ops, ep]
    s.call("tlhip_matmul_quantized", C.byref(qw), xs.data_ptr(), CODE[x], m, y.data_ptr(), CODE[x], 1.0,
           C.byref(ep) if ops else None, None)
    s.out = y


def _decode(s, gen, c):
    m, x, fmt, hid, ffn = c["m"], c["x"], c["fmt"], c["hidden"], c["ffn"]
    dt, code, act = TORCH[x], CODE[x], L.UNARY[c["act"]]
    new = lambda n: s.tensor(m, n, dtype=dt)  # noqa: E731
    h = torch.randn(m, hid, device="cuda", generator=gen).to(dt)
    s.keep.append(h)
    q, kk, v, normed, gate, up, prod = new(c["q"]), new(c["kv"]), new(c["kv"]), new(hid), new(ffn), new(ffn), new(ffn)
    fused = m == 1 and x == "f16" and c["graph"]

    def problems(items):
        probs = (L.GemvProblem * len(items))()
        for p, (w, xi, yi, ep) in zip(probs, items):
            p.w, p.x, p.y = w, xi.data_ptr(), yi.data_ptr()
            if ep is not None:
                p.epilogue = C.pointer(ep)
        s.keep.append(probs)
        return probs

    def matmul(w, xi, yi, *ops):
        ep = _epilogue(*ops)
        s.keep.append(ep)
        s.call("tlhip_matmul_quantized", C.byref(w), xi.data_ptr(), code, m, yi.data_ptr(), code, 1.0,
               C.byref(ep) if ops else None, None)

    for _ in range(c["layers"]):
        w = {}
        for name, n, k in (("q", c["q"], hid), ("k", c["kv"], hid), ("v", c["kv"], hid), ("o", hid, c["q"]),
                           ("gate", ffn, hid), ("up", ffn, hid), ("down", hid, ffn)):
            packed, scales, w[name] = _weight(gen, fmt, n, k)
            s.keep += [packed, scales, w[name]]
        norms = [1.0 + 0.1 * torch.randn(hid, device="cuda", generator=gen) for _ in range(2)]
        s.keep += norms
        mid, out = new(hid), new(hid)
        to_mid, to_out = _epilogue(("add", h)), _epilogue(("add", mid))
        s.keep += [to_mid, to_out]
        qkv = [(w["q"], h if fused else normed, q, None), (w["k"], h if fused else normed, kk, None), (w["v"], h if fused else normed, v, None)]
        pros = [L.Prologue(L.PRO_RMSNORM, 0, EPS, 0, nw.data_ptr()) for nw in norms]
        s.keep += pros
        # attention's input
        if fused:
            s.call("tlhip_gemv_grouped_prologue", problems(qkv), 3, C.byref(pros[0]), code, code, 1.0, None)
        else:
            s.call("tlhip_rmsnorm", h.data_ptr(), code, norms[0].data_ptr(), normed.data_ptr(), code, m, hid, EPS, None)
            if x == "f16" and m <= 16:
                s.call("tlhip_gemv_grouped_rows", problems(qkv), 3, code, m, code, 1.0, None)
            else:
                for wi, xi, yi, _ in qkv:
                    matmul(wi, xi, yi)
        matmul(w["o"], q, mid, ("add", h))
        # the MLP block
        if fused:
            pair = problems([(w["gate"], mid, gate, None), (w["up"], mid, up, None)])
            s.call("tlhip_gemv_grouped_prologue", pair, 2, C.byref(pros[1]), code, code, 1.0, None)
            gated = L.Prologue(L.PRO_GATED_MUL, act, 0.0, 0, up.data_ptr())
            s.keep.append(gated)
            s.call("tlhip_gemv_prologue", C.byref(w["down"]), C.byref(gated), gate.data_ptr(), code, m, out.data_ptr(), code,
                   1.0, C.byref(to_out), None)
        else:
            s.call("tlhip_rmsnorm", mid.data_ptr(), code, norms[1].data_ptr(), normed.data_ptr(), code, m, hid, EPS, None)
            if x == "f16" and m <= 16:
                s.call("tlhip_mlp_decode", C.byref(w["gate"]), C.byref(w["up"]), C.byref(w["down"]), act, normed.data_ptr(),
                       code, m, prod.data_ptr(), out.data_ptr(), code, C.byref(to_out), None)
            else:
                matmul(w["gate"], normed, gate, ("unary", c["act"]))
                matmul(w["up"], normed, prod, ("mul", gate))
                matmul(w["down"], prod, out, ("add", mid))
        h = out
    s.out = (h, kk, v)


def _head(s, gen, c):
    n, k, m, top = c["n"], c["k"], c["m"], c["topk"]
    packed, scales, qw = _weight(gen, c["fmt"], n, k)
    xs = torch.randn(m, k, device="cuda", generator=gen).to(torch.float16)
    logits = s.tensor(m, n, dtype=torch.float32)
    values, indices = s.tensor(m, top, dtype=torch.float32), s.tensor(m, top, dtype=torch.int32)
    s.keep += [packed, scales, qw, xs]
    s.call("tlhip_matmul_quantized", C.byref(qw), xs.data_ptr(), F16, m, logits.data_ptr(), F32, 1.0, None, None)
    for r in range(m):
        s.call("tlhip_topk", logits.data_ptr(), r * n, n, top, values[r].data_ptr(), indices[r].data_ptr(), L.I32, None)
    s.out = (logits, values, indices)


def _load(s, gen, c):
    n, k = c["n"], c["k"]
    code, group = FORMATS[c["fmt"]]
    weight = torch.randn(n, k, device="cuda", generator=gen).mul_(0.02)
    packed, scales = s.tensor(n, k, dtype=torch.int8), s.tensor(n, k // group, dtype=torch.int16)
    back = s.tensor(n, k, dtype=torch.float32)
    qw = L.QWeight(code, group, n, k, packed.data_ptr(), scales.data_ptr())
    s.keep += [weight, qw]
    s.call("tlhip_quantize_int8_grouped_device", weight.data_ptr(), n, k, group, packed.data_ptr(), scales.data_ptr(), None)
    s.call("tlhip_dequant", C.byref(qw), back.data_ptr(), None)
    s.out = (packed, scales, back)


def prepare(case, seed):
    s = _State()
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    {"linear": _linear, "decode": _decode, "head": _head, "load": _load}[case["path"]](s, gen, case)
    torch.cuda.synchronize()  # the library's stream does not wait for torch's
    if case.get("graph"):
        _enqueue(s)  # a stream's first call may allocate, which a capture must not
        L.call("tlhip_stream_synchronize", None)
        s.graph = _Graph(lambda: _enqueue(s))
    return s


def _enqueue(s):
    for fn, args in s.calls:
        rc = fn(*args)
        if rc:
            L.check(rc)


def run(s):
    if s.graph is not None:
        s.graph.launch()
    else:
        _enqueue(s)
    return s.out


# ------------------------------------------------------------------- what it cannot do without

def _weight_bytes(fmt, n, k):
    packed = n * k // 2 if fmt == "int4-32" else n * k
    return packed + (4 * n if fmt == "int8-row" else 2 * n * (k // FORMATS[fmt][1]))


def work(case):
    c = case
    if c["path"] == "load":
        n, k = c["n"], c["k"]
        return {"bytes": 8 * n * k + 2 * _weight_bytes(c["fmt"], n, k), "flops": 0}
    xb = 2 if c["x"] == "f16" else 4
    if c["path"] == "linear":
        n, k, m = c["n"], c["k"], c["m"]
        return {"bytes": _weight_bytes(c["fmt"], n, k) + xb * (m * k + m * n * (2 if c["residual"] else 1) + (n if c["bias"] else 0)),
                "flops": 2 * m * n * k}
    if c["path"] == "head":
        n, k, m = c["n"], c["k"], c["m"]
        return {"bytes": _weight_bytes(c["fmt"], n, k) + 2 * m * k + 4 * m * n + 8 * m * c["topk"], "flops": 2 * m * n * k}
    hid, ffn, q, kv, m = c["hidden"], c["ffn"], c["q"], c["kv"], c["m"]
    shapes = [(q, hid), (kv, hid), (kv, hid), (hid, q), (ffn, hid), (ffn, hid), (hid, ffn)]
    return {"bytes": c["layers"] * (sum(_weight_bytes(c["fmt"], n, k) for n, k in shapes) + 8 * hid) + xb * m * (2 * hid + 2 * kv),
            "flops": c["layers"] * sum(2 * m * n * k for n, k in shapes)}


def tolerance(case):
    """About four times what the path shows with its sums in another order (f32, up to 16
    rows: 32-bit sums of exact products, a few layers deep) or with other roundings of the f16
    values between its steps (28 layers: 2e-3 between two kernel choices)."""
    if case["path"] == "load":
        return "exact"
    if case["path"] == "head":
        return {"rel": 2e-6, "max": 2e-5, "differ": 0.01}
    f32_sums = case["x"] == "f32" and case["m"] <= 16  # more f32 rows are rounded to f16 once
    if case["path"] == "decode":
        return {"rel": 2e-5, "max": 1e-3} if f32_sums else {"rel": 8e-3, "max": 0.1}
    return {"rel": 1e-5, "max": 4e-4} if f32_sums else {"rel": 1e-3, "max": 0.04}
