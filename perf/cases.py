"""The work a program gives this library, for timing: decode (batch 1), tree verify (a few tokens)
and prefill (hundreds to thousands of tokens) on a 2560-wide decoder layer's tensors, through the C ABI.

A case's "kind":
  project  one task group on fp32 rows: qmm_gemm_multi_dispatch, or with "norm" the projection behind
           its RMSNorm (qmm_gemm_multi_dispatch_rmsnorm); "residual" adds one in every task
  ffn      RMSNorm, gate + up (Q4_K), SwiGLU, down (Q6_K) and the residual: qmm_ffn_block_rmsnorm for one
           token, else the engine's calls (qmm_rmsnorm_q8k, the gate + up group, qmm_swiglu_q8k, down)
  lm_head  final RMSNorm, logits of a Q6_K vocabulary and their running argmax (qmm_rmsnorm_q8k,
           qmm_lm_head_argmax)
  decode   one token through the matmuls of several layers as one captured graph: the mixed projection
           group behind its norm, the output projection with its residual, the FFN block

Tensors are synthetic: codes and sub-block scales uniform, super-block scales and mins sized so that the
weights are centred with a deviation of a few hundredths; activations N(0, 1) with one channel in a
hundred ten times larger.
"""
import ctypes
import os
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(_ROOT, "npu880-mtk-npu-llm-runtime_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import qmm_hip  # noqa: E402

TYPES = {"F32": qmm_hip.TYPE_F32, "F16": qmm_hip.TYPE_F16, "Q8_0": qmm_hip.TYPE_Q8_0, "Q4_K": qmm_hip.TYPE_Q4_K,
         "Q5_K": qmm_hip.TYPE_Q5_K, "Q6_K": qmm_hip.TYPE_Q6_K}
VALUES, BYTES = qmm_hip.BLOCK_VALUES, qmm_hip.BLOCK_BYTES
DEV = "cuda"
DECODE_GROUP = "Q5_K:8192,Q4_K:4096,F32:32,F32:32"  # {qkv, gate, alpha, beta} of a layer


def listed():
    return [
        # the smallest call: one key or value projection of one decoded token (launch and latency)
        {"name": "decode_kv", "kind": "project", "tasks": "Q6_K:1024", "M": 1, "K": 2560, "norm": False, "residual": False},
        # one FFN projection of one decoded token
        {"name": "decode_gate", "kind": "project", "tasks": "Q4_K:9728", "M": 1, "K": 2560, "norm": False, "residual": False},
        # a decoded token through eight layers, as a serving loop replays them
        {"name": "decode_layers", "kind": "decode", "layers": 8, "K": 2560, "O": 4096, "N": 9728},
        # the logits of one decoded token
        {"name": "decode_lm_head", "kind": "lm_head", "M": 1, "K": 2560, "V": 151936},
        # the projections of a small draft tree (an odd number of tokens)
        {"name": "verify_qkv", "kind": "project", "tasks": "Q5_K:6144", "M": 7, "K": 2560, "norm": True, "residual": False},
        # the FFN of a larger draft tree
        {"name": "verify_ffn", "kind": "ffn", "M": 37, "K": 2560, "N": 9728},
        # the logits of every position of a draft tree
        {"name": "verify_lm_head", "kind": "lm_head", "M": 16, "K": 2560, "V": 151936},
        # a short prompt through the output projection, with its residual
        {"name": "prefill_o", "kind": "project", "tasks": "Q4_K:2560", "M": 192, "K": 4096, "norm": False, "residual": True},
        # a ragged prompt through an 8-bit projection
        {"name": "prefill_q8_0", "kind": "project", "tasks": "Q8_0:2560", "M": 333, "K": 2560, "norm": False, "residual": False},
        # the projections and the FFN of a 512-token prompt
        {"name": "prefill_qkv", "kind": "project", "tasks": "Q5_K:6144", "M": 512, "K": 2560, "norm": True, "residual": False},
        {"name": "prefill_ffn", "kind": "ffn", "M": 512, "K": 2560, "N": 9728},
        # the FFN of a long prompt
        {"name": "prompt_ffn", "kind": "ffn", "M": 2048, "K": 2560, "N": 9728},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    kind = rng.choice(["project", "project", "project", "ffn", "lm_head"])
    if kind == "lm_head":
        return {"kind": kind, "M": _log_int(rng, 1, 16), "K": 256 * rng.randint(4, 16), "V": _log_int(rng, 8000, 151936)}
    M = _log_int(rng, 1, 2048)
    if kind == "ffn":
        return {"kind": kind, "M": M, "K": 256 * rng.randint(4, 12), "N": 256 * rng.randint(8, 38)}
    t = rng.choice(["Q4_K", "Q5_K", "Q6_K", "Q8_0"])
    norm = rng.random() < 0.4
    K = 32 * _log_int(rng, 16, 304) if t == "Q8_0" and not norm else 256 * _log_int(rng, 2, 38)
    N = _log_int(rng, 256, 16384)
    tasks = "%s:%d" % (t, N) if rng.random() < 0.6 else "%s:%d,%s:%d" % (t, N, t, _log_int(rng, 256, 4096))
    return {"kind": kind, "tasks": tasks, "M": M, "K": K, "norm": norm, "residual": rng.random() < 0.4}


def _tasks(case):
    return [(TYPES[t.split(":")[0]], int(t.split(":")[1])) for t in case["tasks"].split(",")]


# ------------------------------------------------------------------ inputs
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 7919 + 17)
    return g


def _f16(n, lo, hi, g):
    v = torch.empty(n, device=DEV).uniform_(lo, hi, generator=g).to(torch.float16)
    return v, v.view(torch.uint8).reshape(n, 2)


def _weights(t, rows, cols, g):
    """rows x cols of packed blocks: uint8 [rows, row bytes]."""
    if t in (qmm_hip.TYPE_F32, qmm_hip.TYPE_F16):
        v = 0.05 * torch.randn(rows, cols, device=DEV, generator=g)
        return (v if t == qmm_hip.TYPE_F32 else v.half()).view(torch.uint8)
    n = rows * (cols // VALUES[t])
    out = torch.randint(0, 256, (n, BYTES[t]), dtype=torch.uint8, device=DEV, generator=g)
    if t in (qmm_hip.TYPE_Q4_K, qmm_hip.TYPE_Q5_K):
        half = 7.5 if t == qmm_hip.TYPE_Q4_K else 15.5  # the middle code: mins centre the weights
        d, b = _f16(n, 1.2 / half * 1e-3, 2.4 / half * 1e-3, g)
        out[:, 0:2] = b
        out[:, 2:4] = (d.float() * half).half().view(torch.uint8).reshape(n, 2)
    elif t == qmm_hip.TYPE_Q6_K:
        out[:, 192:208] = torch.randint(-64, 64, (n, 16), dtype=torch.int8, device=DEV, generator=g).view(torch.uint8)
        out[:, 208:210] = _f16(n, 2e-5, 1e-4, g)[1]
    else:
        out[:, 0:2] = _f16(n, 2e-4, 8e-4, g)[1]
    return out.reshape(rows, -1)


def _acts(M, K, g):
    x = torch.randn(M, K, device=DEV, generator=g)
    return x * torch.where(torch.rand(K, device=DEV, generator=g) < 0.01, 10.0, 1.0)


def _gamma(K, g):
    return torch.empty(K, device=DEV).uniform_(0.5, 1.5, generator=g)


def _inputs(case, seed):
    """The case's tensors, from the seed alone."""
    g, kind = _gen(seed), case["kind"]
    if kind == "decode":
        K, O, N = case["K"], case["O"], case["N"]
        group = _tasks({"tasks": DECODE_GROUP})
        s = {"x": _acts(1, K, g), "layers": []}
        for _ in range(case["layers"]):
            s["layers"].append({
                "g1": _gamma(K, g), "proj": [_weights(t, n, K, g) for t, n in group], "attn": _acts(1, O, g),
                "o": _weights(qmm_hip.TYPE_Q4_K, K, O, g), "g2": _gamma(K, g),
                "gate": _weights(qmm_hip.TYPE_Q4_K, N, K, g), "up": _weights(qmm_hip.TYPE_Q4_K, N, K, g),
                "down": _weights(qmm_hip.TYPE_Q6_K, K, N, g)})
        return s
    s = {"x": _acts(case["M"], case["K"], g), "gamma": _gamma(case["K"], g)}
    if kind == "ffn":
        s["gate"] = _weights(qmm_hip.TYPE_Q4_K, case["N"], case["K"], g)
        s["up"] = _weights(qmm_hip.TYPE_Q4_K, case["N"], case["K"], g)
        s["down"] = _weights(qmm_hip.TYPE_Q6_K, case["K"], case["N"], g)
    elif kind == "lm_head":
        s["w"] = _weights(qmm_hip.TYPE_Q6_K, case["V"], case["K"], g)
    else:
        s["w"] = [_weights(t, n, case["K"], g) for t, n in _tasks(case)]
        if case["residual"]:
            s["res"] = [torch.randn(case["M"], n, device=DEV, generator=g) for _, n in _tasks(case)]
    return s


# ------------------------------------------------------------------ program
_ctx = None


def _context():
    """The program's one context (it lives as long as the process)."""
    global _ctx
    if _ctx is None:
        _ctx = qmm_hip.Context(0)
    return _ctx


def _p(t):
    return ctypes.c_void_p(t.data_ptr() if t is not None else 0)


def _check(rc):
    if rc:
        raise RuntimeError("qmm status %d: %s" % (rc, _context().last_error()))


def _array(M, K, tasks):
    """[(type, weights, outputs, residual)] as the dispatcher's task array."""
    return qmm_hip.Context._tasks(M, K, [
        qmm_hip.MatrixTask(w.data_ptr(), t, y.shape[1], K, y.data_ptr(), residual=r.data_ptr() if r is not None else None)
        for t, w, y, r in tasks])


def _new(*shape):
    return torch.zeros(*shape, device=DEV)


class _Graph:
    def __init__(self, ctx, record):
        self.ctx = ctx
        ctx.graph_begin()
        record()
        self.exe = ctx.graph_end()

    def __del__(self):
        self.ctx.graph_destroy(self.exe)


def prepare(case, seed):
    ctx = _context()
    lib, h, kind, K = ctx.lib, ctx._h, case["kind"], case["K"]
    s = {"case": case, **_inputs(case, seed)}
    calls = s["calls"] = []  # (entry point, its arguments): what a C program's call sites hold

    def call(name, *args):
        calls.append((getattr(lib, name), (h,) + args))

    if kind == "decode":
        O, N, group, x = case["O"], case["N"], _tasks({"tasks": DECODE_GROUP}), s["x"]
        ctx.reserve(1, max(K, O, N))
        s["out"] = []
        for L in s["layers"]:
            proj = [_new(1, n) for _, n in group]
            x1, x2, gate, up = _new(1, K), _new(1, K), _new(1, N), _new(1, N)
            call("qmm_gemm_multi_dispatch_rmsnorm", _p(x), _p(L["g1"]), 1, K,
                 _array(1, K, [(t, w, y, None) for (t, _), w, y in zip(group, L["proj"], proj)]), len(group))
            call("qmm_gemm_multi_dispatch", _p(L["attn"]), 1, O, _array(1, O, [(qmm_hip.TYPE_Q4_K, L["o"], x1, x)]), 1)
            t = [_array(1, K, [(qmm_hip.TYPE_Q4_K, L["gate"], gate, None)]),
                 _array(1, K, [(qmm_hip.TYPE_Q4_K, L["up"], up, None)]),
                 _array(1, N, [(qmm_hip.TYPE_Q6_K, L["down"], x2, x1)])]
            call("qmm_ffn_block_rmsnorm", _p(x1), _p(L["g2"]), K, *[ctypes.byref(a[0]) for a in t], _p(None))
            s["out"].append(proj[:2] + [x1, gate, up, x2])
            s.setdefault("keep", []).append((proj, t))
            x = x2
        torch.cuda.synchronize()  # the inputs were made on another stream than the library's

        def record():
            for f, args in calls:
                _check(f(*args))

        record()  # once before the capture: the context's buffers get their size
        s["graph"] = _Graph(ctx, record)
        return s

    M = case["M"]
    ctx.reserve(M, max(K, case.get("N", K)))
    if kind == "project":
        outs = s["out"] = [_new(M, n) for _, n in _tasks(case)]
        res = s.get("res") or [None] * len(outs)
        arr = _array(M, K, [(t, w, y, r) for (t, _), w, y, r in zip(_tasks(case), s["w"], outs, res)])
        if case["norm"]:
            call("qmm_gemm_multi_dispatch_rmsnorm", _p(s["x"]), _p(s["gamma"]), M, K, arr, len(outs))
        else:
            call("qmm_gemm_multi_dispatch", _p(s["x"]), M, K, arr, len(outs))
    elif kind == "ffn":
        N = case["N"]
        gate, up, hid, y = _new(M, N), _new(M, N), _new(M, N), _new(M, K)
        s["out"] = [gate, up, hid, y]
        gu = [(qmm_hip.TYPE_Q4_K, s["gate"], gate, None), (qmm_hip.TYPE_Q4_K, s["up"], up, None)]
        dn = [(qmm_hip.TYPE_Q6_K, s["down"], y, s["x"])]
        if M == 1:
            t = [_array(1, K, gu[:1]), _array(1, K, gu[1:]), _array(1, N, dn)]
            s["keep"] = t
            call("qmm_ffn_block_rmsnorm", _p(s["x"]), _p(s["gamma"]), K, *[ctypes.byref(a[0]) for a in t], _p(hid))
        else:
            q1 = torch.zeros(qmm_hip.q8k_bytes(M, K), dtype=torch.uint8, device=DEV)
            q2 = torch.zeros(qmm_hip.q8k_bytes(M, N), dtype=torch.uint8, device=DEV)
            s["q"] = (q1, q2)
            call("qmm_rmsnorm_q8k", _p(s["x"]), _p(s["gamma"]), M, K, _p(None), _p(q1))
            call("qmm_gemm_multi_dispatch_prequantized", _p(q1), _p(None), M, K, _array(M, K, gu), 2)
            call("qmm_swiglu_q8k", _p(gate), _p(up), M, N, _p(hid), _p(q2))
            call("qmm_gemm_multi_dispatch_prequantized", _p(q2), _p(None), M, N, _array(M, N, dn), 1)
    else:
        V = case["V"]
        q = s["q"] = torch.zeros(qmm_hip.q8k_bytes(M, K), dtype=torch.uint8, device=DEV)
        logits, best = _new(M, V), torch.zeros(2 * M, dtype=torch.int32, device=DEV)
        seeds = s["seeds"] = torch.zeros(2 * M, dtype=torch.int32, device=DEV)
        seeds.view(torch.float32)[:M] = -1e30
        s["out"] = [logits, best.view(torch.float32)[:M], best[M:]]
        call("qmm_memcpy_d2d", _p(best), _p(seeds), 8 * M)
        call("qmm_rmsnorm_q8k", _p(s["x"]), _p(s["gamma"]), M, K, _p(None), _p(q))
        call("qmm_lm_head_argmax", _p(q), _p(None), M, K, _p(s["w"]), qmm_hip.TYPE_Q6_K, V, 0, _p(logits), _p(best),
             _p(best[M:]))
    torch.cuda.synchronize()  # the inputs were made on another stream than the library's
    return s


def run(state):
    if "graph" in state:
        _context().graph_launch(state["graph"].exe)
    else:
        for f, args in state["calls"]:
            rc = f(*args)
            if rc:
                _check(rc)
    return state["out"]


# -------------------------------------------------------------------- costs
def _mm(M, K, types):
    """(bytes, flops) of one task group: weights, fp32 rows in, fp32 rows out."""
    n = sum(r for _, r in types)
    return sum(r * qmm_hip.row_bytes(t, K) for t, r in types) + 4 * M * (K + n), 2 * M * K * n


def work(case):
    kind, K = case["kind"], case["K"]
    q4, q6 = qmm_hip.TYPE_Q4_K, qmm_hip.TYPE_Q6_K
    if kind == "project":
        parts = [_mm(case["M"], K, _tasks(case))]
        more = 4 * case["M"] * sum(n for _, n in _tasks(case)) if case["residual"] else 0
        more += 4 * K if case["norm"] else 0
    elif kind == "ffn":  # gate, up and the hidden rows are outputs of their own
        M, N = case["M"], case["N"]
        parts = [_mm(M, K, [(q4, N), (q4, N)]), (K * qmm_hip.row_bytes(q6, N) + 4 * M * K, 2 * M * K * N)]
        more = 4 * M * N + 4 * K
    elif kind == "lm_head":
        parts, more = [_mm(case["M"], K, [(q6, case["V"])])], 4 * K
    else:
        O, N = case["O"], case["N"]
        layer = [_mm(1, K, _tasks({"tasks": DECODE_GROUP})), _mm(1, O, [(q4, K)]), _mm(1, K, [(q4, N), (q4, N)]),
                 (K * qmm_hip.row_bytes(q6, N) + 4 * K, 2 * K * N)]
        parts, more = layer * case["layers"], 8 * K * case["layers"]
    return {"bytes": sum(b for b, _ in parts) + more, "flops": sum(f for _, f in parts)}


def tolerance(case):
    """The sums are fp32: 0.6e-7 to 1.7e-7 from the exact ones. Where fp32 arithmetic comes before a
    quantizer, a last bit moved there moves a code by one here and there (a step is 1/127 of its
    block's largest value): up to 8e-5 behind a norm, 4e-4 behind a norm and SwiGLU."""
    if case["kind"] in ("ffn", "decode"):
        return {"rel": 2e-3, "max": 2e-2}
    if case["kind"] == "project" and not case["norm"]:
        return {"rel": 1e-6, "max": 1e-5}
    return {"rel": 4e-4, "max": 1e-2, "differ": 0.01}


# -------------------------------------------------------------------- exact
def _dequant(t, w, cols):
    """Packed rows -> float64 [rows, cols]."""
    rows = w.shape[0]
    if t in (qmm_hip.TYPE_F32, qmm_hip.TYPE_F16):
        return w.contiguous().view(torch.float32 if t == qmm_hip.TYPE_F32 else torch.float16).double()
    b = w.reshape(-1, BYTES[t])
    n = b.shape[0]
    half = lambda i: b[:, i:i + 2].contiguous().view(torch.float16).double()  # noqa: E731
    i16 = lambda v: v.to(torch.int16)  # noqa: E731
    if t == qmm_hip.TYPE_Q8_0:
        return (half(0) * b[:, 2:].contiguous().view(torch.int8).double()).reshape(rows, cols)
    if t == qmm_hip.TYPE_Q6_K:
        ql, qh = i16(b[:, 0:128]).reshape(n, 2, 2, 32), i16(b[:, 128:192]).reshape(n, 2, 32)
        q = torch.stack([(ql[:, :, 0] & 15) | ((qh & 3) << 4), (ql[:, :, 1] & 15) | ((qh >> 2 & 3) << 4),
                         (ql[:, :, 0] >> 4) | ((qh >> 4 & 3) << 4), (ql[:, :, 1] >> 4) | ((qh >> 6 & 3) << 4)], 2)
        sc = b[:, 192:208].contiguous().view(torch.int8).double().reshape(n, 16, 1)
        return (half(208).reshape(n, 1, 1) * sc * (q.reshape(n, 16, 16).double() - 32)).reshape(rows, cols)
    s = i16(b[:, 4:16])
    sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1).double()
    m = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
    qs = i16(b[:, -128:]).reshape(n, 4, 1, 32)
    q = torch.cat([qs & 15, qs >> 4], 2).reshape(n, 8, 32)
    if t == qmm_hip.TYPE_Q5_K:
        bit = torch.arange(8, device=b.device, dtype=torch.int16).reshape(1, 8, 1)
        q = q + ((i16(b[:, 16:48]).reshape(n, 1, 32) >> bit & 1) << 4)
    return ((half(0) * sc).unsqueeze(2) * q.double() - (half(2) * m).unsqueeze(2)).reshape(rows, cols)


def _codes(x, block):
    """What the quantizers make of rows x: codes times scale, in 64 bits (the codes are defined in
    32: fp16 values, one division per block, round to nearest even)."""
    v = x.half().float().reshape(x.shape[0], -1, block)
    top = v.abs().amax(2, keepdim=True)
    full = torch.full_like(top, 127.0)  # (a tensor: torch divides by a number through its reciprocal)
    q = torch.where(top > 0, (v * (full / top)).round().clamp(-127, 127), torch.zeros_like(v))
    return (q.double() * (top / full).double()).reshape(x.shape)


def _dot(t, w, x):
    xq = x.half().double() if t in (qmm_hip.TYPE_F32, qmm_hip.TYPE_F16) else _codes(x, VALUES[t])
    return torch.cat([xq @ _dequant(t, w[r:r + 8192], x.shape[1]).t() for r in range(0, w.shape[0], 8192)], 1)


def _norm(x, gamma):
    v, g = x.half().double(), gamma.half().double()
    return (v / torch.sqrt((v * v).mean(1, keepdim=True) + 1e-6) * g).half().double()


def _ffn(x, gamma, gate, up, down):
    """(gate, up, hidden, out with the residual x)"""
    y = _norm(x, gamma)
    a, b = _dot(qmm_hip.TYPE_Q4_K, gate, y), _dot(qmm_hip.TYPE_Q4_K, up, y)
    g = a.half().double()
    hid = g / (1 + torch.exp(-g)) * b.half().double()
    return [a, b, hid, _dot(qmm_hip.TYPE_Q6_K, down, hid) + x]


def exact(case, seed):
    s, kind = _inputs(case, seed), case["kind"]
    x = s["x"].double()
    if kind == "project":
        y = _norm(x, s["gamma"]) if case["norm"] else x
        res = s.get("res") or [0] * len(s["w"])
        return [_dot(t, w, y) + r for (t, _), w, r in zip(_tasks(case), s["w"], res)]
    if kind == "ffn":
        return _ffn(x, s["gamma"], s["gate"], s["up"], s["down"])
    if kind == "lm_head":
        return [_dot(qmm_hip.TYPE_Q6_K, s["w"], _norm(x, s["gamma"])), None, None]
    out = []
    for L in s["layers"]:
        y = _norm(x, L["g1"])
        proj = [_dot(t, w, y) for (t, _), w in zip(_tasks({"tasks": DECODE_GROUP})[:2], L["proj"])]
        x1 = _dot(qmm_hip.TYPE_Q4_K, L["o"], L["attn"].double()) + x
        a, b, _, x = _ffn(x1, L["g2"], L["gate"], L["up"], L["down"])
        out.append(proj + [x1, a, b, x])
    return out
