"""Performance cases: the calls a program that serves a Q4_K / Q6_K model makes on one MI355X.

Every case goes through ``kq.gpu4.Engine`` as a serving program does: one-token decode, speculative
verify of a few drafted tokens, prompt prefill and the output head, on the matrices of the 9B-class
layer that the benchmark uses (q/o 4096x4096, k/v 1024x4096, gate/up 12288x4096, down 4096x12288;
Q4_K, with the Q6_K v and down that a Q4_K_M file holds in half of its layers) and on generic sizes
around it.  Decode and verify run as a captured graph, the way the benchmark (and any program whose
steps take tens of microseconds) runs them; everything else is called directly.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oxcoder-9b_amd"))

from kq import gpu4  # noqa: E402
from kq.formats import BLOCK, Q4_K, Q6_K, QK  # noqa: E402

DEV = "cuda"
VOCAB = 4096          # rows of the embedding table of the decode cases

# ---------------------------------------------------------------------------------------- cases

# The 9B-class layer of the benchmark.
DIM, KV, FFN = 4096, 1024, 12288


def listed():
    return [
        # One projection at batch 1, called directly: what a program that runs its own loop pays per
        # call, launch and host work included.
        {"name": "gemv_attn_output", "kind": "gemv", "mode": "q8k", "rows": DIM, "cols": DIM, "q6": False},
        # The token loop: embedding row, then 4 layers with the fused RMSNorm and SwiGLU producers.
        {"name": "decode_layers", "kind": "decode", "mode": "q8k", "layers": 4, "dim": DIM, "kv": KV, "ffn": FFN},
        # The same in the reference's own numerics (fp32 activations).
        {"name": "decode_layers_f32", "kind": "decode", "mode": "f32", "layers": 4, "dim": DIM, "kv": KV, "ffn": FFN},
        # Speculative verify: a short draft, and the largest batch the batched GEMV takes.
        {"name": "verify_4", "kind": "rows", "mode": "q8k", "graph": True, "layers": 4, "tokens": 4, "chunk": 256,
         "dim": DIM, "kv": KV, "ffn": FFN},
        {"name": "verify_16", "kind": "rows", "mode": "q8k", "graph": True, "layers": 4, "tokens": 16, "chunk": 256,
         "dim": DIM, "kv": KV, "ffn": FFN},
        # A short prompt in the reference's numerics.
        {"name": "prompt_f32_24", "kind": "rows", "mode": "f32", "graph": False, "layers": 1, "tokens": 24,
         "chunk": 256, "dim": DIM, "kv": KV, "ffn": FFN},
        # A chat turn's short prompt: fewer tokens than a chunk.
        {"name": "prefill_40", "kind": "rows", "mode": "q8k", "graph": False, "layers": 1, "tokens": 40,
         "chunk": 256, "dim": DIM, "kv": KV, "ffn": FFN},
        # One chunk of the default chunked prefill.
        {"name": "prefill_256", "kind": "rows", "mode": "q8k", "graph": False, "layers": 1, "tokens": 256,
         "chunk": 256, "dim": DIM, "kv": KV, "ffn": FFN},
        # A prompt that fills no whole number of chunks (three, then 9 tokens).
        {"name": "prefill_777", "kind": "rows", "mode": "q8k", "graph": False, "layers": 1, "tokens": 777,
         "chunk": 256, "dim": DIM, "kv": KV, "ffn": FFN},
        # A long prompt with a large chunk: the prefill that is bound by arithmetic.
        {"name": "prefill_2048", "kind": "rows", "mode": "q8k", "graph": False, "layers": 1, "tokens": 2048,
         "chunk": 2048, "dim": DIM, "kv": KV, "ffn": FFN},
        # The output head with the greedy pick, both head types and vocabulary sizes of the benchmark.
        {"name": "head_q6k", "kind": "head", "mode": "q8k", "rows": 151936, "cols": DIM, "q6": True},
        {"name": "head_q4k", "kind": "head", "mode": "q8k", "rows": 248320, "cols": DIM, "q6": False},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: any kind, with hidden sizes from 1024 to 5120 and token counts from 1 to 2048."""
    kind = rng.choice(["gemv", "decode", "verify", "f32", "prefill", "prefill", "prefill", "head"])
    if kind in ("gemv", "head"):
        lo, hi = (64, 2048) if kind == "gemv" else (4000, 31000)
        return {"kind": kind, "mode": "q8k" if kind == "head" else rng.choice(["q8k", "f32"]),
                "rows": 8 * _log_int(rng, lo, hi), "cols": QK * rng.randint(4, 16 if kind == "head" else 48),
                "q6": rng.random() < 0.5}
    dim = QK * rng.randint(4, 20)
    case = {"kind": "decode" if kind == "decode" else "rows", "mode": "q8k", "dim": dim,
            "kv": 8 * _log_int(rng, 16, 256), "ffn": QK * rng.randint(dim // 128, min(56, 3 * dim // 256 + 4))}
    if kind == "decode":
        case.update(mode=rng.choice(["q8k", "q8k", "f32"]), layers=rng.randint(2, 4))
        return case
    if kind == "verify":
        case.update(graph=True, layers=rng.randint(2, 4), tokens=rng.randint(2, 16), chunk=256)
    elif kind == "f32":
        case.update(mode="f32", graph=False, layers=1, tokens=_log_int(rng, 2, 24), chunk=256)
    else:
        chunk = rng.choice([256, 256, 512, 2048])
        case.update(graph=False, layers=1, tokens=_log_int(rng, 17, chunk if chunk > 256 else 1024), chunk=chunk)
    most = max(work(c)["flops"] for c in listed())
    while work(case)["flops"] > most:
        case["tokens"] = case["tokens"] * 3 // 4
    return case


# -------------------------------------------------------------------------------------- weights

def _quantize_q4k(w):
    """fp32 [R][C] -> Q4_K blocks uint8 [R][C/256][144]: per 32 values a 6-bit scale and minimum."""
    R, C = w.shape
    x = w.view(R, C // QK, 8, 32)
    mn = x.amin(-1).clamp(max=0)
    scale, low = (x.amax(-1) - mn) / 15, -mn
    d = (scale.amax(-1, keepdim=True) / 63).half().float()
    dm = (low.amax(-1, keepdim=True) / 63).half().float()
    ls = (scale / d).round().clamp(1, 63)
    lm = (low / dm.clamp(min=1e-8)).round().clamp(0, 63)
    q = ((x + (dm * lm)[..., None]) / (d * ls)[..., None]).round().clamp(0, 15).to(torch.uint8)
    ls, lm = ls.to(torch.uint8), lm.to(torch.uint8)
    sc = torch.cat([ls[..., :4] | (ls[..., 4:] >> 4) << 6, lm[..., :4] | (lm[..., 4:] >> 4) << 6,
                    (ls[..., 4:] & 15) | (lm[..., 4:] & 15) << 4], -1)
    qs = (q[..., 0::2, :] | q[..., 1::2, :] << 4).reshape(R, C // QK, 128)
    dd = torch.cat([d, dm], -1).half().view(torch.uint8)
    return torch.cat([dd, sc, qs], -1)


def _quantize_q6k(w):
    """fp32 [R][C] -> Q6_K blocks uint8 [R][C/256][210]: per 16 values an 8-bit scale."""
    R, C = w.shape
    x = w.view(R, C // QK, 16, 16)
    scale = x.abs().amax(-1) / 31
    d = (scale.amax(-1, keepdim=True) / 127).half().float()
    ls = (scale / d).round().clamp(1, 127)
    q = ((x / (d * ls)[..., None]).round().clamp(-32, 31) + 32).to(torch.uint8).view(R, C // QK, 2, 4, 32)
    lo, hi = q & 15, q >> 4
    ql = torch.cat([lo[..., 0, :] | lo[..., 2, :] << 4, lo[..., 1, :] | lo[..., 3, :] << 4], -1)
    qh = hi[..., 0, :] | hi[..., 1, :] << 2 | hi[..., 2, :] << 4 | hi[..., 3, :] << 6
    return torch.cat([ql.flatten(-2), qh.flatten(-2), ls.to(torch.uint8), d.half().view(torch.uint8)], -1)


def _decode(packed, R, C, ty):
    """Layout bytes [R/8][C/256][8][block] -> the weights in 64 bits."""
    b = packed.view(R // 8, C // QK, 8, BLOCK[ty]).transpose(1, 2).reshape(R, C // QK, BLOCK[ty])
    if ty == Q4_K:
        d = b[..., :4].contiguous().view(torch.float16).double()
        s = b[..., 4:16]
        sc = torch.cat([s[..., :4] & 63, s[..., 8:] & 15 | s[..., :4] >> 6 << 4], -1).double()
        mi = torch.cat([s[..., 4:8] & 63, s[..., 8:] >> 4 | s[..., 4:8] >> 6 << 4], -1).double()
        qs = b[..., 16:].reshape(R, C // QK, 4, 32)
        q = torch.stack([qs & 15, qs >> 4], -2).reshape(R, C // QK, 8, 32).double()
        w = (d[..., :1] * sc)[..., None] * q - (d[..., 1:] * mi)[..., None]
    else:
        ql, qh = b[..., :128].reshape(R, C // QK, 2, 2, 32), b[..., 128:192].reshape(R, C // QK, 2, 32)
        q = torch.stack([ql[..., 0, :] & 15 | (qh & 3) << 4, ql[..., 1, :] & 15 | (qh >> 2 & 3) << 4,
                         ql[..., 0, :] >> 4 | (qh >> 4 & 3) << 4, ql[..., 1, :] >> 4 | qh >> 6 << 4], -2)
        q = q.reshape(R, C // QK, 16, 16).double() - 32
        sc = b[..., 192:208].contiguous().view(torch.int8).double()
        w = (b[..., 208:].contiguous().view(torch.float16).double() * sc)[..., None] * q
    return w.reshape(R, C)


def _matrix(gen, R, C, ty):
    """N(0, 0.02) weights, quantized and in the engine's 8-row layout, a few thousand rows at a time."""
    parts = []
    for r0 in range(0, R, 16384):
        n = min(16384, R - r0)
        w = torch.randn(n, C, generator=gen, device=DEV) * 0.02
        b = _quantize_q4k(w) if ty == Q4_K else _quantize_q6k(w)
        parts.append(b.view(n // 8, 8, C // QK, BLOCK[ty]).transpose(1, 2).reshape(-1))
    return torch.cat(parts)


def _layer(case, i):
    """(name, input group, rows, columns, type) of layer i's matrices, as a Q4_K_M file types them."""
    D, KVR, F = case["dim"], case["kv"], case["ffn"]
    big = Q6_K if i % 2 == 0 else Q4_K
    return [("%d.q" % i, "qkv", D, D, Q4_K), ("%d.k" % i, "qkv", KVR, D, Q4_K), ("%d.v" % i, "qkv", KVR, D, big),
            ("%d.o" % i, "o", D, D, Q4_K), ("%d.gate" % i, "ffn", F, D, Q4_K), ("%d.up" % i, "ffn", F, D, Q4_K),
            ("%d.down" % i, "down", D, F, big)]


def _groups(case, i):
    """[(group, column count, names)] of layer i, in the order a layer runs them."""
    out = {}
    for name, group, _, C, _ in _layer(case, i):
        out.setdefault(group, (C, []))[1].append(name)
    return [(g, C, names) for g, (C, names) in out.items()]


def _matrices(case):
    if case["kind"] in ("gemv", "head"):
        return [("w", "w", case["rows"], case["cols"], Q6_K if case["q6"] else Q4_K)]
    return [m for i in range(case["layers"]) for m in _layer(case, i)]


# ------------------------------------------------------------------------------------ one state

def _capture(call):
    """The call as a graph, captured as the benchmark captures its steps."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call()
    return graph


def _decode_step(s):
    """One token: the embedding row, then every layer (attention itself is not part of the framework:
    o takes q's output, which has its width)."""
    e, case, y = s["engine"], s["case"], s["out"]
    q8k = case["mode"] == "q8k"
    e.embed(s["token"], out=s["h"], name="embd")
    residual = None
    for i in range(case["layers"]):
        qkv, gate = ["%d.%s" % (i, n) for n in "qkv"], ["%d.gate" % i, "%d.up" % i]
        o, down = "%d.o" % i, "%d.down" % i
        _, xq = e.rmsfold_q8k(s["h"], s["norm"], residual=residual, xn=None if q8k else s["xn"])
        e.gemv_q8(qkv, xq, [y[n] for n in qkv]) if q8k else e.gemv(qkv, s["xn"], [y[n] for n in qkv])
        e.gemv([o], y[qkv[0]], [y[o]])
        _, xq = e.rmsfold_q8k(s["h"], s["norm"], residual=y[o], xn=None if q8k else s["xn"])
        e.gemv_q8(gate, xq, [y[n] for n in gate]) if q8k else e.gemv(gate, s["xn"], [y[n] for n in gate])
        _, xq = e.swiglu_q8k(y[gate[0]], y[gate[1]], y=None if q8k else s["act"])
        e.gemv_q8([down], xq, [y[down]]) if q8k else e.gemv([down], s["act"], [y[down]])
        residual = y[down]


def _rows_step(s):
    """Several rows through every layer's matrices, each input group in one call."""
    for i in range(s["case"]["layers"]):
        for group, _, names in _groups(s["case"], i):
            s["engine"].feed_rows(names, s["x"][group], [s["out"][n] for n in names])


def _activations(gen, n, c):
    """Normalised hidden states: unit variance with a few channels several times larger, as they have."""
    x = torch.randn(n, c, generator=gen, device=DEV)
    return x * (1 + 7 * (torch.rand(c, generator=gen, device=DEV) < 0.005))


def _inputs(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    kind = case["kind"]
    weights = {name: (_matrix(gen, R, C, ty), R, C, ty) for name, _, R, C, ty in _matrices(case)}
    s = {"case": case, "weights": weights}
    if kind in ("gemv", "head"):
        s["x"] = _activations(gen, 1, case["cols"])[0]
    elif kind == "decode":
        weights["embd"] = (_matrix(gen, VOCAB, case["dim"], Q4_K), VOCAB, case["dim"], Q4_K)
        s["token"] = int(torch.randint(VOCAB, (1,), generator=gen, device=DEV))
        s["norm"] = 1 + 0.1 * torch.randn(case["dim"], generator=gen, device=DEV)
    else:
        s["x"] = {g: _activations(gen, case["tokens"], C) for g, C, _ in _groups(case, 0)}
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    w = gpu4.Weights(DEV)
    for name, (buf, R, C, ty) in s.pop("weights").items():
        w.add(name, buf, R, C, ty)
    n = case.get("tokens", 1)
    s["out"] = {name: torch.empty((n, R) if case["kind"] == "rows" else R, device=DEV)
                for name, _, R, _, _ in _matrices(case)}
    groups = [names for i in range(case.get("layers", 0)) for _, _, names in _groups(case, i)]
    s["engine"] = gpu4.Engine(w, mode=case["mode"], chunk=case.get("chunk", 0), groups=groups)
    if case["kind"] == "decode":
        s["h"] = torch.empty(case["dim"], device=DEV)
        s["xn"], s["act"] = torch.empty(case["dim"], device=DEV), torch.empty(case["ffn"], device=DEV)
        s["graph"] = _capture(lambda: _decode_step(s))
    elif case.get("graph"):
        s["graph"] = _capture(lambda: _rows_step(s))
    return s


def run(state):
    kind = state["case"]["kind"]
    if kind == "gemv":
        state["engine"].gemv(["w"], state["x"], [state["out"]["w"]])
    elif kind == "head":
        token = state["engine"].head("w", state["x"], state["out"]["w"])
        return {"logits": state["out"]["w"], "token": token}
    elif "graph" in state:
        state["graph"].replay()
    else:
        _rows_step(state)
    return dict(state["out"], h=state["h"]) if kind == "decode" else state["out"]


# ----------------------------------------------------------------------------- work and accuracy

def work(case):
    """Weights, inputs and outputs once each; a multiply and an add per weight and token."""
    n = case.get("tokens", 1)
    mats = _matrices(case)
    cols = {(name.split(".")[0], group): C for name, group, _, C, _ in mats}
    nbytes = sum(R * (C // QK) * BLOCK[ty] + 4 * n * R for _, _, R, C, ty in mats) + 4 * n * sum(cols.values())
    return {"bytes": nbytes, "flops": 2 * n * sum(R * C for _, _, R, C, _ in mats)}


def tolerance(case):
    """fp32 sums in another order over the same (quantized) inputs, about four times what the paths
    measure against 64 bits.  A decode step's layers build on one another: an activation whose last bit
    moved can round to the next 8-bit code."""
    if case["kind"] == "decode":
        return {"rel": 2e-3 if case["mode"] == "q8k" else 1e-5}
    return {"rel": 2e-6, "max": 2e-5, "differ": 0.0}


def _q8k(x):
    """x as the Q8_K activation holds it: 256 values share d = 1 / iscale, iscale = -127 / (the value of
    largest magnitude); codes rounded to nearest even in 32 bits."""
    b = x.float().reshape(-1, QK)
    top = b.gather(1, b.abs().argmax(1, keepdim=True))
    inv = torch.div(torch.full_like(top, -127.0), top)
    q = torch.where(top == 0, torch.zeros_like(b), (b * inv).round().clamp(max=127))
    d = torch.where(top == 0, torch.zeros_like(top), torch.div(torch.ones_like(top), inv))
    return (q.double() * d.double()).view(x.shape)


def exact(case, seed):
    s = _inputs(case, seed)
    seen = _q8k if case["mode"] == "q8k" else (lambda x: x.float().double())

    def product(name, x):
        buf, R, C, ty = s["weights"][name]
        rows = [seen(x) @ _decode(buf.view(R // 8, -1)[r:r + 2048].reshape(-1), min(16384, R - 8 * r), C, ty).T
                for r in range(0, R // 8, 2048)]
        return torch.cat(rows, -1)

    if case["kind"] == "gemv":
        return {"w": product("w", s["x"])}
    if case["kind"] == "head":
        logits = product("w", s["x"])
        return {"logits": logits, "token": int(logits.argmax())}
    if case["kind"] == "rows":
        return {n: product(n, s["x"][g]) for n, g, _, _, _ in _matrices(case)}

    def rms(h):
        return h / (h.square().mean() + 1e-6).sqrt() * s["norm"].double()

    y = {}
    buf, R, C, ty = s["weights"]["embd"]
    h = _decode(buf, R, C, ty)[s["token"]]
    for i in range(case["layers"]):
        n = {k: "%d.%s" % (i, k) for k in ("q", "k", "v", "o", "gate", "up", "down")}
        if i:
            h = h + y["%d.down" % (i - 1)]
        x = rms(h)
        for k in "qkv":
            y[n[k]] = product(n[k], x)
        y[n["o"]] = product(n["o"], y[n["q"]])
        h = h + y[n["o"]]
        x = rms(h)
        y[n["gate"]], y[n["up"]] = product(n["gate"], x), product(n["up"], x)
        y[n["down"]] = product(n["down"], torch.nn.functional.silu(y[n["gate"]]) * y[n["up"]])
    return dict(y, h=h)
