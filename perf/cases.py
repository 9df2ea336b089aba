"""The work a program gives this library, as measurable cases.

Six kinds of call, each through the public Python entry points
(needle-rs_amd/needle_amd.py) over device tensors:

  gemv8    Format B dequant-GEMV: decode, one activation row; one weight or a
           stack of them in one call
  gemm8    Format B GEMM: the rows of many sessions, or a prompt
  cq       Cactus-Quants projection: prepare_input, then matvec (one row) or
           matmul (several); `exact` asks for the reference's summation order
  kv       one decode step of a KV layer: append a token's K and V, attend;
           int8 cache (tolerance or reference order) or f32 cache
  prompt   int8 prompt attention: every prompt row attends to the prompt
  turn     a Needle-3 conversation turn: prefill the message, then greedy
           steps that feed back the token, logits of every step returned

Sizes are the shipped Needle-3 geometry's (768 wide, 12 query heads on 2 kv
heads, qk 48, v 64, 8192 tokens of vocabulary) and the benchmark's (3072 x 768
Format B weights, the 12 x 64 MHA cache at ctx 2048); drawn cases spread over
the sizes the entry points take.
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if os.path.join(ROOT, "needle-rs_amd") not in sys.path:
    sys.path.insert(0, os.path.join(ROOT, "needle-rs_amd"))

import needle_amd as nd  # noqa: E402
import v3_synth  # noqa: E402

TERNARY = 5


def listed():
    return [
        # one projection of one decode step, Format B: the smallest call
        dict(name="gemv8_one", kind="gemv8", count=1, out=3072, inn=768),
        # the benchmark's stack of weights in one call: the HBM stream
        dict(name="gemv8_stack", kind="gemv8", count=448, out=3072, inn=768),
        # the rows of 64 sessions through 20 layers' weights in one call
        dict(name="gemm8_rows64", kind="gemm8", count=20, m=64, out=3072, inn=768),
        # prompts of 500 tokens (ragged) through 32 weights in one call
        dict(name="gemm8_prefill", kind="gemm8", count=32, m=500, out=3072, inn=768),
        # the LM head of one decode step, 4-bit
        dict(name="cq_head_one", kind="cq", bits=4, out=8192, inn=768, rows=1, exact=False),
        # a 500-token prompt through the 4-bit LM-head shape
        dict(name="cq_head_rows", kind="cq", bits=4, out=8192, inn=768, rows=500, exact=False),
        # 64 sessions through a 2-bit layer projection, reference order
        dict(name="cq_exact_rows64", kind="cq", bits=2, out=768, inn=768, rows=64, exact=True),
        # a decode step of one Needle-3 layer for 64 sessions near 2048 tokens
        dict(name="kv_gqa_64", kind="kv", form="i8", heads=12, kv_heads=2, qk=48, cap=2048, ctx=2000,
             sessions=64, quant_query=True),
        # the benchmark's MHA cache, 320 sessions
        dict(name="kv_mha_320", kind="kv", form="i8", heads=12, kv_heads=12, qk=64, cap=2048, ctx=2048,
             sessions=320, quant_query=False),
        # a 2000-token prompt through a global layer's attention
        dict(name="prompt_2000", kind="prompt", heads=12, kv_heads=2, qk=48, seq=2000, window=0,
             quant_query=True),
        # one user's turn: a 128-token message, 32 tokens of answer
        dict(name="turn_one", kind="turn", sessions=1, ctx=256, prompt=128, steps=32, kv_int8=True),
        # a server's 64 sessions: 32 more tokens each, then 8 tokens of answer
        dict(name="turn_64", kind="turn", sessions=64, ctx=512, prompt=32, steps=8, kv_int8=True),
    ]


# ---- drawn cases ------------------------------------------------------------

def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gemv8", "gemm8", "cq", "cq", "kv", "kv", "prompt", "turn"])
    if kind == "gemv8":
        out = _log(rng, 64, 12288)  # any number of rows; widths in sixteens
        inn = 16 * _log(rng, 4, 256) if rng.random() < 0.5 else rng.choice([256, 512, 768, 1024])
        most = max(1, int(1.08e9 / (out * inn + 16 * out)))
        return dict(kind=kind, count=_log(rng, 1, min(448, most)), out=out, inn=inn)
    if kind == "gemm8":
        out, inn, m = 64 * _log(rng, 1, 96), 32 * _log(rng, 2, 96), _log(rng, 2, 2048)
        most = max(1, int(32 * 500 * 3072 * 768 / (m * out * inn)))
        return dict(kind=kind, count=_log(rng, 1, min(64, most)), m=m, out=out, inn=inn)
    if kind == "cq":
        rows = 1 if rng.random() < 0.3 else _log(rng, 2, 1024)
        return dict(kind=kind, bits=rng.choice([2, 2, 3, 4, 4, TERNARY]), out=_log(rng, 64, 8192),
                    inn=768 if rng.random() < 0.5 else _log(rng, 64, 3072), rows=rows,
                    exact=rng.random() < 0.3)
    if kind == "kv":
        heads, kv_heads, qk = rng.choice([(12, 2, 48), (12, 2, 48), (12, 12, 64), (8, 4, 64), (16, 2, 64)])
        form = rng.choice(["i8", "i8", "i8_exact", "f32"])
        cap = rng.choice([512, 1024, 2048, 4096, 8192])
        # past the ring's capacity the span is the last `cap` positions
        ctx = _log(rng, 16, 2 * cap)
        most = int(6.4e8 / (cap * kv_heads * (qk + 64))) if form == "i8" else \
            int(6e7 / (min(cap, ctx) * heads * (qk + 64)))
        return dict(kind=kind, form=form, heads=heads, kv_heads=kv_heads, qk=qk, cap=cap, ctx=ctx,
                    sessions=_log(rng, 1, max(1, min(320, most))),
                    quant_query=form != "f32" and rng.random() < 0.5)
    if kind == "prompt":
        heads, kv_heads, qk = rng.choice([(12, 2, 48), (12, 2, 48), (12, 12, 64), (8, 4, 64)])
        return dict(kind=kind, heads=heads, kv_heads=kv_heads, qk=qk, seq=_log(rng, 8, 3000),
                    window=rng.choice([0, 256, 1024]), quant_query=rng.random() < 0.5)
    sessions = _log(rng, 1, 64)
    prompt = min(_log(rng, 1, 256), max(1, 2048 // sessions))
    return dict(kind=kind, sessions=sessions, ctx=_log(rng, 1, 512), prompt=prompt,
                steps=rng.randint(1, 8), kv_int8=rng.random() < 0.7)


# ---- inputs -----------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


def _codes(g, *shape):
    return torch.randint(0, 256, shape, generator=g, device="cuda", dtype=torch.uint8)


def _cq_host(case, seed):
    """A Cactus-Quants blob: uniform codes, N(1, 0.1) norms sized so that an
    output is about as large as an activation."""
    rng = np.random.default_rng(int(seed))
    bits = 2 if case["bits"] == TERNARY else case["bits"]
    pad = -(-case["inn"] // 128) * 128
    packed = rng.integers(0, 256, size=(case["out"], pad * bits // 8), dtype=np.uint8)
    norms = np.abs(rng.normal(1.0, 0.1, size=(case["out"], pad // 128))) / math.sqrt(case["inn"]) * math.sqrt(128)
    return packed, norms.astype(np.float16)


def _kv_host(case, seed):
    """Per-session positions (ragged: a batch's sessions differ in length) and
    the spans they attend to."""
    n, ctx, cap = case["sessions"], case["ctx"], case["cap"]
    pos = np.array([ctx - 1 - (i * 37) % (ctx // 4 + 1) for i in range(n)], np.int32)
    return pos, np.maximum(pos + 1 - cap, 0).astype(np.int32)


_MODEL = {}


def _model():
    """The Needle-3 model (shipped geometry, random init): one per process, as
    a server has it."""
    if "m" not in _MODEL:
        geom, recs = v3_synth.build_records(seed=0)
        ctx = nd.Ctx(0)
        _MODEL["m"] = nd.V3Model(ctx, geom, recs, v3_synth.CODEBOOK)
    return _MODEL["m"]


def _conversation(st):
    """A batch of sessions that hold `ctx` tokens already."""
    chunk = min(256, max(st["prompt"].shape[1], 32))
    b = nd.V3Batch(_model(), st["prompt"].shape[0], 8192, max_chunk=chunk, kv_int8=st["kv_int8"])
    for t in range(0, st["past"].shape[1], chunk):
        b.prefill(st["past"][:, t:t + chunk], want_next=False)
    return b


def prepare(case, seed):
    kind, f32 = case["kind"], torch.float32
    if kind == "turn":
        rng = np.random.default_rng(int(seed))
        m, S = _model(), case["sessions"]
        st = dict(case=case, kv_int8=case["kv_int8"],
                  past=rng.integers(3, 8192, size=(S, case["ctx"])).astype(np.int32),
                  prompt=rng.integers(3, 8192, size=(S, case["prompt"])).astype(np.int32),
                  logits=torch.empty(case["steps"] + 1, S, m.rows, dtype=f32, device="cuda"))
        st["batch"] = _conversation(st)
        return st
    g = _gen(seed)
    st = dict(case=case, ctx=nd.Ctx(0))
    if kind in ("gemv8", "gemm8"):
        c, out, inn = case["count"], case["out"], case["inn"]
        st["w"] = _codes(g, c, out, inn)
        st["cb"] = _randn(g, c, (out + 63) // 64, 256) * 0.02
        rows = (case["m"],) if kind == "gemm8" else ()
        st["x"] = _randn(g, c, *rows, inn)
        st["y"] = torch.empty(c, *rows, out, dtype=f32, device="cuda")
    elif kind == "cq":
        packed, norms = _cq_host(case, seed)
        blob = np.concatenate([packed.reshape(-1), norms.reshape(-1).view(np.uint8)])
        st["w"] = nd.CqWeight(st["ctx"], blob, case["out"], case["inn"], 128, case["bits"],
                              v3_synth.CODEBOOK)
        st["x"] = _randn(g, case["rows"], case["inn"])
    elif kind == "kv":
        H, KVH, qk, cap, n = (case[k] for k in ("heads", "kv_heads", "qk", "cap", "sessions"))
        st["geom"] = nd.kv_geom(H, KVH, qk, 64, cap)
        alloc, write = (nd.kv_alloc_f32, nd.kv_write_f32) if case["form"] == "f32" else (nd.kv_alloc, nd.kv_write)
        st["kv"], st["stride"] = alloc(st["geom"], n, 0)
        pos, lo = _kv_host(case, seed)
        for i in range(n):  # the tokens before this step's
            old = torch.arange(int(lo[i]), int(pos[i]), dtype=torch.int32, device="cuda")
            if len(old):
                write(st["ctx"], st["geom"], st["kv"][i * st["stride"]:], 0, old,
                      _randn(g, len(old), KVH * qk), _randn(g, len(old), KVH * 64))
        st["k"], st["v"] = _randn(g, n, KVH * qk), _randn(g, n, KVH * 64)
        st["q"] = _randn(g, n, H * qk)
        st["pos"], st["lo"] = torch.from_numpy(pos).cuda(), torch.from_numpy(lo).cuda()
    else:
        H, KVH, qk, n = (case[k] for k in ("heads", "kv_heads", "qk", "seq"))
        st["q"], st["k"], st["v"] = _randn(g, n, H * qk), _randn(g, n, KVH * qk), _randn(g, n, KVH * 64)
    return st


# ---- one pass ---------------------------------------------------------------

def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "gemv8":
        if case["count"] == 1:
            return nd.cb8_gemv(st["ctx"], st["w"][0], st["cb"][0], st["x"][0], st["y"][0])
        return nd.cb8_gemv_batched(st["ctx"], st["w"], st["cb"], st["x"], st["y"])
    if kind == "gemm8":
        return nd.cb8_gemm_batched(st["ctx"], st["x"], st["w"], st["cb"], st["y"])
    if kind == "cq":
        w = st["w"]
        xh = w.prepare_input(st["x"])
        if case["rows"] == 1:
            return w.matvec_rows_prepared(xh, 0, w.out_feat, exact=case["exact"])
        return w.matmul_rows_prepared(xh, case["rows"], 0, w.out_feat, exact=case["exact"])
    if kind == "kv":
        ctx, g = st["ctx"], st["geom"]
        if case["form"] == "f32":
            nd.kv_write_f32(ctx, g, st["kv"], st["stride"], st["pos"], st["k"], st["v"])
            out = nd.attend_step_f32(ctx, g, st["kv"], st["stride"], st["lo"], st["pos"], st["q"])
        else:
            nd.kv_write(ctx, g, st["kv"], st["stride"], st["pos"], st["k"], st["v"])
            out = nd.attend_step_i8(ctx, g, st["kv"], st["stride"], st["lo"], st["pos"], st["q"],
                                    quant_query=case["quant_query"], exact=case["form"] == "i8_exact")
        return out, st["kv"]
    if kind == "prompt":
        if "ctx" not in st:
            st["ctx"] = nd.Ctx(0)
        return nd.attend_i8_prefill(st["ctx"], case["heads"], case["kv_heads"], case["qk"], 64, st["q"],
                                    st["k"], st["v"], window=case["window"], quant_query=case["quant_query"])
    b, logits = st["batch"], st["logits"]
    if int(b.positions()[0]) + case["prompt"] + case["steps"] > 8192:  # this conversation is full
        b = st["batch"] = _conversation(st)
    tokens = np.empty((case["steps"] + 1, case["sessions"]), np.int32)
    tokens[0] = b.prefill(st["prompt"], logits=logits[0]) if case["prompt"] > 1 else \
        b.step(st["prompt"], logits=logits[0])
    for s in range(case["steps"]):
        tokens[s + 1] = b.step(tokens[s], logits=logits[s + 1])
    return logits, tokens


# ---- what a pass cannot do without ------------------------------------------

def work(case):
    kind = case["kind"]
    if kind == "gemv8":
        c, o, i = case["count"], case["out"], case["inn"]
        return dict(bytes=c * (o * i + (o + 63) // 64 * 1024 + 4 * i + 4 * o), flops=2 * c * o * i)
    if kind == "gemm8":
        c, m, o, i = case["count"], case["m"], case["out"], case["inn"]
        return dict(bytes=c * (o * i + o // 64 * 1024 + 4 * m * i + 4 * m * o), flops=2 * c * m * o * i)
    if kind == "cq":
        o, i, r = case["out"], case["inn"], case["rows"]
        pad = -(-i // 128) * 128
        bits = 2 if case["bits"] == TERNARY else case["bits"]
        return dict(bytes=o * pad * bits // 8 + o * (pad // 128) * 2 + 4 * r * (i + o), flops=2 * r * o * pad)
    if kind == "kv":
        H, KVH, qk = case["heads"], case["kv_heads"], case["qk"]
        pos, lo = _kv_host(case, 0)
        span = int((pos + 1 - lo).sum())
        per = KVH * (4 * (qk + 64) if case["form"] == "f32" else qk + 64 + 8)
        io = 4 * case["sessions"] * (H * (qk + 64) + KVH * (qk + 64))
        return dict(bytes=span * per + io, flops=2 * span * H * (qk + 64))
    if kind == "prompt":
        H, KVH, qk, n = case["heads"], case["kv_heads"], case["qk"], case["seq"]
        w = case["window"] or n
        pairs = sum(min(t + 1, w) for t in range(n))
        return dict(bytes=4 * n * (H + KVH) * (qk + 64), flops=2 * pairs * H * (qk + 64))
    S, P, N, ctx = case["sessions"], case["prompt"], case["steps"], case["ctx"]
    # multiply-adds a token: projections, MLP factors, mHC and Engram
    layer = 768 * (576 + 96 + 128 + 768) + 768 * 768 + 3 * 1024 * 64 + 24 * 3072 + 16 * 1024
    macs = 20 * layer + 5 * 2 * 768 * 768
    kv = 20 * 2 * (4 * 112 if not case["kv_int8"] else 112 + 8)
    weights = 20 * (768 * (576 + 96 + 128 + 768 + 768) // 4 + 400_000) + 5 * 2 * 768 * 768 // 4 + 8192 * 768 // 2
    att = 20 * 12 * 112 * (ctx + P)
    return dict(bytes=(N + 1) * weights + S * (N + 1) * (ctx + P) * kv + 4 * S * 8192 * (N + 1),
                flops=2 * S * ((P + N) * (macs + att) + (N + 1) * 768 * 8192))


def tolerance(case):
    kind = case["kind"]
    # the reference's own float order: every bit is given
    if kind == "turn" or (kind == "cq" and case["exact"]) or (kind == "kv" and case["form"] != "i8"):
        return "exact"
    if kind == "gemm8":
        return {"rel": 1e-2}  # both operands rounded to bf16, fp32 sums
    return {"rel": 2e-6, "max": 1e-4}  # fp32 sums in another order


# ---- the same in 64 bits ----------------------------------------------------

def _cq_exact(case, seed):
    packed, norms = _cq_host(case, seed)
    bits = 2 if case["bits"] == TERNARY else case["bits"]
    pad = -(-case["inn"] // 128) * 128
    cb = v3_synth.CODEBOOK
    if case["bits"] == TERNARY:
        s = np.float32(1.2240064) / np.float32(math.sqrt(128))
        lv = np.array([0.0, s, 0.0, -s], np.float64)  # crumb -> level
    else:
        lv = cb[{2: 0, 3: 4, 4: 12}[bits]:][:1 << bits].astype(np.float64)
    b = torch.from_numpy(packed).cuda()
    bit = torch.stack([(b >> i) & 1 for i in range(8)], -1).reshape(case["out"], pad, bits)
    code = sum(bit[..., i].long() << i for i in range(bits))
    w = torch.from_numpy(lv).cuda()[code].reshape(case["out"], pad // 128, 128) * \
        torch.from_numpy(norms.astype(np.float64)).cuda()[..., None]
    x = _randn(_gen(seed), case["rows"], case["inn"]).double()
    x = torch.nn.functional.pad(x, (0, pad - case["inn"])).reshape(case["rows"], pad // 128, 128)
    h = torch.ones(1, 1, dtype=torch.float64, device="cuda")
    while h.shape[0] < 128:
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    xh = (x @ h / math.sqrt(128)).reshape(case["rows"], pad)
    return (xh @ w.reshape(case["out"], pad).t()).reshape(-1)


def _quant(x):
    """The cache's codes and scales (defined by these 32-bit steps)."""
    amax = x.abs().amax(-1, keepdim=True)
    one = torch.ones_like(amax)  # tensor by tensor: the rounded quotient, no product with 1/127
    scale = torch.where(amax > 0, torch.div(amax, one * 127), one)
    y = x * torch.div(one, scale)
    r = torch.sign(y) * torch.floor(y.abs().double() + 0.5).float()
    return r.clamp(-128, 127), scale


def _attend64(q, k, v, lo, hi):
    """q [n][H][qk], k and v [m][KVH][..] in 64 bits; row i sees lo[i]..hi[i]."""
    n, H, qk = q.shape
    rep, at = H // k.shape[1], torch.arange(k.shape[0], device="cuda")
    mask = (at[None] >= lo[:, None]) & (at[None] <= hi[:, None])
    out = torch.empty(n, H, v.shape[2], dtype=torch.float64, device="cuda")
    for h in range(H):
        s = (q[:, h] @ k[:, h // rep].t()) * float(np.float32(1.0) / np.sqrt(np.float32(qk)))
        out[:, h] = torch.softmax(s.masked_fill(~mask, -math.inf), -1) @ v[:, h // rep]
    return out.reshape(n, -1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "turn":
        return None  # a code of the int8 cache that rounds the other way moves all later logits
    if kind == "cq":
        return _cq_exact(case, seed)
    g = _gen(seed)
    if kind in ("gemv8", "gemm8"):
        c, out, inn = case["count"], case["out"], case["inn"]
        w, cb = _codes(g, c, out, inn), _randn(g, c, (out + 63) // 64, 256) * 0.02
        x = _randn(g, c, *((case["m"],) if kind == "gemm8" else ()), inn)
        y = torch.empty(*x.shape[:-1], out, dtype=torch.float64, device="cuda")
        tile = torch.arange(out, device="cuda") // 64
        for i in range(c):
            wd = torch.gather(cb[i].double()[tile], 1, w[i].long())
            y[i] = x[i].double() @ wd.t()
        return y[0] if kind == "gemv8" and c == 1 else y
    H, KVH, qk = case["heads"], case["kv_heads"], case["qk"]
    if kind == "kv":
        n, f32 = case["sessions"], case["form"] == "f32"
        pos, lo = _kv_host(case, seed)
        old = []
        for i in range(n):
            m = int(pos[i] - lo[i])
            old.append((_randn(g, m, KVH * qk), _randn(g, m, KVH * 64)) if m else None)
        k, v, q = _randn(g, n, KVH * qk), _randn(g, n, KVH * 64), _randn(g, n, H * qk)
        out = torch.empty(n, H * 64, dtype=torch.float64, device="cuda")
        for i in range(n):
            ki = torch.cat(([old[i][0]] if old[i] else []) + [k[i:i + 1]]).reshape(-1, KVH, qk)
            vi = torch.cat(([old[i][1]] if old[i] else []) + [v[i:i + 1]]).reshape(-1, KVH, 64)
            out[i] = _one(case, q[i:i + 1].reshape(1, H, qk), ki, vi, f32)[0]
        return out, None
    n = case["seq"]
    q, k, v = _randn(g, n, H * qk), _randn(g, n, KVH * qk), _randn(g, n, KVH * 64)
    return _one(case, q.reshape(n, H, qk), k.reshape(n, KVH, qk), v.reshape(n, KVH, 64), False)


def _one(case, q, k, v, f32):
    m = k.shape[0]
    if case["quant_query"]:
        c, s = _quant(q)
        q = c * s
    if not f32:
        (kc, ks), (vc, vs) = _quant(k), _quant(v)
        k, v = kc.double() * ks.double(), vc.double() * vs.double()
    hi = torch.arange(m, device="cuda") if q.shape[0] > 1 or case["kind"] == "prompt" else \
        torch.tensor([m - 1], device="cuda")
    lo = (hi + 1 - case["window"]).clamp(min=0) if case.get("window") else torch.zeros_like(hi)
    return _attend64(q.double(), k.double(), v.double(), lo, hi)
