"""Timed cases of the framework's public entry points (kestrel_amd.kmoe.Context
and kestrel_amd.decoder.Decoder), over the range of calls a program that serves
a GGUF model makes: one-token decode, decode batches, prompt prefill, single
projections, attention and a whole decode stack.

listed() names the cases, draw() gives more of the same ranges, prepare() makes
what a program holds before the call (weights in HBM, inputs), run() is one
pass, work() the bytes and operations it cannot do without, exact() the same
outputs in 64 bits with plain torch.
"""
import math

import numpy as np
import torch

from kestrel_amd import kmoe
from kestrel_amd.decoder import Decoder

DEV = "cuda:0"
Q8_0, Q4_K, Q6_K = kmoe.Q8_0, kmoe.Q4_K, kmoe.Q6_K
TYPES = {"q8_0": Q8_0, "q4_k": Q4_K, "q6_k": Q6_K}
BLOCK = {Q8_0: (32, 34), Q4_K: (256, 144), Q6_K: (256, 210)}
REGIMES = {"avx2": kmoe.REGIME_AVX2, "int8": kmoe.REGIME_INT8}

# MoE layer shapes the benchmark and the tests use: experts, experts per token,
# hidden, expert FFN, weight types (gate and up, down), renormalised top-k,
# weights scale, Zipf exponent of the routing, shared expert's FFN.
LAYERS = {
    "mixtral": dict(e=8, k=2, d=4096, f=14336, gu=Q4_K, dn=Q4_K, norm=True, scale=0.0, zipf=0.0, shared=0),
    "mixtral-q4km": dict(e=8, k=2, d=4096, f=14336, gu=Q4_K, dn=Q6_K, norm=True, scale=0.0, zipf=0.0, shared=0),
    "qwen3": dict(e=128, k=8, d=2048, f=768, gu=Q4_K, dn=Q4_K, norm=True, scale=0.0, zipf=1.1, shared=0),
    "dsv2lite": dict(e=64, k=6, d=2048, f=1408, gu=Q4_K, dn=Q8_0, norm=False, scale=1.0, zipf=0.0, shared=2816),
    "moe6b": dict(e=32, k=4, d=2048, f=1536, gu=Q4_K, dn=Q4_K, norm=False, scale=0.0, zipf=0.0, shared=0),
}
# The decode stack: moe6b's layers (16 query heads over 4 KV heads of 128,
# Q4_K embedding, Q6_K head over a 32000-word vocabulary), cut in depth.
STACK = dict(layers=2, heads=16, kv=4, hd=128, vocab=32000, steps=4)


def listed():
    return [
        # one projection of one decoding token: the smallest call
        dict(name="matvec-q4k-4096", kind="matmul", t="q4_k", rows=4096, cols=4096, s=1),
        # the same projection over a prompt chunk
        dict(name="proj-q4k-512", kind="matmul", t="q4_k", rows=4096, cols=4096, s=512),
        # one decoding token through a Mixtral-shaped layer (the headline)
        dict(name="mixtral-1", kind="moe", shape="mixtral", s=1, regime="avx2"),
        # one decoding token through a small-expert layer with a shared expert
        dict(name="dsv2lite-1", kind="moe", shape="dsv2lite", s=1, regime="avx2"),
        # a decode batch of 13 sequences, Q4_K_M file mix (Q6_K down)
        dict(name="mixtral-q4km-13", kind="moe", shape="mixtral-q4km", s=13, regime="avx2"),
        # a decode batch of 48 sequences over many small experts, integer path
        dict(name="qwen3-48-int8", kind="moe", shape="qwen3", s=48, regime="int8"),
        # a 512-token prompt chunk on the integer path
        dict(name="mixtral-512-int8", kind="moe", shape="mixtral", s=512, regime="int8"),
        # a long ragged prompt chunk over many small experts, default arithmetic
        dict(name="qwen3-1777", kind="moe", shape="qwen3", s=1777, regime="avx2"),
        # a short prompt through a layer with Q8_0 down rows and a shared expert
        dict(name="dsv2lite-203", kind="moe", shape="dsv2lite", s=203, regime="avx2"),
        # prompt attention: a chunk after an earlier one, grouped-query heads
        dict(name="attn-777-at-611", kind="attn", heads=16, kv=4, hd=128, s=777, pos=611),
        # one decoding token's attention over a long context, multi-head
        dict(name="attn-1-at-3000", kind="attn", heads=16, kv=16, hd=128, s=1, pos=3000),
        # a whole stack: a prompt, then single-token steps, logits of each
        dict(name="stack-96", kind="stack", s=96),
    ]


def _between(rng, lo, hi):
    """A whole number spread evenly over the logarithm of lo..hi."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def draw(rng):
    kind = rng.choice(["matmul", "moe", "moe", "moe", "attn", "attn", "stack"])
    if kind == "matmul":
        s = rng.choice([1, _between(rng, 2, 512)])
        rows, cols = rng.choice([(4096, 4096), (3072, 2048), (6144, 2048), (2048, 2816), (4096, 14336),
                                 (14336, 4096), (10944, 2048), (32000, 2048)])
        if s > 64 and rows * cols > 1 << 25:
            rows, cols = 4096, 4096
        return dict(kind="matmul", t=rng.choice(["q4_k", "q4_k", "q6_k", "q8_0"]), rows=rows, cols=cols, s=s)
    if kind == "moe":
        shape = rng.choice(sorted(LAYERS))
        most = 512 if shape.startswith("mixtral") else 2048
        s = rng.choice([1, _between(rng, 2, 64), _between(rng, 65, most)])
        return dict(kind="moe", shape=shape, s=s, regime=rng.choice(["avx2", "avx2", "int8"]))
    if kind == "attn":
        heads, kv, hd = rng.choice([(16, 4, 128), (16, 16, 128), (32, 8, 128), (16, 8, 64)])
        s = rng.choice([1, _between(rng, 2, 1024)])
        return dict(kind="attn", heads=heads, kv=kv, hd=hd, s=s, pos=_between(rng, 1, 4096 if s == 1 else 1024) - 1)
    return dict(kind="stack", s=_between(rng, 5, 400))


# ------------------------------------------------------------------- inputs

def _gen(seed, *more):
    g = torch.Generator(device=DEV)
    v = 1469598103934665603
    for m in (seed,) + more:
        v = ((v ^ (int(m) & 0xffffffff)) * 1099511628211) & 0x7fffffffffffffff
    g.manual_seed(v)
    return g


def _f16_bytes(v):
    return v.to(torch.float16).view(torch.uint8).reshape(-1, 2)


def _blocks(t, rows, cols, g, std=0.02):
    """Random well-formed blocks: uniform quants and sub-scales, block scales
    spread around the one that gives zero-mean weights of about `std`."""
    n, size = rows * cols // BLOCK[t][0], BLOCK[t][1]
    raw = torch.randint(0, 256, (n * size,), dtype=torch.uint8, device=DEV, generator=g).view(n, size)
    spread = torch.exp(0.3 * torch.randn(n, device=DEV, generator=g))
    if t == Q4_K:
        raw[:, 0:2] = _f16_bytes(spread * (std / 0.02) * 1.4e-4)
        raw[:, 2:4] = _f16_bytes(spread * (std / 0.02) * 7.5 * 1.4e-4)
    elif t == Q6_K:
        raw[:, 208:210] = _f16_bytes(spread * (std / 0.02) * 1.5e-5)
    else:
        raw[:, 0:2] = _f16_bytes(spread * std / 74.0)
    return raw.view(-1)


def _normal(g, *shape, std=1.0, mean=0.0):
    return torch.randn(*shape, device=DEV, generator=g) * std + mean


def _moe_tensors(case, seed):
    """Router, the three expert parts [E, bytes], the shared expert's parts, activations."""
    c = LAYERS[case["shape"]]
    g = _gen(seed, 1)
    router = _normal(g, c["e"], c["d"], std=0.02)
    x = _normal(g, case["s"], c["d"])
    if c["zipf"]:  # a rank-1 term that activations of mean 1 carry into the logits
        rank = torch.from_numpy(np.random.RandomState(seed & 0x7fffffff).permutation(c["e"]) + 1).to(DEV)
        router += (-c["zipf"] * torch.log(rank.float()) / c["d"])[:, None]
        x += 1.0
    shapes = ((c["gu"], c["f"], c["d"]), (c["gu"], c["f"], c["d"]), (c["dn"], c["d"], c["f"]))
    parts = [_blocks(t, c["e"] * r, n, g).view(c["e"], -1) for t, r, n in shapes]
    shared = None
    if c["shared"]:
        shared = [_blocks(t, r, n, g) for t, r, n in ((Q4_K, c["shared"], c["d"]), (Q4_K, c["shared"], c["d"]),
                                                     (Q6_K, c["d"], c["shared"]))]
    return c, router, parts, shared, x


def _attn_tensors(case, seed):
    g = _gen(seed, 2)
    n = case["pos"] + case["s"]
    q = _normal(g, case["s"], case["heads"] * case["hd"])
    k, v = (_normal(g, n, case["kv"] * case["hd"]).to(torch.float16) for _ in range(2))
    return q, k, v


def _matmul_tensors(case, seed):
    g = _gen(seed, 3)
    return _blocks(TYPES[case["t"]], case["rows"], case["cols"], g), _normal(g, case["s"], case["cols"])


def _stack_tensors(case, seed):
    """(hp, tensors by GGUF name as device bytes, prompt, step tokens)."""
    c, m = STACK, LAYERS["moe6b"]
    g = _gen(seed, 4)
    d, f, e, hd = m["d"], m["f"], m["e"], c["hd"]
    hp = dict(arch="llama", n_layer=c["layers"], n_embd=d, n_head=c["heads"], n_head_kv=c["kv"], head_dim=hd,
              rope_dim=hd, rope_freq_base=10000.0, rms_eps=1e-5, n_ctx=case["s"] + c["steps"], n_batch=512,
              n_expert=e, n_expert_used=m["k"], norm_topk=m["norm"], weights_scale=m["scale"])

    def mat(t, rows, cols, std, n=0):
        return (t, [cols, rows] + ([n] if n else []), _blocks(t, rows * max(1, n), cols, g, std))

    def f32(*shape, std, mean=0.0):
        return (kmoe.F32, list(shape)[::-1], _normal(g, *shape, std=std, mean=mean).view(torch.uint8).reshape(-1))

    t = {"token_embd.weight": mat(Q4_K, c["vocab"], d, 1.0), "output_norm.weight": f32(d, std=0.1, mean=1.0),
         "output.weight": mat(Q6_K, c["vocab"], d, d ** -0.5)}
    for l in range(c["layers"]):
        p = "blk.%d." % l
        t[p + "attn_norm.weight"] = f32(d, std=0.1, mean=1.0)
        t[p + "ffn_norm.weight"] = f32(d, std=0.1, mean=1.0)
        for n, rows in (("q", c["heads"]), ("k", c["kv"]), ("v", c["kv"])):
            t[p + "attn_%s.weight" % n] = mat(Q4_K, rows * hd, d, d ** -0.5)
        t[p + "attn_output.weight"] = mat(Q4_K, d, c["heads"] * hd, d ** -0.5)
        t[p + "ffn_gate_inp.weight"] = f32(e, d, std=4.0 * d ** -0.5)
        t[p + "ffn_gate_exps.weight"] = mat(Q4_K, f, d, d ** -0.5, e)
        t[p + "ffn_up_exps.weight"] = mat(Q4_K, f, d, d ** -0.5, e)
        t[p + "ffn_down_exps.weight"] = mat(Q4_K, d, f, f ** -0.5, e)
    ids = np.random.RandomState(seed & 0x7fffffff).randint(0, c["vocab"], case["s"] + c["steps"]).tolist()
    return hp, t, ids[:case["s"]], ids[case["s"]:]


# -------------------------------------------------------------------- passes

def prepare(case, seed):
    ctx = kmoe.Context(0)
    ctx.set_regime(REGIMES[case.get("regime", "avx2")])
    s = dict(case=case, ctx=ctx)
    if case["kind"] == "matmul":
        s["w"], s["x"] = _matmul_tensors(case, seed)
    elif case["kind"] == "moe":
        c, router, parts, shared, s["x"] = _moe_tensors(case, seed)
        ctx.layer_create(0, c["e"], c["k"], c["d"], c["f"], c["gu"], c["gu"], c["dn"], c["norm"], c["scale"])
        ctx.router_upload(0, router.cpu().numpy())
        for p in range(3):
            for e in range(c["e"]):
                ctx.expert_upload(0, e, p, parts[p][e])
        if shared:
            ctx.shared_expert(0, c["shared"], (Q4_K, Q4_K, Q6_K), *[w.cpu().numpy() for w in shared])
        ctx.sync()
    elif case["kind"] == "attn":
        s["q"], k, v = _attn_tensors(case, seed)
        s["k"], s["v"] = k.view(torch.int16), v.view(torch.int16)
    else:
        hp, t, s["prompt"], s["steps"] = _stack_tensors(case, seed)
        s["dec"] = Decoder(ctx, hp, {n: (ty, dims, b.cpu().numpy()) for n, (ty, dims, b) in t.items()})
    return s


def run(s):
    case, ctx = s["case"], s["ctx"]
    if case["kind"] == "matmul":
        return ctx.matmul(TYPES[case["t"]], s["w"], case["rows"], case["cols"], s["x"])
    if case["kind"] == "moe":
        return ctx.moe_ffn(0, s["x"])
    if case["kind"] == "attn":
        return ctx.attention(s["q"], s["k"], s["v"], case["heads"], case["kv"], case["hd"], case["pos"],
                             case["pos"] + case["s"])
    dec = s["dec"]
    dec.cached = 0  # a new sequence
    return [dec.forward(s["prompt"])] + [dec.forward([t]) for t in s["steps"]]


def _bytes(t, rows, cols):
    return rows * cols // BLOCK[t][0] * BLOCK[t][1]


def _moe_work(c, s):
    if c["zipf"]:
        z = np.arange(1, c["e"] + 1, dtype=np.float64) ** -c["zipf"]
        p = np.minimum(1.0, c["k"] * z / z.sum())
    else:
        p = np.full(c["e"], c["k"] / c["e"])
    touched = float(np.sum(1.0 - (1.0 - p) ** s))
    expert = 2 * _bytes(c["gu"], c["f"], c["d"]) + _bytes(c["dn"], c["d"], c["f"])
    b = touched * expert + 4 * c["e"] * c["d"] + 8 * s * c["d"]
    fl = 2.0 * s * c["d"] * (3 * c["k"] * c["f"] + c["e"])
    if c["shared"]:
        b += 2 * _bytes(Q4_K, c["shared"], c["d"]) + _bytes(Q6_K, c["d"], c["shared"])
        fl += 6.0 * s * c["d"] * c["shared"]
    return b, fl


def _attn_work(heads, kv, hd, s, pos):
    seen = s * pos + s * (s + 1) / 2.0
    return 8.0 * s * heads * hd + 4.0 * (pos + s) * kv * hd, 4.0 * heads * hd * seen


def work(case):
    if case["kind"] == "matmul":
        rows, cols, s = case["rows"], case["cols"], case["s"]
        b, f = _bytes(TYPES[case["t"]], rows, cols) + 4.0 * s * (rows + cols), 2.0 * s * rows * cols
    elif case["kind"] == "moe":
        b, f = _moe_work(LAYERS[case["shape"]], case["s"])
    elif case["kind"] == "attn":
        b, f = _attn_work(case["heads"], case["kv"], case["hd"], case["s"], case["pos"])
    else:
        c, m = STACK, LAYERS["moe6b"]
        d, nq, nkv = m["d"], c["heads"] * c["hd"], c["kv"] * c["hd"]
        b = f = 0.0
        for s, pos in [(case["s"], 0)] + [(1, case["s"] + i) for i in range(c["steps"])]:
            mb, mf = _moe_work(m, s)
            ab, af = _attn_work(c["heads"], c["kv"], c["hd"], s, pos)
            b += c["layers"] * (mb + ab + _bytes(Q4_K, nq + 2 * nkv, d) + _bytes(Q4_K, d, nq))
            b += _bytes(Q6_K, c["vocab"], d) + 4 * c["vocab"] + 4 * s * d
            f += c["layers"] * (mf + af + 2.0 * s * d * (2 * nq + 2 * nkv)) + 2.0 * c["vocab"] * d
    return {"bytes": b, "flops": f}


def tolerance(case):
    # Four times what the paths were seen to be off by in 64 bits. Where sums
    # are rounded to int8 on the way (the integer path, experts of fewer than
    # four rows), a rounding that falls the other way moves a value by 1/127 of
    # its block's largest; through a stack of single-token steps such roundings
    # multiply (1.5e-2 seen).
    if case["kind"] == "attn":
        return {"rel": 1.2e-6, "max": 5e-5}
    if case["kind"] == "matmul":
        return {"rel": 2.8e-6, "max": 5e-5}
    if case["kind"] == "moe":
        if case["regime"] == "int8":
            return {"rel": 8e-4, "max": 1.5e-2}
        return {"rel": 4e-4 if case["s"] <= 64 else 1e-4, "max": 1e-2}
    return {"rel": 3e-2, "max": 5e-1}


# --------------------------------------------------- the same in 64 bits

def _dequant(t, raw, rows, cols):
    """GGUF block bytes -> weights in float64."""
    b = raw.view(-1, BLOCK[t][1])

    def half(i):
        return b[:, i:i + 2].contiguous().view(torch.float16).double()

    if t == Q8_0:
        w = b[:, 2:].contiguous().view(torch.int8).double() * half(0)
    elif t == Q4_K:
        sc = b[:, 4:16].to(torch.int32)
        lo, hi, x = sc[:, 0:4], sc[:, 4:8], sc[:, 8:12]
        scale = torch.cat([lo & 63, (x & 15) | ((lo >> 6) << 4)], 1).double() * half(0)
        minus = torch.cat([hi & 63, (x >> 4) | ((hi >> 6) << 4)], 1).double() * half(2)
        qs = b[:, 16:].reshape(-1, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).reshape(-1, 8, 32).double()
        w = q * scale[:, :, None] - minus[:, :, None]
    else:
        ql = b[:, :128].reshape(-1, 2, 2, 32).to(torch.int32)
        qh = b[:, 128:192].reshape(-1, 2, 1, 32).to(torch.int32)
        rows4 = [(ql[:, :, r & 1] >> (4 * (r >> 1))) & 15 for r in range(4)]
        q = torch.stack([rows4[r] | (((qh[:, :, 0] >> (2 * r)) & 3) << 4) for r in range(4)], 2) - 32
        sc = b[:, 192:208].contiguous().view(torch.int8).double() * half(208)
        w = q.reshape(-1, 16, 16).double() * sc[:, :, None]
    return w.reshape(rows, cols)


def _int8_rows(x, block):
    """Activations as the integer path rounds them: int8 per block, times the block's scale."""
    v = x.float().reshape(x.shape[0], -1, block)
    scale = v.abs().amax(2, keepdim=True) / 127.0
    inv = torch.where(scale > 0, 1.0 / scale, torch.zeros_like(scale))
    t = v * inv
    q = torch.sign(t) * torch.floor(t.abs() + 0.5)
    return (q.clamp(-127, 127).double() * scale.double()).reshape(x.shape)


def _mm(t, w, x, regime):
    """x [n, cols] times w [rows, cols]: quant::matmul's choice of arithmetic, sums in float64."""
    if regime == "int8" or x.shape[0] < 4:
        x = _int8_rows(x, 32 if t == Q8_0 else 256)
    return x.double() @ w.T


def _moe64(c, router, parts, shared, x, regime):
    logits = x.double() @ router.double().T
    p, idx = torch.topk(torch.softmax(logits, 1), c["k"], dim=1)
    if c["norm"]:
        p = p / p.sum(1, keepdim=True).clamp_min(2.0 ** -14)
    if c["scale"] not in (0.0, 1.0):
        p = p * c["scale"]
    out = torch.zeros(x.shape, dtype=torch.float64, device=x.device)

    def ffn(w3, types, f, rows):
        g, u = (_mm(types[i], _dequant(types[i], w3[i], f, c["d"]), rows, regime) for i in range(2))
        h = g / (1.0 + torch.exp(-g)) * u
        return _mm(types[2], _dequant(types[2], w3[2], c["d"], f), h, regime)

    for e in range(c["e"]):
        tok, slot = torch.nonzero(idx == e, as_tuple=True)
        if tok.numel():
            y = ffn([q[e] for q in parts], (c["gu"], c["gu"], c["dn"]), c["f"], x[tok])
            out[tok] += y * p[tok, slot][:, None]
    if shared:
        out += ffn(shared, (Q4_K, Q4_K, Q6_K), c["shared"], x)
    return out


def _attn64(q, k, v, heads, kv, hd, pos):
    s, n = q.shape[0], pos + q.shape[0]
    keep = torch.arange(n, device=q.device)[None, :] <= pos + torch.arange(s, device=q.device)[:, None]
    qh = q.double().reshape(s, heads, hd)
    out = torch.empty_like(qh)
    for h in range(heads):
        kh, vh = (t.double().reshape(-1, kv, hd)[:n, h // (heads // kv)] for t in (k, v))
        sc = (qh[:, h] @ kh.T) / math.sqrt(hd)
        out[:, h] = torch.softmax(sc.masked_fill(~keep, float("-inf")), 1) @ vh
    return out.reshape(s, heads * hd)


def exact(case, seed):
    if case["kind"] == "matmul":
        w, x = _matmul_tensors(case, seed)
        t = TYPES[case["t"]]
        return _mm(t, _dequant(t, w, case["rows"], case["cols"]), x, "avx2")
    if case["kind"] == "moe":
        return _moe64(*_moe_tensors(case, seed), case["regime"])
    if case["kind"] == "attn":
        return _attn64(*_attn_tensors(case, seed), case["heads"], case["kv"], case["hd"], case["pos"])
    # A stack has no one value in 64 bits: each step rounds activations to int8,
    # and roundings that fall the other way spread through the layers.
    return None
