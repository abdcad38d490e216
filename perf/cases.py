"""The workloads whose speed is tracked: blocks of Qwen3-shaped models at the sizes of this repository's benchmark and
tests, each run through the public C ABI (include/malkin_hip.h, include/malkin_model.h) as the model's forward runs
it. A case is a dict of plain values; its "kind" says which block it is:

  mlp       rmsnorm, gate|up matmul, silu(gate) * up, down matmul over n tokens
  attn      rmsnorm, q|k|v matmul, QK-norm + RoPE + int8 KV write, attention, attn_output matmul. mode "decode": n
            sequences with one new token each; "prefill": n tokens of one sequence behind `past` keys; "tree": the
            verification tree of a speculative step (next token, a chain of drafts and one alternative per draft)
  head      final norm, LM head and token selection for n rows: the greedy top-2, or the sampler's top-k
  generate  a whole model: prompt, greedy decoding (the captured decode graph), then the logits of the last token

Weights are N(0, 0.02) quantized to the case's type, activations N(0, 1) with a few large channels, cached keys and
values N(0, 1) rows quantized as the KV write quantizes them. Everything follows from the seed.
"""
import ctypes
import math
import os
import tempfile

import numpy as np
import torch

import malkin_amd as mk

TYPES = {"f16": mk.F16, "bf16": mk.BF16, "q8_0": mk.Q8_0, "q4_k": mk.Q4_K, "q5_k": mk.Q5_K, "q6_k": mk.Q6_K}
BLOCK = {"f16": (1, 2), "bf16": (1, 2), "q8_0": (32, 34), "q4_k": (256, 144), "q5_k": (256, 176), "q6_k": (256, 210)}
EPS, ROPE_BASE, D = 1e-6, 1e6, 128


def listed():
    return [
        # One decode step of a small draft model (Qwen3-0.6B width, Q4_K): the smallest calls, launches count.
        {"name": "mlp_decode_q4k_small", "kind": "mlp", "type": "q4_k", "n": 1, "embd": 1024, "ff": 3072},
        # Single-stream decoding, 8B width in Q8_0, some 600 tokens into a chat: the attention half of a layer.
        {"name": "attn_decode_q8", "kind": "attn", "mode": "decode", "type": "q8_0", "n": 1, "embd": 4096,
         "heads": 32, "past": 600, "ctx": 4096},
        # Eight users decoding together (continuous batching), contexts of 256 to 1024 tokens.
        {"name": "attn_batch8_q8", "kind": "attn", "mode": "decode", "type": "q8_0", "n": 8, "embd": 4096,
         "heads": 32, "past": 1024, "ctx": 4096},
        # Speculative verification of 17 tree nodes on a 14B-width Q6_K target: the MLP, then the attention over a
        # 2048-token prefix.
        {"name": "mlp_tree17_q6k", "kind": "mlp", "type": "q6_k", "n": 17, "embd": 5120, "ff": 17408},
        {"name": "attn_tree17_q6k", "kind": "attn", "mode": "tree", "type": "q6_k", "n": 17, "embd": 5120,
         "heads": 40, "past": 2048, "ctx": 4096},
        # A long prompt on the 8B width: a full 512-token forward, its MLP and the attention of the second chunk.
        {"name": "mlp_prompt512_q8", "kind": "mlp", "type": "q8_0", "n": 512, "embd": 4096, "ff": 12288},
        {"name": "attn_prompt512_q8", "kind": "attn", "mode": "prefill", "type": "q8_0", "n": 512, "embd": 4096,
         "heads": 32, "past": 512, "ctx": 4096},
        # A prompt of ordinary, ragged length on a 4B-width Q4_K model.
        {"name": "mlp_prompt203_q4k", "kind": "mlp", "type": "q4_k", "n": 203, "embd": 2560, "ff": 9728},
        # Q5_K, a common GGUF choice between Q4_K and Q6_K: a decode step at 4B width.
        {"name": "mlp_decode_q5k", "kind": "mlp", "type": "q5_k", "n": 1, "embd": 2560, "ff": 9728},
        # An unquantized BF16 GGUF: a chat prompt on the 0.6B width.
        {"name": "mlp_prompt96_bf16", "kind": "mlp", "type": "bf16", "n": 96, "embd": 1024, "ff": 3072},
        # The LM head over the Qwen3 vocabulary and the top-40 cut of eight sampled requests.
        {"name": "head_sample8_q8", "kind": "head", "type": "q8_0", "n": 8, "embd": 4096, "vocab": 151936,
         "top_k": 40},
        # A chat turn end to end on four layers of the 8B width: 512-token prompt, 64 greedy tokens.
        {"name": "generate_8b_layers", "kind": "generate", "type": "q8_0", "layers": 4, "vocab": 16384, "prompt": 512,
         "gen": 64, "ctx": 1024},
    ]


# What the largest listed cases cost: 512 tokens through the 8B-width MLP.
MOST_MACS = 512 * 4096 * 12288


def log_int(rng, lo, hi):
    return min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))


def draw(rng):
    kind = rng.choice(["mlp", "mlp", "mlp", "mlp", "attn", "attn", "attn", "attn", "head", "generate"])
    if kind == "mlp":
        t = rng.choice(["q8_0", "q8_0", "q4_k", "q4_k", "q6_k", "q6_k", "q5_k", "bf16", "f16"])
        packed = t in ("q8_0", "q4_k", "q6_k")
        embd = 256 * rng.randint(4, 20 if packed else 10)
        ff = 256 * round(embd * rng.uniform(2.4, 3.8) / 256)
        n = log_int(rng, 1, 512 if packed else 256)
        return {"kind": kind, "type": t, "n": max(1, min(n, MOST_MACS // (embd * ff))), "embd": embd, "ff": ff}
    if kind == "attn":
        heads = rng.choice([16, 32, 40])
        c = {"kind": kind, "mode": rng.choice(["decode", "prefill", "tree"]), "type": rng.choice(["q8_0", "q4_k", "q6_k"]),
             "embd": {16: 1024, 32: rng.choice([2560, 4096]), 40: 5120}[heads], "heads": heads, "ctx": 4096}
        if c["mode"] == "decode":
            c.update(n=log_int(rng, 1, 15), past=log_int(rng, 16, 2048))
        elif c["mode"] == "prefill":
            c.update(n=log_int(rng, 17, 512), past=rng.choice([0, log_int(rng, 16, 2048)]))
        else:
            c.update(n=2 * rng.randint(2, 14) + 1, past=log_int(rng, 64, 3000))
        return c
    if kind == "head":
        return {"kind": kind, "type": rng.choice(["q8_0", "q6_k"]), "n": log_int(rng, 1, 16),
                "embd": 256 * rng.randint(4, 20), "vocab": rng.choice([32768, 151936]),
                "top_k": rng.choice([0, 0, rng.randint(1, 64), log_int(rng, 1, 1024)])}
    return {"kind": kind, "type": "q8_0", "layers": rng.randint(1, 3), "vocab": 16384, "prompt": log_int(rng, 16, 512),
            "gen": rng.randint(8, 48), "ctx": 1024}


# ---- inputs ----

def generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def normal(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


def activations(g, n, k):
    """A residual stream: N(0, 1) with a few channels several times larger."""
    x = normal(g, n, k)
    x[:, ::97] *= 6.0
    return x


def half_bytes(d):
    return d.to(torch.float16).view(torch.uint8).reshape(*d.shape, 2)


def quantize_weight(t, w):
    """GGUF rows of w [rows][cols] as uint8 [rows][row bytes], and the values they stand for in 64 bits (a function, so
    that only the check against 64-bit sums makes them)."""
    rows, cols = w.shape
    if t in ("f16", "bf16"):
        h = w.to(torch.float16 if t == "f16" else torch.bfloat16)
        return h.view(torch.uint8).reshape(rows, -1), lambda: h.double()
    if t == "q8_0":
        b = w.reshape(rows, cols // 32, 32)
        d = (b.abs().amax(-1) / 127).to(torch.float16)
        q = (b / d.float().clamp_min(1e-8)[..., None]).round().clamp(-127, 127).to(torch.int8)
        raw = torch.cat([half_bytes(d), q.view(torch.uint8)], -1).reshape(rows, -1)
        return raw, lambda: (q.double() * d.double()[..., None]).reshape(rows, cols)
    if t == "q6_k":
        b = w.reshape(rows, cols // 256, 16, 16)
        s = b.abs().amax(-1) / 31
        d = (s.amax(-1) / 127).to(torch.float16)
        sc = (s / d.float().clamp_min(1e-8)[..., None]).round().clamp(1, 127)
        q = (b / (d.float()[..., None] * sc).clamp_min(1e-9)[..., None]).round().clamp(-32, 31)
        u = (q + 32).to(torch.uint8).reshape(rows, cols // 256, 2, 4, 32)
        ql = torch.stack([u[..., 0, :] & 15 | (u[..., 2, :] & 15) << 4, u[..., 1, :] & 15 | (u[..., 3, :] & 15) << 4], -2)
        qh = u[..., 0, :] >> 4 | (u[..., 1, :] >> 4) << 2 | (u[..., 2, :] >> 4) << 4 | (u[..., 3, :] >> 4) << 6
        raw = torch.cat([ql.flatten(2), qh.flatten(2), sc.to(torch.int8).view(torch.uint8), half_bytes(d)], -1)
        return raw.reshape(rows, -1), \
            lambda: (q.double() * (d.double()[..., None] * sc.double())[..., None]).reshape(rows, cols)
    top = 15 if t == "q4_k" else 31
    b = w.reshape(rows, cols // 256, 8, 32)
    lo = b.amin(-1).clamp_max(0)
    s, m = (b.amax(-1) - lo) / top, -lo
    d, dmin = (s.amax(-1) / 63).to(torch.float16), (m.amax(-1) / 63).to(torch.float16)
    sc = (s / d.float().clamp_min(1e-8)[..., None]).round().clamp(1, 63)
    mn = (m / dmin.float().clamp_min(1e-8)[..., None]).round().clamp(0, 63)
    step, off = d.float()[..., None] * sc, dmin.float()[..., None] * mn
    u = ((b + off[..., None]) / step.clamp_min(1e-9)[..., None]).round().clamp(0, top).to(torch.uint8)
    a, z = sc.to(torch.uint8), mn.to(torch.uint8)
    scales = torch.cat([a[..., :4] | (a[..., 4:] >> 4) << 6, z[..., :4] | (z[..., 4:] >> 4) << 6,
                        a[..., 4:] & 15 | (z[..., 4:] & 15) << 4], -1)
    pair = u.reshape(rows, cols // 256, 4, 2, 32)
    qs = (pair[..., 0, :] & 15 | (pair[..., 1, :] & 15) << 4).flatten(2)
    parts = [half_bytes(d), half_bytes(dmin), scales]
    if t == "q5_k":
        bits = torch.arange(8, device=w.device, dtype=torch.uint8)[:, None]
        parts.append(((u >> 4) << bits).sum(-2).to(torch.uint8))
    raw = torch.cat(parts + [qs], -1).reshape(rows, -1)
    return raw, lambda: (u.double() * (d.double()[..., None] * sc.double())[..., None]
                         - (dmin.double()[..., None] * mn.double())[..., None]).reshape(rows, cols)


_ctx = None


def context():
    """The program's one library context."""
    global _ctx
    if _ctx is None:
        _ctx = mk.Context(0)
    return _ctx


class Weight:
    """One matrix as the program holds it after loading: packed (Q8_0, Q4_K, Q6_K), or its GGUF rows."""

    def __init__(self, t, raw, cols):
        self.type, self.rows, self.cols, self.row_bytes = TYPES[t], raw.shape[0], cols, raw.shape[1]
        self.packed = t in ("q8_0", "q4_k", "q6_k")
        self.data = raw
        if self.packed:
            L, ctx = mk.load(), context()
            self.data = torch.empty(L.mk_packed_bytes(self.type, self.rows, cols), dtype=torch.uint8, device="cuda")
            torch.cuda.synchronize()  # the library packs on its own stream
            mk.check(L.mk_pack_weight(ctx.h, self.type, raw.data_ptr(), self.row_bytes, self.rows, cols,
                                      self.data.data_ptr()))
            ctx.sync()
            self.w = mk.MkWeight(self.type, 1, self.rows, cols, self.data.data_ptr())


def interleave4(gate, up):
    """Rows of gate and up interleaved by 4 (include/malkin_hip.h, silu_pairs)."""
    return torch.stack([gate.reshape(-1, 4, gate.shape[1]), up.reshape(-1, 4, up.shape[1])], 1).reshape(-1, gate.shape[1])


def f32(*shape):
    return torch.zeros(*shape, device="cuda")


def q8_rows(n, k):
    return torch.zeros(n, k // 32 * 40, dtype=torch.uint8, device="cuda")


def i32(v):
    return torch.tensor(v, dtype=torch.int32, device="cuda")


def mlp_inputs(c, seed):
    g = generator(seed)
    E, F = c["embd"], c["ff"]
    x, norm = activations(g, c["n"], E), torch.rand(E, generator=g, device="cuda") + 0.5
    return x, norm, [quantize_weight(c["type"], normal(g, r, k) * 0.02) for r, k in ((F, E), (F, E), (E, F))]


def tree_parents(n):
    """[next, chain0, alt0, chain1, alt1, ...]: a draft and its alternative share a parent, the draft before."""
    return [-1] + [max(0, 2 * ((t - 1) // 2) - 1) for t in range(1, n)]


def attn_layout(c):
    """Per token: RoPE position, sequence, KV row, plain keys and the ancestors' rows."""
    n, past = c["n"], c["past"]
    if c["mode"] == "decode":  # sequences of past/4 .. past keys, spread evenly
        pos = [past - (3 * past // 4) * t // max(1, n - 1) for t in range(n)]
        return pos, list(range(n)), pos, [p + 1 for p in pos], [[] for _ in pos]
    if c["mode"] == "prefill":
        pos = [past + t for t in range(n)]
        return pos, [0] * n, pos, [p + 1 for p in pos], [[] for _ in pos]
    parent, pos, anc = tree_parents(n), [past], [[]]
    for t in range(1, n):
        pos.append(pos[parent[t]] + 1)
        anc.append(anc[parent[t]] + [past + t])
    return pos, [0] * n, [past + t for t in range(n)], [past + 1] * n, anc


def attn_inputs(c, seed):
    g = generator(seed)
    E, H, KV, ctx = c["embd"], c["heads"], 8, c["ctx"]
    n_seq = c["n"] if c["mode"] == "decode" else 1
    i = {"x": activations(g, c["n"], E), "norm": torch.rand(E, generator=g, device="cuda") + 0.5,
         "qn": torch.rand(D, generator=g, device="cuda") + 0.5, "kn": torch.rand(D, generator=g, device="cuda") + 0.5}
    i["qkv"] = quantize_weight(c["type"], normal(g, (H + 2 * KV) * D, E) * 0.02)
    i["wo"] = quantize_weight(c["type"], normal(g, E, H * D) * 0.02)
    for s in ("k", "v"):
        v = normal(g, 1, n_seq, KV, ctx, D)
        i[s + "s"] = v.abs().amax(-1) / 127
        i[s] = (v / i[s + "s"][..., None]).round().to(torch.int8)
    ang = torch.arange(ctx, dtype=torch.float64)[:, None] * ROPE_BASE ** (-torch.arange(0, D, 2, dtype=torch.float64) / D)
    i["cos"], i["sin"] = ang.cos().float().cuda(), ang.sin().float().cuda()
    return i


def head_inputs(c, seed):
    g = generator(seed)
    x, norm = activations(g, c["n"], c["embd"]), torch.rand(c["embd"], generator=g, device="cuda") + 0.5
    return x, norm, quantize_weight(c["type"], normal(g, c["vocab"], c["embd"]) * 0.02)


class State:
    """The calls of one pass (function, arguments), its outputs, and what they refer to."""

    def __init__(self, *keep):
        self.calls, self.out, self.keep = [], {}, list(keep)

    def call(self, name, *args):
        self.calls.append((getattr(mk.load(), name),
                           tuple(a.data_ptr() if isinstance(a, torch.Tensor) else a for a in args)))
        self.keep.append(args)


def matmul(s, ctx, w, xf, x_stride, xq, n, y):
    """One matmul the way the weight's type takes it, from fp32 rows or their BlockQ8 rows."""
    if w.packed:
        s.call("mk_matmul", ctx.h, ctypes.byref(w.w), xq, n, y, w.rows, 0)
    elif w.type == mk.Q5_K:
        s.call("mk_matmul_gguf", ctx.h, w.type, w.data, w.row_bytes, w.rows, w.cols, xq, n, y, w.rows, 0)
    else:
        s.call("mk_matmul_rows", ctx.h, w.type, w.data, w.row_bytes, w.rows, w.cols, xf, x_stride, None, n, y, w.rows, 0)
    s.keep.append(w)


def fused(w, n, norm):
    """Whether the decode step's fused matmul takes this weight (include/malkin_hip.h, mk_matmul_f32)."""
    return w.packed and n <= 2 and (not norm or w.cols <= 8192)


def prepare_mlp(c, seed):
    x, norm, ws = mlp_inputs(c, seed)
    n, E, F, ctx = c["n"], c["embd"], c["ff"], context()
    gate, up, down = (raw for raw, _ in ws)
    packed = c["type"] in ("q8_0", "q4_k", "q6_k")
    wg, wd = Weight(c["type"], interleave4(gate, up) if packed else torch.cat([gate, up]), E), Weight(c["type"], down, F)
    gu, y, xq, hq = f32(n, 2 * F), f32(n, E), q8_rows(n, E), q8_rows(n, F)
    s = State(wg, wd)
    if fused(wg, n, True):
        s.call("mk_matmul_f32", ctx.h, ctypes.byref(wg.w), x, E, norm, EPS, n, gu, F, 0, 1)
        s.call("mk_matmul_f32", ctx.h, ctypes.byref(wd.w), gu, F, None, 0.0, n, y, E, 0, 0)
    elif c["type"] in ("f16", "bf16"):
        h = f32(n, E)
        s.call("mk_rmsnorm_rows", ctx.h, x, None, norm, n, E, EPS, h)
        matmul(s, ctx, wg, h, E, None, n, gu)
        s.call("mk_silu_mul_rows", ctx.h, gu, n, F)
        matmul(s, ctx, wd, gu, 2 * F, None, n, y)
    else:
        s.call("mk_rmsnorm_q8", ctx.h, x, None, norm, n, E, EPS, xq)
        matmul(s, ctx, wg, None, 0, xq, n, gu)
        s.call("mk_silu_mul_q8", ctx.h, gu, n, F, 1 if packed else 0, hq)
        matmul(s, ctx, wd, None, 0, hq, n, y)
    s.out = {"y": y}
    return s


def prepare_attn(c, seed):
    i, ctx = attn_inputs(c, seed), context()
    n, E, H, KV = c["n"], c["embd"], c["heads"], 8
    QKV, HD = (H + 2 * KV) * D, H * D
    wq, wo = Weight(c["type"], i["qkv"][0], E), Weight(c["type"], i["wo"][0], HD)
    rpos, seq, rows, keys, anc = attn_layout(c)
    off = [sum(len(a) for a in anc[:t]) for t in range(n + 1)]
    d_pos, d_seq, d_row, d_key = i32(rpos), i32(seq), i32(rows), i32(keys)
    tree = c["mode"] == "tree"
    d_off, d_anc = i32(off), i32([r for a in anc for r in a] + [0])
    kv = mk.MkKvCache(i["k"].data_ptr(), i["v"].data_ptr(), i["ks"].data_ptr(), i["vs"].data_ptr(), 1, i["k"].shape[1],
                      KV, D, c["ctx"])
    kvp = ctypes.byref(kv)
    most = max(k + len(a) for k, a in zip(keys, anc))
    qkv, att, y, xq, aq = f32(n, QKV), f32(n, HD), f32(n, E), q8_rows(n, E), q8_rows(n, HD)
    s = State(i, wq, wo, kv, d_off, d_anc)
    f = fused(wq, n, True)
    if f:
        s.call("mk_matmul_f32", ctx.h, ctypes.byref(wq.w), i["x"], E, i["norm"], EPS, n, qkv, QKV, 0, 0)
    else:
        s.call("mk_rmsnorm_q8", ctx.h, i["x"], None, i["norm"], n, E, EPS, xq)
        matmul(s, ctx, wq, None, 0, xq, n, qkv)
    lib, done = mk.load(), False
    if c["mode"] == "decode":  # one launch where the library has it, two otherwise, as the model's forward chooses
        args = (ctx.h, qkv, QKV, n, H, i["qn"], i["kn"], EPS, i["cos"], i["sin"], d_pos, d_seq, d_row, d_key, kvp, 0,
                att, HD, most)
        name = "mk_attention_decode" if f else "mk_attention_decode_q8"
        args += () if f else (aq,)
        torch.cuda.synchronize()
        rc = getattr(lib, name)(*(a.data_ptr() if isinstance(a, torch.Tensor) else a for a in args))
        done = rc != mk.MK_ERR_UNSUPPORTED
        if done:
            mk.check(rc)
            s.call(name, *args)
    if not done:
        base = qkv.data_ptr()
        s.call("mk_qk_norm_rope_kv", ctx.h, qkv, base + 4 * HD, base + 4 * (HD + KV * D), QKV, n, H, i["qn"], i["kn"],
               EPS, i["cos"], i["sin"], d_pos, d_seq, d_row, kvp, 0)
        args = (ctx.h, qkv, QKV, att, HD, n, H, kvp, 0, d_seq, d_key, d_off if tree else None, d_anc if tree else None,
                most)
        s.call("mk_attention" if f else "mk_attention_q8", *(args + (() if f else (aq,))))
    if f:
        s.call("mk_matmul_f32", ctx.h, ctypes.byref(wo.w), att, HD, None, 0.0, n, y, E, 0, 0)
    else:
        matmul(s, ctx, wo, None, 0, aq, n, y)
    s.out = {"y": y, "k": i["k"], "v": i["v"], "ks": i["ks"], "vs": i["vs"]}
    return s


def prepare_head(c, seed):
    x, norm, (raw, _) = head_inputs(c, seed)
    n, E, V, k, ctx = c["n"], c["embd"], c["vocab"], c["top_k"], context()
    w = Weight(c["type"], raw, E)
    xq, logits = q8_rows(n, E), f32(n, V)
    s = State(w)
    s.call("mk_rmsnorm_q8", ctx.h, x, None, norm, n, E, EPS, xq)
    matmul(s, ctx, w, None, 0, xq, n, logits)
    if k:
        vals, ids = f32(n, k), torch.zeros(n, k, dtype=torch.int32, device="cuda")
        s.call("mk_topk", ctx.h, logits, V, None, n, V, k, vals, ids)
        s.out = {"logits": logits, "values": vals, "ids": ids}
    else:
        t1, t2 = (torch.zeros(n, dtype=torch.int32, device="cuda") for _ in range(2))
        s.call("mk_argmax_top2", ctx.h, logits, n, V, t1, t2)
        s.out = {"logits": logits, "top1": t1, "top2": t2}
    return s


def prepare_generate(c, seed):
    from malkin_amd import synth
    cfg = synth.make_config("qwen3-8b", TYPES[c["type"]], seed=int(seed), n_layer=c["layers"], n_vocab=c["vocab"])
    d = "/dev/shm" if os.path.isdir("/dev/shm") and os.access("/dev/shm", os.W_OK) else None
    with tempfile.TemporaryDirectory(dir=d) as tmp:
        path = os.path.join(tmp, "model.gguf")
        synth.write_gguf(path, cfg)
        m = mk.Model(context(), path, c["ctx"])
    rng = np.random.default_rng(int(seed))
    return m, rng.integers(0, c["vocab"], c["prompt"]).astype(np.int32), c["gen"]


PREPARE = {"mlp": prepare_mlp, "attn": prepare_attn, "head": prepare_head, "generate": prepare_generate}


def prepare(case, seed):
    s = PREPARE[case["kind"]](case, seed)
    torch.cuda.synchronize()  # inputs made on torch's stream; the library works on its own
    return s


def run(state):
    if isinstance(state, State):
        for f, args in state.calls:
            rc = f(*args)
            if rc:
                mk.check(rc)
        return state.out
    m, prompt, gen = state
    toks, _ = m.generate(prompt, gen)
    return {"tokens": toks, "logits": m.forward(toks[-1:], len(prompt) + gen - 1)}


# ---- what a pass cannot do without ----

def weight_bytes(t, rows, cols):
    qk, size = BLOCK[t]
    return rows * cols // qk * size


def layer_work(t, n, E, H, KV, F, keys, kv_rows):
    """Bytes and operations of a layer's attention half and MLP half: (attention, MLP)."""
    QKV, HD = (H + 2 * KV) * D, H * D
    attn = {"bytes": weight_bytes(t, QKV, E) + weight_bytes(t, E, HD) + 8 * n * E + (kv_rows + n) * 2 * KV * (D + 4),
            "flops": 2 * n * (QKV * E + E * HD) + 4 * HD * keys}
    mlp = {"bytes": 3 * weight_bytes(t, F, E) + 8 * n * E + 4 * E, "flops": 6 * n * E * F}
    return attn, mlp


def work(case):
    c = case
    if c["kind"] == "mlp":
        return layer_work(c["type"], c["n"], c["embd"], 8, 8, c["ff"], 0, 0)[1]
    if c["kind"] == "attn":
        _, _, _, keys, anc = attn_layout(c)
        rows = sum(keys) - c["n"] if c["mode"] == "decode" else c["past"]
        return layer_work(c["type"], c["n"], c["embd"], c["heads"], 8, 256, sum(keys) + sum(map(len, anc)), rows)[0]
    if c["kind"] == "head":
        w = weight_bytes(c["type"], c["vocab"], c["embd"])
        return {"bytes": w + 4 * c["n"] * (c["embd"] + c["vocab"] + 2 * max(1, c["top_k"])),
                "flops": 2 * c["n"] * c["vocab"] * c["embd"]}
    E, F, H, KV, p, total = 4096, 12288, 32, 8, c["prompt"], {"bytes": 0, "flops": 0}
    for n, keys, rows in [(p, p * (p + 1) // 2, 0)] + [(1, p + i, p + i) for i in range(c["gen"])]:
        for half in layer_work(c["type"], n, E, H, KV, F, keys, rows):
            for k in total:
                total[k] += c["layers"] * half[k]
        total["bytes"] += weight_bytes(c["type"], c["vocab"], E) + 4 * c["vocab"]
        total["flops"] += 2 * c["vocab"] * E
    return total


def tolerance(case):
    # An fp32 sum in another order moves an output by some 1e-7; where it lands on the other side of a rounding to the
    # 8-bit activations or keys and values that the next step reads, that input moves by a whole step, which is what
    # shows. Each is about four times what `exact` differs by (mlp 3e-4, attention 1.3e-3, unquantized rows 4e-7).
    if case["kind"] == "head":
        return {"rel": 1e-4, "max": 5e-3, "differ": 0.002}
    if case["kind"] == "generate":
        return {"rel": 1e-2, "max": 0.2, "differ": 0.0}
    if case["kind"] == "attn":
        return {"rel": 5e-3, "max": 0.1, "differ": 1e-3}
    if case["type"] in ("f16", "bf16"):
        return {"rel": 2e-6, "max": 2e-5}
    return {"rel": 1.2e-3, "max": 5e-2}


# ---- the same results in 64 bits ----

def rms64(x, w):
    x = x.double()
    return x / (x.square().mean(-1, keepdim=True) + EPS).sqrt() * w.double()


def q8_64(x):
    """The values of x after the 8-bit rounding of activations (blocks of 32, amax / 127 steps)."""
    b = x.reshape(*x.shape[:-1], -1, 32)
    d = b.abs().amax(-1, keepdim=True) / 127
    return torch.where(d > 0, (b / d.clamp_min(1e-300)).round() * d, 0.0).reshape(x.shape)


def exact_mlp(c, seed):
    x, norm, ws = mlp_inputs(c, seed)
    gate, up, down = (v() for _, v in ws)
    act = (lambda v: v) if c["type"] in ("f16", "bf16") else q8_64
    h = act(rms64(x, norm))
    g = h @ gate.T
    return {"y": act(g / (1 + (-g).exp()) * (h @ up.T)) @ down.T}


def exact_attn(c, seed):
    i, n, H, KV, ctx = attn_inputs(c, seed), c["n"], c["heads"], 8, c["ctx"]
    rpos, seq, rows, keys, anc = attn_layout(c)
    qkv = (q8_64(rms64(i["x"], i["norm"])) @ i["qkv"][1]().T).reshape(n, H + 2 * KV, D)
    cos, sin = i["cos"][rpos].double()[:, None], i["sin"][rpos].double()[:, None]

    def rope(v, w):
        a, b = rms64(v, w).chunk(2, -1)
        return torch.cat([a * cos - b * sin, a * sin + b * cos], -1)

    def rows8(v):
        d = v.abs().amax(-1, keepdim=True) / 127
        return (v / d).round() * d

    q = rope(qkv[:, :H], i["qn"])
    k_new, v_new = rows8(rope(qkv[:, H:H + KV], i["kn"])), rows8(qkv[:, H + KV:])
    # Cached key rows hold element e at byte 8 * (e % 16) + e / 16.
    back = torch.arange(D, device="cuda")
    back = 8 * (back % 16) + back // 16
    k = i["k"][0].double()[..., back] * i["ks"][0].double()[..., None]
    v = i["v"][0].double() * i["vs"][0].double()[..., None]
    att = torch.zeros(n, H, D, dtype=torch.float64, device="cuda")
    for t in range(n):
        k[seq[t], :, rows[t]], v[seq[t], :, rows[t]] = k_new[t], v_new[t]
    for t in range(n):
        at = list(range(keys[t])) + anc[t]
        kt, vt = k[seq[t]][:, at], v[seq[t]][:, at]
        p = torch.softmax(q[t].reshape(KV, H // KV, D) @ kt.transpose(1, 2).contiguous() / math.sqrt(D), -1)
        att[t] = (p @ vt).reshape(H, D)
    return {"y": q8_64(att.reshape(n, H * D)) @ i["wo"][1]().T, "k": None, "v": None, "ks": None, "vs": None}


def exact_head(c, seed):
    x, norm, (_, w) = head_inputs(c, seed)
    logits = q8_64(rms64(x, norm)) @ w().T
    out = {"logits": logits}
    if c["top_k"]:
        out["values"] = logits.topk(c["top_k"]).values
    return out


def exact(case, seed):
    """A whole model's tokens feed back into its inputs, so `generate` has no 64-bit counterpart."""
    f = {"mlp": exact_mlp, "attn": exact_attn, "head": exact_head}.get(case["kind"])
    return f(case, seed) if f else None
