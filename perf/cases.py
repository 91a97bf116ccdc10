"""The work that users of this library have it do, as cases that can be timed and checked.

A case is a dict of plain values; `prepare` makes what a program holds before
the call (inputs, weights, engine), `run` is one pass through the public entry
points, `exact` the same answer in 64-bit torch without the library.

Kinds
  linear   activation rows -> one W8A8 linear (brain_amd.ops): decode rows
           through linear_i8, bf16 prompt rows through quantize_rows_bf16 +
           matmul_i8
  w4a8     the same with int4 weights (ops.matmul_q4)
  dit      the int8 linears of DiT blocks, bf16 between them (brain_amd.dit)
  moe      one sparse-MoE projection: every expert's gated linear over the
           tokens of a batch (ops.moe_linear_gated_i8)
  paged    one decode step of attention over the int8 paged KV cache: append
           the new token, scores, softmax, weighted values (the C ABI's
           bh_paged_* calls; the softmax is torch's, as the library has none)
  prefill  the Qwen3-0.6B engine on whole prompts: next tokens and logits
  generate the engine's prompt + greedy decode: all tokens and final logits
"""
import math

import numpy as np
import torch

from brain_amd import load, ops
from brain_amd._lib import check
from brain_amd.dit import DIT_D, DIT_FF, DIT_QKV, DitInt8Stack
from brain_amd.qwen3 import QWEN3_0_6B, Qwen3Engine

# The hidden size, MLP size, head counts and vocabulary of the Qwen3-0.6B
# configuration and the (K, N) pairs of the decode and prefill sweeps in
# bench.py are where the sizes below come from; the ragged ones are generic.


def listed():
    return [
        # One projection of a single-sequence decode step: launch and latency.
        dict(name="linear_decode_m1", kind="linear", m=1, k=1024, n=3072, dtype="f32", bias=False),
        # The vocabulary projection of 8 decoding sequences.
        dict(name="linear_head_m8", kind="linear", m=8, k=1024, n=151936, dtype="f32", bias=False),
        # A generic layer whose sizes are no multiple of any tile, with bias.
        dict(name="linear_ragged", kind="linear", m=333, k=2900, n=1111, dtype="f32", bias=True),
        # Attention projection of a 2048-token prompt, bf16 activations.
        dict(name="linear_prompt_2048", kind="linear", m=2048, k=4096, n=4096, dtype="bf16", bias=False),
        # MLP projection of a long batch of prompts: the largest GEMM.
        dict(name="linear_prompt_8192", kind="linear", m=8192, k=4096, n=11008, dtype="bf16", bias=False),
        # Two DiT blocks' int8 linears at 1024 image patches + 128 text tokens.
        dict(name="dit_blocks", kind="dit", m=1152, layers=2),
        # int4 weights in a decode step of 8 sequences.
        dict(name="w4a8_decode_m8", kind="w4a8", m=8, k=3072, n=1024),
        # int4 weights on a 512-token prompt.
        dict(name="w4a8_prompt_512", kind="w4a8", m=512, k=4096, n=11008),
        # 8 experts, 2 of them for each of 2048 tokens.
        dict(name="moe_experts", kind="moe", m=2048, k=1024, n=3072, experts=8, top=2),
        # One decode step's attention of 8 sequences of up to 2048 tokens.
        dict(name="paged_attention", kind="paged", batch=8, ctx=2048, heads=16, kv_heads=8, head_dim=128, block=32),
        # A 2000-token prompt through the whole model, int8 KV cache.
        dict(name="qwen3_prefill", kind="prefill", batch=1, prompt=2000, kv_int8=True),
        # A chat turn of 8 sequences: 128-token prompts, 64 new tokens each.
        dict(name="qwen3_generate", kind="generate", batch=8, prompt=128, steps=64, kv_int8=False),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "w4a8", "w4a8", "dit", "moe", "paged", "prefill", "generate"])
    if kind == "linear":
        m = _log(rng, 1, 8192)
        if rng.random() < 0.3 and m > 64:
            m = m // 64 * 64
        if rng.random() < 0.6:
            k, n = rng.choice([(1024, 3072), (3072, 1024), (1024, 4096), (2048, 1024), (4096, 4096), (4096, 11008)])
        else:
            k, n = 4 * _log(rng, 64, 2700), _log(rng, 256, 11008)
        dtype = "f32" if m <= 32 else rng.choice(["f32", "bf16"])
        return dict(kind=kind, m=m, k=k, n=n, dtype=dtype, bias=rng.random() < 0.3)
    if kind == "w4a8":
        m = _log(rng, 1, 2048)
        if rng.random() < 0.7:
            k, n = rng.choice([(1024, 3072), (3072, 1024), (4096, 4096), (4096, 11008)])
        else:
            k, n = 8 * _log(rng, 32, 1375), _log(rng, 256, 11008)
        return dict(kind=kind, m=m, k=k, n=n)
    if kind == "dit":
        return dict(kind=kind, m=_log(rng, 128, 1152), layers=rng.choice([1, 2]))
    if kind == "moe":
        return dict(kind=kind, m=_log(rng, 1, 2048), k=rng.choice([512, 1024, 2048]),
                    n=rng.choice([768, 1000, 1536, 3072]), experts=rng.choice([4, 8]), top=rng.choice([1, 2]))
    if kind == "paged":
        heads, kv_heads, head_dim = rng.choice([(16, 8, 128), (16, 8, 128), (32, 8, 128), (8, 8, 64)])
        return dict(kind=kind, batch=_log(rng, 1, 16), ctx=_log(rng, 32, 2048), heads=heads, kv_heads=kv_heads,
                    head_dim=head_dim, block=rng.choice([16, 32]))
    kv = rng.random() < 0.5
    if kind == "prefill":
        batch = _log(rng, 1, 8)
        return dict(kind=kind, batch=batch, prompt=_log(rng, 16, 2000 // batch), kv_int8=kv)
    return dict(kind=kind, batch=_log(rng, 1, 8), prompt=_log(rng, 4, 128), steps=_log(rng, 8, 64), kv_int8=kv)


def _gen(seed, salt=0):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 1000003 + salt)
    return g


def _randn(g, *shape):
    return torch.randn(*shape, device="cuda", generator=g)


def _weights(g, n, k, top=127):
    """Normal weights with one scale per output row, as a quantized layer of variance 1/k has them."""
    w = _randn(g, n, k) / k ** 0.5
    scale = w.abs().amax(1).clamp_min(1e-8) / top
    return (w / scale[:, None]).round().clamp(-top, top).to(torch.int8), scale


def _pack8(q):
    return q.contiguous().view(torch.int32)


def _pack4(q):
    """int4 codes [n, k] -> words [n, k/8], element b of a word in bits 4b."""
    v = (q.to(torch.int32) & 15).view(q.shape[0], -1, 8)
    out = torch.zeros(v.shape[:2], device=q.device, dtype=torch.int32)
    for b in range(8):
        out |= v[:, :, b] << (4 * b)
    return out


def _acts(g, m, k):
    """Activation rows: normal, with a few larger channels as trained models have."""
    x = _randn(g, m, k)
    x[:, ::61] *= 6.0
    return x


# ------------------------------------------------------------------ one linear


def _linear_inputs(c, seed):
    g = _gen(seed)
    x = _acts(g, c["m"], c["k"])
    q, sw = _weights(g, c["n"], c["k"], 7 if c["kind"] == "w4a8" else 127)
    bias = _randn(g, c["n"]) if c.get("bias") else None
    return (x.to(torch.bfloat16) if c.get("dtype") == "bf16" else x), q, sw, bias


def _run_linear(s):
    if s["x"].dtype == torch.bfloat16:
        sx, xq = ops.quantize_rows_bf16(s["x"])
        return ops.matmul_i8(xq, s["w"], sx, s["sw"], s["bias"], torch.bfloat16)
    return ops.linear_i8(s["x"], s["w"], s["sw"], s["bias"])


def _run_w4a8(s):
    sx, xq = ops.quantize_rows(s["x"])
    return ops.matmul_q4(xq, s["w"], sx, s["sw"])


def _quant64(x):
    """64-bit per-row int8 codes (as float64) and scales."""
    sx = x.abs().amax(1).clamp_min(1e-8) / 127
    return (x / sx[:, None]).round().clamp(-127, 127), sx


def _lin64(x, q, sw, bias=None):
    xq, sx = _quant64(x)
    out = (xq @ q.double().t()) * sx[:, None] * sw.double()
    return out if bias is None else out + bias.double()


# ------------------------------------------------------------------ MoE


def _moe_inputs(c, seed):
    g = _gen(seed)
    x = _acts(g, c["m"], c["k"])
    w = [_weights(g, c["n"], c["k"]) for _ in range(c["experts"])]
    p = torch.softmax(_randn(g, c["m"], c["experts"]), 1)
    keep = torch.zeros_like(p).scatter_(1, p.topk(c["top"], 1).indices, 1.0)
    return x, w, (p * keep).contiguous()


def _run_moe(s):
    sx, xq = ops.quantize_rows(s["x"])
    return [ops.moe_linear_gated_i8(xq, w, sx, sw, s["gate"], e) for e, (w, sw) in enumerate(s["w"])]


# ------------------------------------------------------------------ paged attention


def _paged_inputs(c, seed):
    g = _gen(seed)
    b, bs, kvd = c["batch"], c["block"], c["kv_heads"] * c["head_dim"]
    lens = torch.randint(max(1, c["ctx"] // 2), c["ctx"] + 1, (b,), device="cuda", generator=g)
    lens[0] = c["ctx"]
    max_bt = (c["ctx"] + bs - 1) // bs
    nblk = b * max_bt
    table = torch.randperm(nblk, device="cuda", generator=g).to(torch.int32).view(b, max_bt)
    st = dict(lens=lens.to(torch.int32), table=table, q=_randn(g, b, c["heads"], c["head_dim"]))
    for which in "kv":
        st[which + "new"] = _randn(g, b, kvd)
        st[which + "pool"] = torch.randint(-127, 128, (nblk * bs, kvd), device="cuda", generator=g, dtype=torch.int8)
        st[which + "scale"] = (torch.rand(nblk * bs, c["kv_heads"], device="cuda", generator=g) + 0.5) / 40
    last = (lens - 1).to(torch.int64)
    st["blk"] = table.gather(1, (last // bs)[:, None]).view(-1).contiguous()
    st["off"] = (last % bs).to(torch.int32)
    return st


def _prepare_paged(c, seed):
    s = _paged_inputs(c, seed)
    s["clip"] = torch.full((c["kv_heads"],), 3.0e38, device="cuda")
    # Positions past a sequence's length are never written: they stay -inf for the softmax.
    s["scores"] = torch.full((c["batch"], c["heads"], c["ctx"]), -math.inf, device="cuda")
    s["ctx"] = torch.empty(c["batch"], c["heads"], c["head_dim"], device="cuda")
    s["c"] = c
    return s


def _run_paged(s):
    c, lib = s["c"], load()
    st = torch.cuda.current_stream().cuda_stream
    kvd = c["kv_heads"] * c["head_dim"]
    for w in "kv":
        check(lib.bh_paged_kv_append_i8(st, s[w + "new"].data_ptr(), s["blk"].data_ptr(), s["off"].data_ptr(),
                                        s["clip"].data_ptr(), s[w + "pool"].data_ptr(), s[w + "pool"].numel() // 4,
                                        s[w + "scale"].data_ptr(), s[w + "scale"].numel(), c["batch"], kvd, c["block"],
                                        c["head_dim"]))
    shape = (c["batch"], c["heads"], c["heads"] // c["kv_heads"], c["head_dim"], c["block"], kvd, c["ctx"],
             s["table"].shape[1])
    check(lib.bh_paged_decode_scores_i8(st, s["q"].data_ptr(), s["kpool"].data_ptr(), s["kpool"].numel() // 4,
                                        s["table"].data_ptr(), s["lens"].data_ptr(), s["kscale"].data_ptr(),
                                        s["kscale"].numel(), s["scores"].data_ptr(), *shape, c["head_dim"] ** -0.5))
    probs = torch.softmax(s["scores"], -1)
    check(lib.bh_paged_decode_apply_i8(st, probs.data_ptr(), s["vpool"].data_ptr(), s["vpool"].numel() // 4,
                                       s["table"].data_ptr(), s["lens"].data_ptr(), s["vscale"].data_ptr(),
                                       s["vscale"].numel(), s["ctx"].data_ptr(), *shape))
    return [s["scores"], s["ctx"], s["kpool"], s["vpool"], s["kscale"], s["vscale"]]


def _exact_paged(c, seed):
    s = _paged_inputs(c, seed)
    b, nkv, hd, bs, ctx = c["batch"], c["kv_heads"], c["head_dim"], c["block"], c["ctx"]
    slot = (s["blk"].long() * bs + s["off"].long())
    full = {}
    for w in "kv":
        x = s[w + "new"].double().view(b, nkv, hd)
        scale = x.abs().amax(2) / 127
        pool, sc = s[w + "pool"].double().view(-1, nkv, hd), s[w + "scale"].double()
        pool[slot] = (x / scale[:, :, None]).round().clamp(-127, 127)
        sc[slot] = scale
        full[w] = (pool * sc[:, :, None], sc)
    at = torch.arange(ctx, device="cuda")
    rows = s["table"].long()[:, at // bs] * bs + at % bs
    group = c["heads"] // nkv
    k = full["k"][0][rows].repeat_interleave(group, 2)
    v = full["v"][0][rows].repeat_interleave(group, 2)
    sco = torch.einsum("bhd,bjhd->bhj", s["q"].double(), k) * hd ** -0.5
    sco.masked_fill_(at[None, None, :] >= s["lens"][:, None, None], -math.inf)
    out = torch.einsum("bhj,bjhd->bhd", torch.softmax(sco, -1), v)
    return [sco, out, None, None, full["k"][1], full["v"][1]]


# ------------------------------------------------------------------ DiT blocks


def _run_dit(s):
    s.x.copy_(s.x0)
    s.step()
    return [s.x, s.qkv, s.o, s.h]


def _exact_dit(c, seed):
    s = DitInt8Stack(layers=c["layers"], m=c["m"], seed=seed)  # for its weights and input only
    half = lambda t: t.to(torch.bfloat16).double()  # noqa: E731
    x = s.x0.double()
    for lw in s.w:
        lin = lambda t, name: half(_lin64(t, lw[name][0].view(torch.int8), lw[name][1]))  # noqa: E731
        qkv, o = lin(x, "qkv"), lin(x, "o")
        h = lin(o, "w1")
        x = lin(h, "w2")
    return [x, qkv, o, h]


# ------------------------------------------------------------------ Qwen3 engine


def _qwen3_weights(seed):
    """Weights of the 0.6B configuration in the scale of its initialisation;
    the embedding is larger, so that the greedy choice has the margin of a
    trained model and not the near ties of a random one."""
    c = QWEN3_0_6B
    d, hq, hkv, ff = c["d_model"], c["n_heads"] * c["head_dim"], c["n_kv_heads"] * c["head_dim"], c["d_ff"]
    down = 0.02 / (2 * c["n_layers"]) ** 0.5
    shapes = [("attn.wq", hq, d, 0.02), ("attn.wk", hkv, d, 0.02), ("attn.wv", hkv, d, 0.02), ("attn.wo", d, hq, down),
              ("mlp.gate", ff, d, 0.02), ("mlp.up", ff, d, 0.02), ("mlp.down", d, ff, down)]
    layers = []
    for i in range(c["n_layers"]):
        g = _gen(seed, 1 + i)
        w = {}
        for name, n, k, std in shapes:
            q, s = _weights(g, n, k)
            w[name] = (q, s * (std * k ** 0.5))
        layers.append(w)
    return layers, _randn(_gen(seed, 99), c["vocab"], d) * 0.4


def _prompts(c, seed):
    g = _gen(seed, 500)
    return torch.randint(0, QWEN3_0_6B["vocab"], (c["batch"], c["prompt"]), device="cuda", generator=g)


def _prepare_qwen3(c, seed):
    cfg = dict(QWEN3_0_6B, kv_int8=int(c["kv_int8"]))
    eng = Qwen3Engine(cfg, c["batch"], c["prompt"] + c.get("steps", 0))
    layers, emb = _qwen3_weights(seed)
    eng.set_weight("tok.weight", emb.cpu().numpy())
    ones = np.ones(cfg["d_model"], np.float32)
    eng.set_weight("norm.weight", ones)
    for i, w in enumerate(layers):
        for name, (q, s) in w.items():
            eng.set_weight_i8(f"blocks.{i}.{name}.weight", q.cpu().numpy().view(np.uint32), s.cpu().numpy())
        for name in ("ln1", "ln2"):
            eng.set_weight(f"blocks.{i}.{name}.weight", ones)
        for name in ("q_norm", "k_norm"):
            eng.set_weight(f"blocks.{i}.attn.{name}.weight", ones[: cfg["head_dim"]])
    return dict(c=c, eng=eng, prompts=_prompts(c, seed).cpu().numpy().astype(np.uint32))


def _run_prefill(s):
    nxt = s["eng"].prefill(s["prompts"])
    return [nxt.astype(np.int64), s["eng"].logits()]


def _run_generate(s):
    toks = s["eng"].generate(s["prompts"], s["c"]["steps"])
    return [toks.astype(np.int64), s["eng"].logits()]


def _exact_qwen3(c, seed):
    cfg = QWEN3_0_6B
    nh, nkv, hd, eps = cfg["n_heads"], cfg["n_kv_heads"], cfg["head_dim"], cfg["rms_eps"]
    layers, emb = _qwen3_weights(seed)
    hs = emb.abs().amax(1).clamp_min(1e-8) / 127
    head = (emb / hs[:, None]).round().clamp(-127, 127)
    freq = cfg["rope_theta"] ** (-torch.arange(0, hd, 2, device="cuda", dtype=torch.float64) / hd)
    rms = lambda x: x / (x.square().mean(-1, keepdim=True) + eps).sqrt()  # noqa: E731
    b = c["batch"]
    cache = [None] * len(layers)

    def forward(tok, pos0):
        t = tok.shape[1]
        x = emb.double()[tok].view(b * t, -1)
        ang = torch.arange(pos0, pos0 + t, device="cuda", dtype=torch.float64)[:, None] * freq
        cos, sin = ang.cos()[None, :, None], ang.sin()[None, :, None]

        def rope(y):
            y = rms(y)
            a, e = y[..., : hd // 2], y[..., hd // 2:]
            return torch.cat([a * cos - e * sin, e * cos + a * sin], -1)

        for i, w in enumerate(layers):
            y = rms(x)
            q, k, v = (_lin64(y, *w["attn." + n]).view(b, t, -1, hd) for n in ("wq", "wk", "wv"))
            q, k = rope(q), rope(k)
            if c["kv_int8"]:
                k, v = (((z / (sc := z.abs().amax(-1, keepdim=True) / 127)).round().clamp(-127, 127) * sc) for z in (k, v))
            if cache[i] is not None:
                k, v = torch.cat([cache[i][0], k], 1), torch.cat([cache[i][1], v], 1)
            cache[i] = (k, v)
            out = torch.empty_like(q)
            mask = torch.arange(k.shape[1], device="cuda")[None, :] > torch.arange(pos0, pos0 + t, device="cuda")[:, None]
            for s in range(b):
                for h in range(nh):
                    p = (q[s, :, h] @ k[s, :, h * nkv // nh].t()) * hd ** -0.5
                    out[s, :, h] = torch.softmax(p.masked_fill_(mask, -math.inf), -1) @ v[s, :, h * nkv // nh]
            x = x + _lin64(out.view(b * t, -1), *w["attn.wo"])
            y = rms(x)
            gate = _lin64(y, *w["mlp.gate"])
            x = x + _lin64(gate / (1 + (-gate).exp()) * _lin64(y, *w["mlp.up"]), *w["mlp.down"])
        return _lin64(rms(x.view(b, t, -1)[:, -1]), head, hs)

    logits = forward(_prompts(c, seed), 0)
    toks = [logits.argmax(1)]
    for j in range(c.get("steps", 0)):
        logits = forward(toks[-1][:, None], c["prompt"] + j)
        toks.append(logits.argmax(1))
    return [None, logits]


# ------------------------------------------------------------------ the interface


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("linear", "w4a8"):
        x, q, sw, bias = _linear_inputs(case, seed)
        return dict(kind=kind, x=x, w=_pack4(q) if kind == "w4a8" else _pack8(q), sw=sw, bias=bias)
    if kind == "dit":
        return dict(kind=kind, s=DitInt8Stack(layers=case["layers"], m=case["m"], seed=seed))
    if kind == "moe":
        x, w, gate = _moe_inputs(case, seed)
        return dict(kind=kind, x=x, w=[(_pack8(q), s) for q, s in w], gate=gate)
    if kind == "paged":
        return dict(kind=kind, s=_prepare_paged(case, seed))
    return dict(kind=kind, s=_prepare_qwen3(case, seed))


def run(state):
    kind = state["kind"]
    if kind == "linear":
        return _run_linear(state)
    if kind == "w4a8":
        return _run_w4a8(state)
    if kind == "moe":
        return _run_moe(state)
    return dict(dit=_run_dit, paged=_run_paged, prefill=_run_prefill, generate=_run_generate)[kind](state["s"])


def exact(case, seed):
    kind = case["kind"]
    if kind in ("linear", "w4a8"):
        x, q, sw, bias = _linear_inputs(case, seed)
        return _lin64(x.double(), q, sw, bias)
    if kind == "moe":
        x, w, gate = _moe_inputs(case, seed)
        return [torch.where(gate[:, e:e + 1] > 0, _lin64(x.double(), *w[e]), 0.0) for e in range(len(w))]
    return dict(dit=_exact_dit, paged=_exact_paged, prefill=_exact_qwen3, generate=_exact_qwen3)[kind](case, seed)


def _attn_keys(c):
    """(query rows, sum of keys they attend) of a whole engine call."""
    p, st = c["prompt"], c.get("steps", 0)
    total = p + st
    return c["batch"] * total, c["batch"] * total * (total + 1) // 2


def work(case):
    c, kind = case, case["kind"]
    if kind == "linear":
        m, k, n = c["m"], c["k"], c["n"]
        e = 2 if c["dtype"] == "bf16" else 4
        return dict(bytes=e * m * k + n * k + 4 * n * (2 if c["bias"] else 1) + e * m * n, flops=2 * m * n * k)
    if kind == "w4a8":
        m, k, n = c["m"], c["k"], c["n"]
        return dict(bytes=4 * m * k + n * k // 2 + 4 * n + 4 * m * n, flops=2 * m * n * k)
    if kind == "dit":
        per = DIT_D * DIT_QKV + DIT_D * DIT_D + 2 * DIT_D * DIT_FF
        scales = 4 * (DIT_QKV + 2 * DIT_D + DIT_FF)
        acts = 2 * c["m"] * (3 * DIT_D + DIT_QKV + DIT_FF)
        return dict(bytes=c["layers"] * (per + scales) + acts, flops=2 * c["layers"] * c["m"] * per)
    if kind == "moe":
        m, k, n, e = c["m"], c["k"], c["n"], c["experts"]
        return dict(bytes=4 * m * k + 4 * m * e + e * (n * k + 4 * n) + 4 * e * m * n, flops=2 * m * c["top"] * n * k)
    if kind == "paged":
        b, h, nkv, hd, ctx = c["batch"], c["heads"], c["kv_heads"], c["head_dim"], c["ctx"]
        keys = b * ctx * 3 // 4
        return dict(bytes=2 * keys * nkv * (hd + 4) + 4 * keys * h + 8 * b * h * hd, flops=4 * keys * h * hd)
    cfg = QWEN3_0_6B
    rows, pairs = _attn_keys(c)
    kvd = cfg["n_kv_heads"] * cfg["head_dim"]
    hq = cfg["n_heads"] * cfg["head_dim"]
    per = cfg["d_model"] * (2 * hq + 2 * kvd + 3 * cfg["d_ff"])
    head = cfg["vocab"] * cfg["d_model"]
    steps = c.get("steps", 0)
    kv_row = cfg["n_layers"] * 2 * (kvd + 4 * cfg["n_kv_heads"] if c["kv_int8"] else 4 * kvd)
    kv_read = c["batch"] * steps * (c["prompt"] + steps // 2) * kv_row
    return dict(bytes=(1 + steps) * (cfg["n_layers"] * per + head) + rows * kv_row + kv_read + 4 * c["batch"] * cfg["vocab"],
                flops=2 * rows * cfg["n_layers"] * per + 2 * (1 + steps) * c["batch"] * head
                + 4 * pairs * hq * cfg["n_layers"])


def tolerance(case):
    kind = case["kind"]
    if kind in ("linear", "w4a8", "moe"):
        # The integer sums are exact; the scales and the products round once each.
        return dict(rel=1e-2) if case.get("dtype") == "bf16" else dict(rel=1e-5)
    if kind == "dit":
        return dict(rel=2e-2)  # bf16 between the linears: an output rounded the other way moves a code of the next
    if kind == "paged":
        return dict(rel=1e-5, differ=1e-5)  # 32-bit sums over head_dim and positions
    # 28 layers of int8 codes: a rounding that moves one code travels on.
    return dict(rel=3e-2)
