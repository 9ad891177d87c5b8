"""The work a user of this library has it do, as measurable cases.

Every case is one call, or one layer's sequence of calls, through the public
torch-facing ops (``gemm``, ``linear``, ``rms_norm``, ``rms_norm_linear``,
``gemv``, ``w8a16_linear``, ``bgemm``, ``softmax``, ``attention``,
``decode_step``), eagerly on the current stream as a model's forward makes
them.  ``listed()`` holds the cases themselves, ``draw(rng)`` takes one more
from the same ranges, ``prepare`` makes what a program has in hand before the
call, ``run`` is one pass, ``work`` what the pass cannot do without,
``tolerance`` how far another correct implementation may be off and ``exact``
the same results in 64 bits.
"""
import math
import random

import torch
import torch.nn.functional as F

import __graft_entry__

pkg = __graft_entry__.load_package()

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}
EPS = 1e-5

# (hidden, intermediate, heads, kv heads, head dim, projections carry a bias)
TINYLLAMA = dict(hidden=2048, inter=5632, heads=32, kv_heads=4, head_dim=64, bias=False)
QWEN = dict(hidden=896, inter=4864, heads=14, kv_heads=2, head_dim=64, bias=True)


def listed():
    return [
        # the smallest row kernel of a 512-token TinyLlama prefill: launch and latency bound
        dict(name="rms_norm_512x2048", kind="rms_norm", rows=512, cols=2048, dtype="fp16"),
        # the smallest decode projection of Qwen2.5-0.5B, one token
        dict(name="gemv_896x896_m1", kind="gemv", m=1, n=896, k=896, dtype="fp16"),
        # int8 weight-only lm_head of Qwen2.5-0.5B over a prompt chunk of 256 tokens
        dict(name="w8a16_lm_head_m256", kind="w8a16", m=256, n=151936, k=896),
        # the repository's first benchmark configuration: one 1024^3 product, B as [K, N]
        dict(name="gemm_nn_1024", kind="gemm", m=1024, n=1024, k=1024, layout="nn", dtype="fp16", epi="none"),
        # its large product: 4096^3, B as nn.Linear holds it
        dict(name="gemm_nt_4096", kind="gemm", m=4096, n=4096, k=4096, layout="nt", dtype="fp16", epi="none"),
        # the headline workload: the projections of one TinyLlama-1.1B layer, 512-token prefill
        dict(name="llama_block_512", kind="block", tokens=512, dtype="fp16", **TINYLLAMA),
        # the same layer over a long prompt, in the other 16-bit type
        dict(name="llama_block_4096_bf16", kind="block", tokens=4096, dtype="bf16", **TINYLLAMA),
        # ViT-B/16, batch 8: fused attention over 197 tokens, fc1 + GELU, fc2
        dict(name="vit_block_b8", kind="vit", batch=8, tokens=197, heads=12, head_dim=64, mlp=3072, dtype="fp16"),
        # ViT-B/16, batch 8: the reference's own three steps with the scores materialised, every row 197 long
        dict(name="vit_attention_steps_b8", kind="steps", slices=96, tokens=197, head_dim=64, dtype="fp16"),
        # causal prefill attention with grouped heads, TinyLlama at 2048 tokens
        dict(name="attention_gqa_2048", kind="attention", batch=1, heads=32, kv_heads=4, s=2048, skv=2048, d=64,
             dtype="fp16", causal=1, pad=False),
        # causal prefill attention at head dim 128 in bf16
        dict(name="attention_bf16_d128", kind="attention", batch=2, heads=16, kv_heads=4, s=1024, skv=1024, d=128,
             dtype="bf16", causal=1, pad=False),
        # one-token forward of all 24 layers and the lm_head of Qwen2.5-0.5B, logits out
        dict(name="decode_qwen", kind="decode", layers=24, vocab=151936, fold=True, **QWEN),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng: random.Random):
    kind = rng.choice(["rms_norm", "gemv", "w8a16", "gemm", "gemm", "block", "block", "vit", "steps", "attention",
                       "attention", "decode"])
    dtype = rng.choice(["fp16", "fp16", "bf16"])
    if kind == "rms_norm":
        # rows: tokens of a decode batch up to a long prefill; columns: hidden sizes, some not multiples of 8
        cols = rng.choice([896, 2048, 768, 4096, 8 * _log_int(rng, 16, 1024), _log_int(rng, 128, 8192)])
        return dict(kind=kind, rows=_log_int(rng, 1, 4096), cols=cols, dtype=dtype)
    if kind == "gemv":
        n, k = rng.choice([(896, 896), (128, 896), (4864, 896), (9728, 896), (896, 4864), (151936, 896),
                           (2560, 2048), (2048, 2048), (11264, 2048), (2048, 5632), (32000, 2048),
                           (8 * _log_int(rng, 16, 2048), 8 * _log_int(rng, 16, 1024))])
        return dict(kind=kind, m=rng.randint(1, 16), n=n, k=k, dtype=dtype)
    if kind == "w8a16":
        n, k = rng.choice([(896, 896), (4864, 896), (896, 4864), (151936, 896), (2048, 2048), (2048, 5632),
                           (8 * _log_int(rng, 16, 2048), 16 * _log_int(rng, 8, 512))])
        return dict(kind=kind, m=_log_int(rng, 1, 256), n=n, k=k)
    if kind == "gemm":
        # rows are tokens, so any number; K and N are widths, multiples of 8 but for a few odd heads and tables
        layout = rng.choice(["nt", "nt", "nn"])
        epi = rng.choice(["none", "bias", "bias_gelu_tanh"]) if layout == "nt" else "none"
        m = _log_int(rng, 17, 4096)
        if rng.random() < 0.2:
            n, k = _log_int(rng, 33, 1024), _log_int(rng, 33, 1024)
            m = min(m, 1024)
        else:
            n, k = 8 * _log_int(rng, 8, 512), 8 * _log_int(rng, 8, 512)
        return dict(kind=kind, m=m, n=n, k=k, layout=layout, dtype=dtype, epi=epi)
    if kind == "block":
        return dict(kind=kind, tokens=_log_int(rng, 17, 4096), dtype=dtype, **rng.choice([TINYLLAMA, QWEN]))
    if kind == "vit":
        tokens = rng.choice([197, 50, 145, 257, 577, rng.randint(40, 640)])
        return dict(kind=kind, batch=rng.randint(1, 8), tokens=tokens, heads=12, head_dim=64, mlp=3072, dtype=dtype)
    if kind == "steps":
        tokens = rng.choice([197, 50, 145, 257, rng.randint(40, 320)])
        most = max(1, 96 * 197 * 197 // (tokens * tokens))
        return dict(kind=kind, slices=min(12 * rng.randint(1, 8), most), tokens=tokens,
                    head_dim=rng.choice([64, 64, 80]), dtype=dtype)
    if kind == "attention":
        kv = rng.choice([1, 2, 4, 8])
        heads = kv * rng.choice([1, 2, 4, 8])
        batch = rng.choice([1, 1, 2, 4])
        while heads > 32 or batch * heads > 64:
            batch, heads, kv = max(1, batch // 2), heads // 2 if heads > 32 else heads, max(1, kv // 2) if heads > 32 else kv
        s = _log_int(rng, 64, 2048)
        causal = rng.choice([0, 1, 1, 2])
        skv = s + _log_int(rng, 16, 1024) if causal == 2 else s  # 2: a prompt chunk behind earlier keys
        return dict(kind=kind, batch=batch, heads=heads, kv_heads=kv, s=s, skv=skv,
                    d=rng.choice([64, 64, 128, 128, 80]), dtype=dtype, causal=causal,
                    pad=batch > 1 and rng.random() < 0.5)
    return dict(kind="decode", layers=rng.randint(2, 24), vocab=8 * _log_int(rng, 1000, 18992), fold=rng.random() < 0.7,
                **QWEN)


# ---- inputs -----------------------------------------------------------------


def _rng(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(g, *shape, std=1.0, mean=0.0, dtype=torch.float16):
    return (torch.randn(*shape, generator=g, device="cuda") * std + mean).to(dtype)


def _inputs(c, seed):
    """The tensors of a case before anything of the library touches them:
    activations N(0,1) (uniform [-1,1] for the plain products), weights
    N(0,0.02), norm weights around 1, int8 codes uniform with scales
    U(1e-3, 1e-2)."""
    g = _rng(seed)
    kind = c["kind"]
    dt = DTYPES[c.get("dtype", "fp16")]
    t = {}
    if kind == "rms_norm":
        t["x"] = _normal(g, c["rows"], c["cols"], dtype=dt)
        t["w"] = _normal(g, c["cols"], std=0.02, mean=1.0, dtype=dt)
    elif kind == "gemv":
        t["x"] = _normal(g, c["m"], c["k"], dtype=dt)
        t["w"] = _normal(g, c["n"], c["k"], std=0.02, dtype=dt)
    elif kind == "w8a16":
        t["x"] = _normal(g, c["m"], c["k"], dtype=dt)
        t["q"] = torch.randint(-127, 128, (c["n"], c["k"]), generator=g, device="cuda", dtype=torch.int8)
        t["s"] = (torch.rand(c["n"], generator=g, device="cuda") * 9e-3 + 1e-3).half()
    elif kind == "gemm":
        b = (c["n"], c["k"]) if c["layout"] == "nt" else (c["k"], c["n"])
        if c["epi"] == "none":
            t["a"] = (torch.rand(c["m"], c["k"], generator=g, device="cuda") * 2 - 1).to(dt)
            t["b"] = (torch.rand(*b, generator=g, device="cuda") * 2 - 1).to(dt)
        else:
            t["a"] = _normal(g, c["m"], c["k"], dtype=dt)
            t["b"] = _normal(g, *b, std=0.02, dtype=dt)
            t["bias"] = _normal(g, c["n"], std=0.02, dtype=dt)
    elif kind == "block":
        h, i, kv = c["hidden"], c["inter"], c["kv_heads"] * c["head_dim"]
        t["x"] = _normal(g, c["tokens"], h, dtype=dt)
        t["xa"] = _normal(g, c["tokens"], h, dtype=dt)  # the attention's output
        t["gn"] = _normal(g, h, std=0.02, mean=1.0, dtype=dt)
        t["wqkv"] = _normal(g, h + 2 * kv, h, std=0.02, dtype=dt)
        t["bqkv"] = _normal(g, h + 2 * kv, std=0.1, dtype=dt) if c["bias"] else None
        t["wo"] = _normal(g, h, h, std=0.02, dtype=dt)
        t["wg"] = _normal(g, i, h, std=0.02, dtype=dt)
        t["wu"] = _normal(g, i, h, std=0.02, dtype=dt)
        t["wd"] = _normal(g, h, i, std=0.02, dtype=dt)
    elif kind == "vit":
        e = c["heads"] * c["head_dim"]
        for n in "qkv":
            t[n] = _normal(g, c["batch"], c["heads"], c["tokens"], c["head_dim"], dtype=dt)
        t["x"] = _normal(g, c["batch"], c["tokens"], e, dtype=dt)
        t["w1"], t["b1"] = _normal(g, c["mlp"], e, std=0.02, dtype=dt), _normal(g, c["mlp"], std=0.02, dtype=dt)
        t["w2"], t["b2"] = _normal(g, e, c["mlp"], std=0.02, dtype=dt), _normal(g, e, std=0.02, dtype=dt)
    elif kind == "steps":
        for n in "qkv":
            t[n] = _normal(g, c["slices"], c["tokens"], c["head_dim"], dtype=dt)
    elif kind == "attention":
        t["q"] = _normal(g, c["batch"], c["heads"], c["s"], c["d"], dtype=dt)
        for n in "kv":
            t[n] = _normal(g, c["batch"], c["kv_heads"], c["skv"], c["d"], dtype=dt)
        if c["pad"]:
            # right-padded batch: row b keeps its first keys (additive mask [B, 1, S, S_kv])
            keep = torch.randint(max(1, c["skv"] // 2), c["skv"] + 1, (c["batch"], 1, 1, 1), generator=g, device="cuda")
            gone = torch.arange(c["skv"], device="cuda").view(1, 1, 1, -1) >= keep
            t["mask"] = torch.zeros(c["batch"], 1, c["s"], c["skv"], dtype=torch.float16, device="cuda").masked_fill_(
                gone, float("-inf"))
    else:
        L, h, i, kv = c["layers"], c["hidden"], c["inter"], c["kv_heads"] * c["head_dim"]
        t["x"] = _normal(g, h)
        t["w_qkv"], t["b_qkv"] = _normal(g, L, h + 2 * kv, h, std=0.02), _normal(g, L, h + 2 * kv, std=0.1)
        t["w_o"] = _normal(g, L, h, h, std=0.02)
        t["w_gu"], t["w_down"] = _normal(g, L, 2 * i, h, std=0.02), _normal(g, L, h, i, std=0.02)
        t["g_attn"], t["g_mlp"] = _normal(g, L, h, std=0.1, mean=1.0), _normal(g, L, h, std=0.1, mean=1.0)
        t["g_final"], t["w_lm"] = _normal(g, h, std=0.1, mean=1.0), _normal(g, c["vocab"], h, std=0.02)
    return t


def prepare(case, seed):
    t = _inputs(case, seed)
    kind = case["kind"]
    if kind == "block":
        # load-time weight layouts: gate and up interleaved, the norm weight folded into its consumers
        t["wqkv_f"] = pkg.fold_rms_weight(t["wqkv"], t["gn"])
        t["wgu_f"] = pkg.fold_rms_weight(pkg.pack_gate_up(t["wg"], t["wu"]), t["gn"])
        t["rs"] = torch.empty(case["tokens"], dtype=torch.float32, device="cuda")
        for n in ("wqkv", "wg", "wu"):
            del t[n]
    elif kind == "decode":
        x = t.pop("x")
        stack = pkg.hxmi.DecoderStack(**t, heads=case["heads"], kv_heads=case["kv_heads"], eps=1e-6)
        t = {"x": x, "stack": stack.fold_o() if case["fold"] else stack}
    return {"case": case, **t}


# ---- one pass ---------------------------------------------------------------


def run(state):
    c = state["case"]
    kind = c["kind"]
    if kind == "rms_norm":
        return pkg.rms_norm(state["x"], state["w"], EPS)
    if kind == "gemv":
        return pkg.gemv(state["x"], state["w"])
    if kind == "w8a16":
        return pkg.w8a16_linear(state["x"], state["q"], state["s"])
    if kind == "gemm":
        if c["layout"] == "nn" or c["epi"] == "none":
            return pkg.gemm(state["a"], state["b"], b_layout=c["layout"])
        return pkg.linear(state["a"], state["b"], state["bias"],
                          epilogue="gelu_tanh" if c["epi"] == "bias_gelu_tanh" else None)
    if kind == "block":
        qkv = pkg.rms_norm_linear(state["x"], state["wqkv_f"], EPS, rscale_out=state["rs"], bias=state["bqkv"])
        o = pkg.linear(state["xa"], state["wo"])
        h = pkg.rms_norm_linear(state["x"], state["wgu_f"], EPS, epilogue="silu_mul", rscale_in=state["rs"])
        return {"qkv": qkv, "o": o, "h": h, "down": pkg.linear(h, state["wd"])}
    if kind == "vit":
        attn = pkg.attention(state["q"], state["k"], state["v"])
        h = pkg.linear(state["x"], state["w1"], state["b1"], epilogue="gelu_tanh")
        return {"attn": attn, "h": h, "y": pkg.linear(h, state["w2"], state["b2"])}
    if kind == "steps":
        s = pkg.bgemm(state["q"], state["k"], b_layout="nt")
        p = pkg.softmax(s, c["head_dim"] ** -0.5)
        return {"scores": s, "p": p, "o": pkg.bgemm(p, state["v"])}
    if kind == "attention":
        return pkg.attention(state["q"], state["k"], state["v"], mask=state.get("mask"), causal=c["causal"])
    out = pkg.hxmi.decode_step(state["x"], state["stack"])
    return {"h": out["h"], "x": out["x"], "logits": out["logits"]}


# ---- what a pass cannot do without ------------------------------------------


def work(case):
    """Each input read once, each output written once; the products' flops."""
    c, kind = case, case["kind"]
    if kind == "rms_norm":
        return {"bytes": 2 * (2 * c["rows"] * c["cols"] + c["cols"]), "flops": 4 * c["rows"] * c["cols"]}
    if kind in ("gemv", "gemm"):
        m, n, k = c["m"], c["n"], c["k"]
        return {"bytes": 2 * (m * k + n * k + m * n), "flops": 2 * m * n * k}
    if kind == "w8a16":
        m, n, k = c["m"], c["n"], c["k"]
        return {"bytes": n * k + 2 * n + 2 * m * k + 2 * m * n, "flops": 2 * m * n * k}
    if kind == "block":
        t, h, i, q = c["tokens"], c["hidden"], c["inter"], c["hidden"] + 2 * c["kv_heads"] * c["head_dim"]
        weights = q * h + h * h + 2 * i * h + h * i
        return {"bytes": 2 * (weights + t * (2 * h + q + h + 2 * i + h)), "flops": 2 * t * weights}
    if kind == "vit":
        b, s, e, f = c["batch"], c["tokens"], c["heads"] * c["head_dim"], c["mlp"]
        return {"bytes": 2 * (b * s * (4 * e + e + 2 * f + e) + 2 * e * f),
                "flops": 4 * b * s * s * e + 4 * b * s * e * f}
    if kind == "steps":
        n, s, d = c["slices"], c["tokens"], c["head_dim"]
        return {"bytes": 2 * n * (4 * s * d + 4 * s * s), "flops": 4 * n * s * s * d}
    if kind == "attention":
        pairs = c["s"] * c["skv"]
        if c["causal"]:  # query r sees r + 1 keys, behind skv - s earlier ones for the second rule
            pairs = c["s"] * (c["s"] + 1) // 2 + c["s"] * (c["skv"] - c["s"])
        kv = c["kv_heads"] * c["skv"]
        mask = c["batch"] * c["s"] * c["skv"] * 2 if c["pad"] else 0
        return {"bytes": 2 * c["batch"] * c["d"] * 2 * (c["heads"] * c["s"] + kv) + mask,
                "flops": 4 * c["batch"] * c["heads"] * pairs * c["d"]}
    h, i, q = c["hidden"], c["inter"], c["hidden"] + 2 * c["kv_heads"] * c["head_dim"]
    weights = c["layers"] * (q * h + h * h + 3 * h * i) + c["vocab"] * h
    return {"bytes": 2 * (weights + c["vocab"]), "flops": 2 * weights}


def tolerance(case):
    """One rounding of each output to its 16-bit type (relative 2-norm ~1.7e-4
    in fp16, ~1.4e-3 in bf16), with those of the intermediates that stay in
    16 bits: about four times what the path measures against ``exact``."""
    bf = case.get("dtype") == "bf16"
    if case["kind"] == "decode":
        return {"rel": 1e-2}  # 24 layers of fp16 roundings
    if case["kind"] in ("rms_norm", "block"):
        return {"rel": 1.2e-2 if bf else 1.5e-3}  # the folded norm weight / the normalised row round once more
    if case["kind"] in ("steps", "attention", "vit"):
        return {"rel": 1.5e-2 if bf else 2e-3}  # 16-bit probabilities (and scores, in the three steps)
    return {"rel": 8e-3 if bf else 1e-3}


# ---- the same in 64 bits ----------------------------------------------------


def _rms(x, eps):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps)


def _sdpa(q, k, v, scale, mask=None, causal=0):
    """softmax(scale q k^T + mask) v over [N, S, D] slices, a slice at a time."""
    out = torch.empty(q.shape[0], q.shape[1], v.shape[2], dtype=q.dtype, device=q.device)
    s, skv = q.shape[1], k.shape[1]
    gone = None
    if causal:
        off = skv - s if causal == 2 else 0
        gone = torch.arange(skv, device=q.device)[None, :] > torch.arange(s, device=q.device)[:, None] + off
    for n in range(q.shape[0]):
        p = q[n] @ k[n].t().contiguous() * scale
        if mask is not None:
            p = p + mask[n]
        if gone is not None:
            p = p.masked_fill(gone, float("-inf"))
        out[n] = torch.softmax(p, -1) @ v[n]
    return out


def exact(case, seed):
    c, kind = case, case["kind"]
    t = {n: v.double() for n, v in _inputs(case, seed).items() if v is not None}
    if kind == "rms_norm":
        return _rms(t["x"], EPS) * t["w"]
    if kind == "gemv":
        return t["x"] @ t["w"].t()
    if kind == "w8a16":
        return (t["x"] @ t["q"].t()) * t["s"]
    if kind == "gemm":
        y = t["a"] @ (t["b"].t() if c["layout"] == "nt" else t["b"])
        if c["epi"] != "none":
            y = y + t["bias"]
        return F.gelu(y, approximate="tanh") if c["epi"] == "bias_gelu_tanh" else y
    if kind == "block":
        xn = _rms(t["x"], EPS) * t["gn"]
        qkv = xn @ t["wqkv"].t()
        if c["bias"]:
            qkv = qkv + t["bqkv"]
        h = F.silu(xn @ t["wg"].t()) * (xn @ t["wu"].t())
        return {"qkv": qkv, "o": t["xa"] @ t["wo"].t(), "h": h, "down": h @ t["wd"].t()}
    if kind == "vit":
        q, k, v = (t[n].flatten(0, 1) for n in "qkv")
        h = F.gelu(t["x"] @ t["w1"].t() + t["b1"], approximate="tanh")
        return {"attn": _sdpa(q, k, v, c["head_dim"] ** -0.5).view(t["q"].shape), "h": h,
                "y": h @ t["w2"].t() + t["b2"]}
    if kind == "steps":
        s = torch.stack([t["q"][n] @ t["k"][n].t().contiguous() for n in range(c["slices"])])
        p = torch.softmax(s * c["head_dim"] ** -0.5, -1)
        return {"scores": s, "p": p, "o": torch.stack([p[n] @ t["v"][n] for n in range(c["slices"])])}
    if kind == "attention":
        q, grp = t["q"], c["heads"] // c["kv_heads"]
        k, v = (t[n].repeat_interleave(grp, dim=1).flatten(0, 1) for n in "kv")
        mask = t["mask"].expand(c["batch"], c["heads"], c["s"], c["skv"]).flatten(0, 1) if c["pad"] else None
        return _sdpa(q.flatten(0, 1), k, v, c["d"] ** -0.5, mask, c["causal"]).view(q.shape)
    # the decoder forward at position 0: attention over one key returns its value row
    h, i, kv, hd = c["hidden"], c["inter"], c["kv_heads"] * c["head_dim"], c["head_dim"]
    grp = c["heads"] // c["kv_heads"]
    x = t["x"]
    for n in range(c["layers"]):
        qkv = t["w_qkv"][n] @ (_rms(x, 1e-6) * t["g_attn"][n]) + t["b_qkv"][n]
        x = x + t["w_o"][n] @ qkv[h + kv:].view(-1, hd).repeat_interleave(grp, dim=0).reshape(-1)
        gu = t["w_gu"][n] @ (_rms(x, 1e-6) * t["g_mlp"][n])
        x = x + t["w_down"][n] @ (F.silu(gu[:i]) * gu[i:])
    out = _rms(x, 1e-6) * t["g_final"]
    return {"h": out, "x": x, "logits": t["w_lm"] @ out}
