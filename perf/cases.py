"""What this framework is measured on: the calls that a batch-1 decode and
prefill program makes, over the sizes of its model configurations.

The operator cases are the single projections, heads, attention layers and norm
rows of the 1.7B, 8B, 9B and 27B geometries (lib.CONFIGS), called through
``Ctx`` as a plugin host calls them; the two whole calls are
``Model.generate`` on the 8B dense decoder at 2k context and on the 9B hybrid
with a 512-token prompt.  Weights are random blocks of the GGUF formats.
"""
import math

import numpy as np
import torch

from hearth_amd import (CONFIGS, GGML_PQ2_0, GGML_PTQ1_0, GGML_Q1_0, GGML_Q1_0_G128, GGML_Q2_0, GGML_Q8_0, Ctx,
                        Model, row_bytes)

FORMATS = {"q1_0": GGML_Q1_0, "q1_0_g128": GGML_Q1_0_G128, "q2_0": GGML_Q2_0, "pq2_0": GGML_PQ2_0,
           "ptq1_0": GGML_PTQ1_0, "q8_0": GGML_Q8_0}

_CTX = None


def _ctx():
    """The program's one device context."""
    global _CTX
    if _CTX is None:
        _CTX = Ctx(0)
    return _CTX


def listed():
    return [
        # one small projection of the 1.7B decoder: what a single call costs
        {"name": "gemv_q1_2048x2048", "kind": "gemv", "fmt": "q1_0", "rows": 2048, "cols": 2048},
        # the 27B FFN down projection in the 1.75-bit ternary format
        {"name": "gemv_ptq1_5120x17408", "kind": "gemv", "fmt": "ptq1_0", "rows": 5120, "cols": 17408},
        # the 8B fused gate+up projection
        {"name": "gemv_q2_24576x4096", "kind": "gemv", "fmt": "q2_0", "rows": 24576, "cols": 4096},
        # the 8B LM head and the greedy choice with the repetition penalty over a reply's tokens
        {"name": "head_q8_151936x4096", "kind": "head", "rows": 151936, "cols": 4096, "past": 200},
        # a short chat message through the 1.7B q/k/v rows
        {"name": "gemm_q1_37x4096x2048", "kind": "gemm", "fmt": "q1_0", "seq": 37, "rows": 4096, "cols": 2048},
        # a long prompt through the 8B gate+up rows
        {"name": "gemm_q2_2048x24576x4096", "kind": "gemm", "fmt": "q2_0", "seq": 2048, "rows": 24576, "cols": 4096},
        # one decode step's attention in an 8B layer at 2k context
        {"name": "attn_8b_2049", "kind": "attn", "heads": 32, "kv": 8, "hd": 128, "cap": 2304, "seq": 2049},
        # a follow-up message's attention in an 8B layer, over the conversation so far
        {"name": "attn_prefill_8b_777", "kind": "attn_prefill", "heads": 32, "kv": 8, "hd": 128, "cap": 2304,
         "pos0": 250, "tokens": 777, "mode": 0},
        # a 1k prompt in a hybrid's full-attention layer, matrix-core form
        {"name": "attn_prefill_mfma_9b_1024", "kind": "attn_prefill", "heads": 16, "kv": 4, "hd": 256, "cap": 1088,
         "pos0": 0, "tokens": 1024, "mode": 1},
        # the norm and the Q8_0 activations in front of a projection, 512 prompt tokens
        {"name": "norm_quant_512x4096", "kind": "rows", "rows": 512, "cols": 4096},
        # a reply from the 8B decoder, 2k tokens into a conversation
        {"name": "decode_8b_2k", "kind": "model", "config": "8b-q2", "layers": 36, "kv_type": 0, "context": 2048,
         "prompt": 1, "gen": 32},
        # a fresh 512-token prompt and the first reply token from the 9B hybrid
        {"name": "prompt_9b_512", "kind": "model", "config": "9b-hybrid-q2", "layers": 32, "kv_type": 0, "context": 0,
         "prompt": 512, "gen": 1},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gemv", "gemv", "gemm", "gemm", "gemm", "head", "attn", "attn_prefill", "attn_prefill", "rows",
                       "model", "model"])
    if kind == "gemv":
        fmt = rng.choice(sorted(FORMATS))
        cols = 256 * _log(rng, 4, 68)
        return {"kind": kind, "fmt": fmt, "rows": min(_log(rng, 512, 151936), 151936 * 4096 // cols), "cols": cols}
    if kind == "head":
        return {"kind": kind, "rows": _log(rng, 32000, 151936), "cols": 1024 * rng.randint(1, 4),
                "past": _log(rng, 1, 2000)}
    if kind == "gemm":
        fmt = rng.choice(["q1_0", "q1_0_g128", "q2_0", "q2_0", "pq2_0", "ptq1_0", "q8_0"])
        cols = 128 * _log(rng, 8, 136)
        seq = _log(rng, 2, 2048)
        cap = 2048 * 24576 * 4096 // (4 if fmt == "q8_0" else 1)
        return {"kind": kind, "fmt": fmt, "seq": seq, "rows": min(_log(rng, 512, 34816), cap // (cols * seq)),
                "cols": cols}
    if kind in ("attn", "attn_prefill"):
        heads, kv, hd = rng.choice([(16, 8, 128), (32, 8, 128), (16, 4, 256), (24, 4, 256), (16, 2, 128)])
        if kind == "attn":
            seq = _log(rng, 1, 16384)
            return {"kind": kind, "heads": heads, "kv": kv, "hd": hd, "cap": seq + rng.randint(0, 300), "seq": seq}
        pos0, tokens = rng.choice([0, _log(rng, 1, 1500)]), _log(rng, 2, 1024)
        return {"kind": kind, "heads": heads, "kv": kv, "hd": hd, "cap": pos0 + tokens + rng.randint(0, 300),
                "pos0": pos0, "tokens": tokens, "mode": rng.randint(0, 1)}
    if kind == "rows":
        return {"kind": kind, "rows": _log(rng, 1, 2048), "cols": 32 * _log(rng, 32, 544)}
    name = rng.choice(["1.7b-q1", "8b-q2", "9b-hybrid-q2"])
    cfg = CONFIGS[name]
    context = 0 if cfg.arch else rng.choice([0, _log(rng, 16, 3000)])
    return {"kind": kind, "config": name, "layers": 4 * rng.randint(1, cfg.n_layers // 4),
            "kv_type": rng.choice([0, GGML_Q8_0]), "context": context, "prompt": _log(rng, 1, 512),
            "gen": rng.randint(1, 16)}


# ---- inputs ----

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _f16_scales(n, lo, hi, g):
    """n positive f16 block scales, spread over lo..hi, as little-endian byte pairs."""
    s = (lo + (hi - lo) * torch.rand(n, generator=g, device="cuda")).to(torch.float16)
    return s.view(torch.uint8).view(n, 2)


def _weights(fmt, rows, cols, g):
    """rows x cols random weights in the format's native blocks."""
    t = FORMATS[fmt]
    el = 32 if fmt == "q8_0" else 128
    nb = rows * (cols // el)
    w = torch.randint(0, 256, (nb, row_bytes(t, el)), dtype=torch.uint8, device="cuda", generator=g)
    at = 26 if fmt == "ptq1_0" else 0
    w[:, at:at + 2] = _f16_scales(nb, 1e-4, 4e-4, g) if fmt == "q8_0" else _f16_scales(nb, 0.01, 0.04, g)
    return w


def _activations(seq, cols, g):
    """Q8_0 blocks of an N(0,1)-like activation: bytes spread as a block's own maximum scales them."""
    nb = seq * (cols // 32)
    q = torch.randn(nb, 32, generator=g, device="cuda")
    q = torch.round(q * (127.0 / q.abs().amax(1, keepdim=True))).to(torch.int8)
    x = torch.empty(nb, 34, dtype=torch.uint8, device="cuda")
    x[:, :2] = _f16_scales(nb, 0.01, 0.03, g)
    x[:, 2:] = q.view(torch.uint8)
    return x


def _qkv(case, g):
    n = case.get("tokens", 1)
    q = torch.randn(n, case["heads"], case["hd"], generator=g, device="cuda")
    k = torch.randn(case["kv"], case["cap"], case["hd"], generator=g, device="cuda")
    v = torch.randn(case["kv"], case["cap"], case["hd"], generator=g, device="cuda")
    return q, k, v


def _row_inputs(case, g):
    x = 2.0 * torch.randn(case["rows"], case["cols"], generator=g, device="cuda")
    w = 1.0 + 0.02 * torch.randn(case["cols"], generator=g, device="cuda")
    return x, w


def _past(case, g):
    return torch.randint(0, case["rows"], (case["past"],), dtype=torch.int32, device="cuda", generator=g)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "model":
        return _prepare_model(case, seed)
    ctx, g = _ctx(), _gen(seed)
    s = {"kind": kind, "case": case, "ctx": ctx}
    if kind in ("gemv", "head"):
        s["w"] = _weights(case.get("fmt", "q8_0"), case["rows"], case["cols"], g)
        s["x"] = _activations(1, case["cols"], g)
        s["y"] = torch.zeros(case["rows"], dtype=torch.float32, device="cuda")
        if kind == "head":
            s["past"] = _past(case, g)
            s["token"] = torch.zeros(1, dtype=torch.int32, device="cuda")
    elif kind == "gemm":
        s["w"] = _weights(case["fmt"], case["rows"], case["cols"], g)
        s["x"] = _activations(case["seq"], case["cols"], g)
        s["y"] = torch.zeros(case["seq"], case["rows"], dtype=torch.float32, device="cuda")
    elif kind in ("attn", "attn_prefill"):
        s["q"], s["k"], s["v"] = _qkv(case, g)
        s["out"] = torch.zeros_like(s["q"])
    else:
        s["x"], s["w"] = _row_inputs(case, g)
        s["y"] = torch.zeros_like(s["x"])
        s["q8"] = torch.zeros(case["rows"], case["cols"] // 32 * 34, dtype=torch.uint8, device="cuda")
    return s


def _prepare_model(case, seed):
    c = CONFIGS[case["config"]].replace(n_layers=case["layers"], kv_type=case["kv_type"])
    c = c.replace(max_seq=max(256, -(-(case["context"] + case["prompt"] + case["gen"]) // 256) * 256))
    m = Model(_ctx(), c)
    m.synthesize(seed)
    if case["context"]:
        m.prefill_kv_synthetic(seed + 1, case["context"])
    toks = np.random.default_rng(seed).integers(0, c.vocab, case["prompt"]).astype(np.uint32)
    return {"kind": "model", "case": case, "model": m, "prompt": toks}


# ---- one pass ----

def run(s):
    kind, c = s["kind"], s["case"]
    if kind == "model":
        m = s["model"]
        if not c["context"]:
            m.reset()   # a fresh session
        toks, logits = m.generate(s["prompt"], c["gen"], start_pos=c["context"], repeat_pen=1.1, want_logits=True)
        return {"tokens": toks.astype(np.int64), "logits": logits}
    ctx = s["ctx"]
    if kind == "gemv":
        ctx.gemv_q8(FORMATS[c["fmt"]], s["w"], c["rows"], c["cols"], s["x"], s["y"])
        return s["y"]
    if kind == "head":
        ctx.gemv_q8(GGML_Q8_0, s["w"], c["rows"], c["cols"], s["x"], s["y"])
        ctx.argmax(s["y"], c["rows"], s["past"], c["past"], 1.1, 0, s["token"])
        return {"logits": s["y"], "token": s["token"]}
    if kind == "gemm":
        ctx.gemm_q8(FORMATS[c["fmt"]], s["w"], c["rows"], c["cols"], s["x"], c["seq"], s["y"])
        return s["y"]
    if kind == "attn":
        ctx.attention(s["q"], s["k"], s["v"], c["heads"], c["kv"], c["hd"], c["cap"], c["seq"], s["out"])
        return s["out"]
    if kind == "attn_prefill":
        ctx.attention_prefill(s["q"], s["k"], s["v"], c["heads"], c["kv"], c["hd"], c["cap"], c["pos0"], c["tokens"],
                              c["mode"], s["out"])
        return s["out"]
    ctx.rms_norm(s["x"], s["w"], 1e-6, c["rows"], c["cols"], s["y"])
    ctx.quantize_q8_0(s["y"], c["rows"] * c["cols"], s["q8"])
    return {"normed": s["y"], "q8": s["q8"]}


# ---- what a pass cannot do without ----

def work(case):
    kind = case["kind"]
    if kind in ("gemv", "gemm", "head"):
        n, k, s = case["rows"], case["cols"], case.get("seq", 1)
        wb = n * row_bytes(FORMATS[case.get("fmt", "q8_0")], k)
        return {"bytes": wb + s * (k // 32) * 34 + 4 * s * n + (4 * case["past"] + 4 if kind == "head" else 0),
                "flops": 2 * s * n * k}
    if kind in ("attn", "attn_prefill"):
        n, pos0 = case.get("tokens", 1), case.get("pos0", case.get("seq", 1) - 1)
        rows = sum(pos0 + t + 1 for t in range(n))
        return {"bytes": 4 * case["hd"] * (2 * case["kv"] * (pos0 + n) + 2 * n * case["heads"]),
                "flops": 4 * case["heads"] * case["hd"] * rows}
    if kind == "rows":
        n = case["rows"] * case["cols"]
        return {"bytes": 8 * n + 4 * case["cols"] + n // 32 * 34, "flops": 6 * n}
    cfg = CONFIGS[case["config"]].replace(n_layers=case["layers"], kv_type=case["kv_type"])
    d, f, hd, nq, nkv = cfg.d_model, cfg.d_ffn, cfg.head_dim, cfg.n_heads * cfg.head_dim, cfg.n_kv_heads * cfg.head_dim
    kdim, vdim = cfg.ssm_n_k_heads * cfg.ssm_head_dim, cfg.ssm_n_v_heads * cfg.ssm_head_dim
    conv = 2 * kdim + vdim
    w_bytes = flops_tok = kv_row = rec = attn = 0
    for i in range(cfg.n_layers):
        gdn = cfg.arch == 1 and (i + 1) % cfg.full_attn_interval != 0
        n_in = conv + vdim if gdn else (1 + cfg.attn_out_gate) * nq + 2 * nkv
        k_out = vdim if gdn else nq
        w_bytes += n_in * row_bytes(cfg.wtype, d) + d * row_bytes(cfg.wtype, k_out)
        w_bytes += 2 * f * row_bytes(cfg.wtype, d) + d * row_bytes(cfg.wtype, f)
        flops_tok += 2 * (n_in * d + d * k_out + 3 * f * d)
        if gdn:
            rec += 4 * cfg.ssm_n_v_heads * cfg.ssm_head_dim ** 2
            flops_tok += 8 * cfg.ssm_n_v_heads * cfg.ssm_head_dim ** 2
        else:
            attn += 1
            kv_row += 2 * (row_bytes(GGML_Q8_0, nkv) if cfg.kv_type else 4 * nkv)
    head = cfg.vocab * row_bytes(GGML_Q8_0, d)
    ctx, p, n = case["context"], case["prompt"], case["gen"]
    # one pass over the prompt but its last token, then one token a step; the logits of the last token too
    byts = (w_bytes + kv_row * (ctx + p) + 2 * rec if p > 1 else 0) + (n + 1) * (w_bytes + head + 2 * rec)
    byts += sum(kv_row * (ctx + p + t) for t in range(n + 1))
    flops = (p + n) * flops_tok + (n + 1) * 2 * cfg.vocab * d
    flops += 4 * nq * attn * sum(ctx + t + 1 for t in range(p + n))
    return {"bytes": byts, "flops": flops}


def tolerance(case):
    """Four times the distance from the 64-bit answer that f32 sums of these sizes show."""
    kind = case["kind"]
    if kind == "model":
        # Q8_0 activations sit between the layers: one rounding that falls the other way travels through all
        # that follow (4e-2 between two orders of the attention's sums over 36 random-weight layers)
        return {"rel": 3e-2, "max": 0.3, "differ": 1e-2}
    if kind == "rows":
        return {"rel": 4e-7, "max": 4e-6}      # 5.5e-8
    if kind in ("attn", "attn_prefill"):
        return {"rel": 2e-6, "max": 4e-5}      # 1.7e-7 to 4.8e-7
    return {"rel": 1e-6, "max": 2e-5}          # 8e-8 to 2.1e-7: exact block dots, f32 sums over the blocks


# ---- 64-bit answers ----

def _int8(b):
    return b.contiguous().view(torch.int8).double()


def _dequant(fmt, w, rows, cols):
    """Native blocks -> f64 [rows][cols]."""
    at = 26 if fmt == "ptq1_0" else 0
    d = w[:, at:at + 2].contiguous().view(torch.float16).double()
    if fmt == "q8_0":
        v = _int8(w[:, 2:])
    elif fmt == "ptq1_0":
        b = w.to(torch.int32)
        trit = lambda x, n: ((((x * 3 ** n) & 255) * 3) >> 8).double() - 1.0
        parts = [trit(b[:, 0:16], n) for n in range(5)] + [trit(b[:, 16:24], n) for n in range(5)]
        parts += [trit(b[:, 24:26], n) for n in range(4)]
        v = torch.cat(parts, 1)
    elif fmt in ("q1_0", "q1_0_g128"):
        bits = (w[:, 2:, None] >> torch.arange(8, device="cuda", dtype=torch.uint8)) & 1
        v = bits.reshape(len(w), 128).double() * 2.0 - 1.0
    else:
        codes = (w[:, 2:, None] >> torch.arange(0, 8, 2, device="cuda", dtype=torch.uint8)) & 3
        v = codes.reshape(len(w), 128).double() - 1.0
    return (v * d).reshape(rows, cols)


def _exact_product(case, seed):
    g = _gen(seed)
    fmt, n, k = case.get("fmt", "q8_0"), case["rows"], case["cols"]
    w = _weights(fmt, n, k, g)
    x = _activations(case.get("seq", 1), k, g)
    xd = _dequant("q8_0", x, case.get("seq", 1), k).t().contiguous()
    per = w.shape[0] // n
    y = torch.empty(case.get("seq", 1), n, dtype=torch.float64, device="cuda")
    for r in range(0, n, 8192):
        e = min(n, r + 8192)
        y[:, r:e] = torch.matmul(_dequant(fmt, w[r * per:e * per], e - r, k), xd).t()
    return y if "seq" in case else y[0]


def _exact_attention(case, seed):
    q, k, v = (t.double() for t in _qkv(case, _gen(seed)))
    n, pos0 = case.get("tokens", 1), case.get("pos0", case.get("seq", 1) - 1)
    end, rep = pos0 + n, case["heads"] // case["kv"]
    mask = torch.arange(end, device="cuda")[None, :] > torch.arange(pos0, end, device="cuda")[:, None]
    out = torch.empty_like(q)
    for h in range(case["heads"]):
        kt = k[h // rep, :end].t().contiguous()
        p = torch.matmul(q[:, h].contiguous(), kt) / math.sqrt(case["hd"])
        p = torch.softmax(p.masked_fill(mask, float("-inf")), dim=1)
        out[:, h] = torch.matmul(p, v[h // rep, :end].contiguous())
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "model":
        return None
    if kind in ("gemv", "gemm"):
        return _exact_product(case, seed)
    if kind == "head":
        return {"logits": _exact_product(case, seed), "token": None}
    if kind in ("attn", "attn_prefill"):
        return _exact_attention(case, seed)
    x, w = (t.double() for t in _row_inputs(case, _gen(seed)))
    return {"normed": x * torch.rsqrt(x.square().mean(1, keepdim=True) + 1e-6) * w, "q8": None}
