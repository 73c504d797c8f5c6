"""Performance cases of the framework's main path, each through public entry
points: whole engine calls (decode, speculative verify, prompts), and the
blocks a program calls by itself (an FFN, prompt and decode attention, a
Gated DeltaNet block, the logits head, the sampling pick, a weight upload).

A case is a dict of plain values:
  kind    decode | verify | prompt | ffn | attn_prompt | attn_decode | gdn |
          gemv | sample | load
  and the sizes of that kind. Weights are random file bytes (GGUF blocks or
  MatMulNBits rows) whose dequantized values are about N(0, 0.02), uploaded
  through the loaders' packers; `exact` dequantizes the same bytes itself
  and computes in float64.
"""
import dataclasses
import math

import numpy as np
import torch

from webgllm_amd import engine as E
from webgllm_amd import ops
from webgllm_amd.delta_layer import LinearAttention

DEV = "cuda"
MODELS = {"llama8b": E.LLAMA3_8B, "qwen2-0.5b": E.QWEN2_05B, "lfm2-1.2b": E.LFM2_12B}
BYTES_PER_WEIGHT = {"q4_0": 18 / 32, "q4_k": 144 / 256, "nbits": 18.5 / 32, "q8_0": 34 / 32,
                    "q6_k": 210 / 256}
# The Gated DeltaNet block: the benchmark's heads (16 of 128) at the width
# of the LFM2 shape, 4 convolution taps.
GDN = {"D": 2048, "H": 16, "dk": 128, "dv": 128, "W": 4}


def listed():
    return [
        # A token of a long chat: the benchmark's own model and context.
        {"name": "decode-llama8b", "kind": "decode", "model": "llama8b", "layers": 32,
         "pos": 4085},
        # Speculative decoding: a token and four drafts, convolution states
        # rolled back.
        {"name": "verify-lfm2", "kind": "verify", "model": "lfm2-1.2b", "layers": 16,
         "pos": 1003, "rows": 5},
        # A long prompt (time to the first token): two layers of the 8B shape
        # and the head, a whole batch of 2048 rows.
        {"name": "prompt-llama8b-2048", "kind": "prompt", "model": "llama8b", "layers": 2,
         "tokens": 2048},
        # A chat turn's prompt on a small ONNX model, an odd number of rows.
        {"name": "prompt-qwen2-131", "kind": "prompt", "model": "qwen2-0.5b", "layers": 24,
         "tokens": 131},
        # One FFN of a 512-row prompt.
        {"name": "ffn-llama8b-512", "kind": "ffn", "fmt": "q4_k", "D": 4096, "F": 14336,
         "rows": 512},
        # One FFN of a short prompt of an 8-bit model.
        {"name": "ffn-lfm2-q8-45", "kind": "ffn", "fmt": "q8_0", "D": 2048, "F": 8192,
         "rows": 45},
        # The attention of a later batch of a long prompt: 2048 rows over
        # 8192 keys.
        {"name": "attn-prompt-8k", "kind": "attn_prompt", "model": "llama8b", "rows": 2048,
         "pos": 6144},
        # A token's attention at a long context.
        {"name": "attn-decode-32k", "kind": "attn_decode", "model": "llama8b", "rows": 1,
         "pos": 32701},
        # A linear-attention block over a prompt, its last chunk ragged.
        {"name": "gdn-prompt-1500", "kind": "gdn", "fmt": "q4_0", "rows": 1500},
        # The logits of a real GGUF file's Q6_K head, one token.
        {"name": "head-q6k", "kind": "gemv", "fmt": "q6_k", "N": 128256, "K": 4096, "rows": 1},
        # The sampled pick of one row.
        {"name": "sample-128k", "kind": "sample", "V": 128256, "rows": 1, "count": 64},
        # Loading a GGUF file: one Q4_K gate|up matrix into the device layout.
        {"name": "load-q4k", "kind": "load", "fmt": "q4_k", "N": 28672, "K": 4096},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "verify", "prompt", "prompt", "ffn", "ffn", "attn_prompt",
                       "attn_decode", "gdn", "gdn", "gemv", "sample", "load"])
    model = rng.choice(sorted(MODELS))
    c = {"kind": kind}
    if kind in ("decode", "verify"):
        c.update(model=model, layers=rng.randint(2, 6 if model == "llama8b" else 16),
                 pos=_log(rng, 1, 4000))
        if kind == "verify":
            c["rows"] = rng.randint(2, 8)
    elif kind == "prompt":
        c.update(model=model, layers=rng.randint(1, 2), tokens=_log(rng, 9, 2048))
    elif kind == "ffn":
        fmt = rng.choice(["q4_0", "q4_k", "nbits", "q8_0"])
        D, F = rng.choice([(896, 4864), (2048, 8192), (4096, 14336), (1024, 4608)])
        if fmt == "q4_k" and D % 256:
            fmt = "nbits"
        c.update(fmt=fmt, D=D, F=F, rows=_log(rng, 9, 2048))
    elif kind == "attn_prompt":
        c.update(model=model, rows=_log(rng, 9, 2048), pos=_log(rng, 1, 6144) - 1)
    elif kind == "attn_decode":
        c.update(model=model, rows=rng.randint(1, 8), pos=_log(rng, 2, 65000))
    elif kind == "gdn":
        c.update(fmt=rng.choice(["q4_0", "q8_0"]), rows=_log(rng, 1, 2048))
    elif kind == "gemv":
        fmt = rng.choice(["q4_0", "q4_k", "nbits", "q8_0", "q6_k"])
        c.update(fmt=fmt, N=4 * _log(rng, 256, 32064), K=256 * rng.randint(4, 32),
                 rows=rng.randint(1, 8))
    elif kind == "sample":
        c.update(V=rng.choice([65536, 128256, 151936, 4 * _log(rng, 5000, 40000) + 1]),
                 rows=rng.randint(1, 5), count=rng.randint(8, 64))
    else:
        c.update(fmt=rng.choice(["q4_0", "q4_k", "nbits", "q8_0", "q6_k"]),
                 N=4 * _log(rng, 256, 8192), K=256 * rng.randint(4, 32))
    return c


# ------------------------------------------------------------ random files

def _gen(seed, salt=0):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed * 1000003 + salt)
    return g


def _bytes(n, g):
    return torch.empty(n, dtype=torch.uint8, device=DEV).random_(0, 256, generator=g)


def _halves(n, lo, hi, g):
    return torch.empty(n, device=DEV).uniform_(lo, hi, generator=g).half()


def _raw(fmt, N, K, g):
    """A matrix as a file holds it: device bytes (MatMulNBits: quants, half
    scales, zero points)."""
    if fmt == "q4_0":
        b = _bytes(N * K // 32 * 18, g).view(-1, 18)
        b[:, 0:2] = _halves(b.shape[0], 0.003, 0.006, g).view(torch.uint8).view(-1, 2)
        return b.view(-1)
    if fmt == "q4_k":
        # the mins near 7.5 scales, as quantized zero-mean weights have them
        S = N * K // 256
        b = _bytes(S * 144, g).view(-1, 144)
        d = _halves(S, 0.7e-4, 1.3e-4, g)
        b[:, 0:2] = d.view(torch.uint8).view(-1, 2)
        b[:, 2:4] = (d.float() * 7.5).half().view(torch.uint8).view(-1, 2)
        sc = torch.randint(24, 64, (S, 8), generator=g, device=DEV)
        mn = (sc + torch.randint(-3, 4, (S, 8), generator=g, device=DEV)).clamp_(0, 63)
        b[:, 4:8] = (sc[:, :4] | ((sc[:, 4:] >> 4) << 6)).to(torch.uint8)
        b[:, 8:12] = (mn[:, :4] | ((mn[:, 4:] >> 4) << 6)).to(torch.uint8)
        b[:, 12:16] = ((sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)).to(torch.uint8)
        return b.view(-1)
    if fmt == "nbits":
        B = K // 32
        quant = _bytes(N * B * 16, g)
        scales = _halves(N * B, 0.003, 0.006, g)
        z = torch.randint(6, 10, (N, B + B % 2), generator=g, device=DEV, dtype=torch.uint8)
        return quant, scales, (z[:, 0::2] | (z[:, 1::2] << 4)).contiguous().view(-1)
    if fmt == "q8_0":
        b = _bytes(N * K // 32 * 34, g).view(-1, 34)
        b[:, 0:2] = _halves(b.shape[0], 1.8e-4, 3.6e-4, g).view(torch.uint8).view(-1, 2)
        return b.view(-1)
    b = _bytes(N * K // 256 * 210, g).view(-1, 210)  # q6_k
    b[:, 208:210] = _halves(b.shape[0], 1.0e-5, 2.0e-5, g).view(torch.uint8).view(-1, 2)
    return b.view(-1)


def _upload(fmt, raw, N, K, order=None):
    src_rows = None if order is None else torch.tensor(order, dtype=torch.int32, device=DEV)
    if fmt == "q4_0":
        m = ops.Q4Matrix.from_q4_0(raw, N, K, src_rows=src_rows)
    elif fmt == "q4_k":
        m = ops.Q4Matrix.from_q4_k(raw, N, K, native=False, src_rows=src_rows, records=True)
        m.prompt_desc()
    elif fmt == "nbits":
        m = ops.Q4Matrix.from_nbits(raw[0], raw[1].view(torch.uint8), raw[2], N, K,
                                    src_rows=src_rows)
    elif fmt == "q8_0":
        m = ops.Q4Matrix.from_q8_0(raw, N, K, src_rows=src_rows)
    else:
        m = ops.Q4Matrix.from_q6_k(raw, N, K, src_rows=src_rows)
    m.row_order = order
    return m


def _dense(fmt, raw, N, K):
    """The file's weights in float64 [N, K]."""
    f64 = torch.float64
    if fmt in ("q4_0", "q8_0"):
        b = raw.view(-1, 18 if fmt == "q4_0" else 34)
        d = b[:, 0:2].contiguous().view(torch.float16).to(f64)
        if fmt == "q8_0":
            q = b[:, 2:].contiguous().view(torch.int8).to(f64)
        else:
            q = torch.cat([b[:, 2:] & 15, b[:, 2:] >> 4], 1).to(f64) - 8
        return (d * q).view(N, K)
    if fmt == "q4_k":
        b = raw.view(-1, 144)
        dd = b[:, 0:4].contiguous().view(torch.float16).to(f64)
        s = b[:, 4:16].to(torch.int64)
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1).to(f64)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).to(f64)
        q = b[:, 16:].view(-1, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], 2).view(-1, 8, 32).to(f64)
        w = (dd[:, 0:1] * sc)[:, :, None] * q - (dd[:, 1:2] * mn)[:, :, None]
        return w.view(N, K)
    if fmt == "nbits":
        quant, scales, zp = raw
        B = K // 32
        q = quant.view(N, B, 16, 1)
        q = torch.cat([q & 15, q >> 4], 3).view(N, B, 32).to(f64)
        z = zp.view(N, -1, 1)
        z = torch.cat([z & 15, z >> 4], 2).view(N, -1)[:, :B].to(f64)
        return (scales.view(N, B, 1).to(f64) * (q - z[:, :, None])).view(N, K)
    b = raw.view(-1, 210)  # q6_k
    d = b[:, 208:210].contiguous().view(torch.float16).to(f64)
    sc = b[:, 192:208].contiguous().view(torch.int8).to(f64)
    ql = b[:, :128].view(-1, 2, 2, 32).to(torch.int64)
    qh = b[:, 128:192].view(-1, 2, 32).to(torch.int64)
    parts = [(ql[:, :, 0] & 15) | ((qh & 3) << 4), (ql[:, :, 1] & 15) | (((qh >> 2) & 3) << 4),
             (ql[:, :, 0] >> 4) | (((qh >> 4) & 3) << 4), (ql[:, :, 1] >> 4) | ((qh >> 6) << 4)]
    q = torch.stack(parts, 2).view(-1, 16, 16).to(f64) - 32
    return (d[:, :, None] * sc[:, :, None] * q).view(N, K)


# ------------------------------------------------------------ whole models

def _shape(c):
    s = MODELS[c["model"]]
    return dataclasses.replace(s, layers=c["layers"],
                               conv_layers=tuple(i for i in s.conv_layers if i < c["layers"]))


def _shown(s):
    """The layers whose updated states are returned beside the logits: all of
    them, or every second one of a deep model."""
    return range(0, s.layers, 1 if s.layers <= 24 else 2)


def _fmt(s):
    return {"q4_k_records": "q4_k"}.get(s.fmt, s.fmt)


def _norm_w(n, g):
    return 1.0 + 0.1 * torch.randn(n, generator=g, device=DEV)


def _layer_parts(s, i, seed):
    """Layer i's vectors and raw matrices {name: tensor or (raw, N, K)}."""
    g, f = _gen(seed, 10 + i), _fmt(s)
    D, F, A = s.hidden, s.intermediate, s.heads * s.head_dim
    p = {"op_norm": _norm_w(D, g), "ffn_norm": _norm_w(D, g),
         "gate_up": (_raw(f, 2 * F, D, g), 2 * F, D), "down": (_raw(f, D, F, g), D, F)}
    if s.layer_type(i) == "conv":
        p["in_proj"] = (_raw(f, 3 * D, D, g), 3 * D, D)
        p["out_proj"] = (_raw(f, D, D, g), D, D)
        p["taps"] = (torch.randn((D, s.conv_kernel), generator=g, device=DEV) * 0.5).contiguous()
    else:
        p["qkv"] = (_raw(f, s.qkv_rows, D, g), s.qkv_rows, D)
        p["o"] = (_raw(f, D, A, g), D, A)
        if s.qk_norm:
            p["q_norm"], p["k_norm"] = _norm_w(s.head_dim, g), _norm_w(s.head_dim, g)
    return p


def _embedding_parts(s, seed):
    g = _gen(seed, 1)
    return (_raw(_fmt(s), s.vocab, s.hidden, g), s.vocab, s.hidden), _norm_w(s.hidden, g)


def _cache_parts(s, pos, seed, i):
    """Layer i's cached keys and values [pos, kv_heads * head_dim] halves."""
    g = _gen(seed, 1000 + i)
    n = s.kv_heads * s.head_dim
    return (torch.randn((pos, n), generator=g, device=DEV).half(),
            torch.randn((pos, n), generator=g, device=DEV).half())


def _conv_parts(s, seed, i):
    g = _gen(seed, 2000 + i)
    return torch.randn((s.conv_kernel - 1, s.hidden), generator=g, device=DEV)


def _tokens(c, s, seed):
    n = c.get("tokens") or c.get("rows") or 1
    return np.random.default_rng(seed).integers(0, s.vocab, n).tolist()


def _weights(s, seed):
    f = _fmt(s)
    orders = {"gate_up": E.gate_up_row_order(s.intermediate),
              "qkv": E.qkv_row_order(s) if s.rope_in_epilogue else None}
    w = E.Weights.blank(s, device=DEV)
    (raw, N, K), w.final_norm = _embedding_parts(s, seed)
    w.embedding = _upload(f, raw, N, K)
    for i in range(s.layers):
        lw = {}
        for name, v in _layer_parts(s, i, seed).items():
            lw[name] = _upload(f, *v, order=orders.get(name)) if isinstance(v, tuple) else v
        w.layers.append(lw)
    return w


def _model_state(c, seed):
    s = _shape(c)
    pos = c.get("pos", 0)
    toks = _tokens(c, s, seed)
    n = pos + len(toks)
    eng = E.Engine(_weights(s, seed), max(n, min(4096, n + 64)))
    st = {"case": c, "eng": eng, "toks": toks, "pos": pos}
    if c["kind"] == "prompt":
        return st
    eng.reserve(n)
    saved, out = [], []
    for i in range(s.layers):
        if s.layer_type(i) == "conv":
            eng.state[i].copy_(_conv_parts(s, seed, i))
            saved.append(eng.state[i].clone())
        else:
            for cache, part in zip((eng.k_cache[i], eng.v_cache[i]),
                                   _cache_parts(s, pos, seed, i)):
                cache[:pos].copy_(part)
    eng.position = pos
    if c["kind"] == "decode":
        eng.capture_step(toks[0])
    else:
        eng.capture_verify(len(toks))
    for i in _shown(s):
        if s.layer_type(i) == "conv":
            out.append(eng.state[i])
        else:
            out += [eng.k_cache[i][pos:n], eng.v_cache[i][pos:n]]
    st["states"] = [eng.state[i] for i in sorted(eng.state)]
    st["saved"] = saved
    st["out"] = [eng.logits[:len(toks)]] + out
    return st


def _run_model(st):
    c, eng = st["case"], st["eng"]
    if c["kind"] == "prompt":  # a new conversation
        eng.reset()
        eng.forward(st["toks"])
        T = len(st["toks"])
        out = [eng.logits[:T % 8 or 8]]
        for i in _shown(eng.shape):
            if i in eng.state:
                out.append(eng.state[i])
            else:
                out += [eng.k_cache[i][:T], eng.v_cache[i][:T]]
        return out
    if st["states"]:  # the sequence's states before this token
        torch._foreach_copy_(st["states"], st["saved"])
    eng.position = st["pos"]
    if c["kind"] == "decode":
        eng.decode(st["toks"][0], 1)
    else:
        eng.verify_drafts(st["toks"][0], [st["toks"][1:]])
    return st["out"]


# --- float64

def _rms64(x, w, eps):
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + eps) * w.double()


def _rope64(x, pos, theta):
    """x [rows, heads, hd] rotated at positions pos [rows]: pairs (j, j + hd/2)."""
    half = x.shape[-1] // 2
    freq = theta ** (-2.0 * torch.arange(half, dtype=torch.float64, device=DEV) / (2 * half))
    ang = pos[:, None, None].double() * freq
    a, b = x[..., :half], x[..., half:]
    co, si = torch.cos(ang), torch.sin(ang)
    return torch.cat([a * co - b * si, b * co + a * si], -1)


def _attend64(q, k, v, pos0, kv):
    """q [M, H, hd] over keys k, v [n, kv, hd]; row m sees keys 0 .. pos0 + m."""
    M, H, hd = q.shape
    n, G = k.shape[0], H // kv
    keys = torch.arange(n, device=DEV)
    out = torch.empty_like(q)
    for r0 in range(0, M, 512):
        r1 = min(M, r0 + 512)
        hidden = keys[None, :] > pos0 + torch.arange(r0, r1, device=DEV)[:, None]
        for h in range(H):
            sc = q[r0:r1, h] @ k[:, h // G].T / math.sqrt(hd)
            sc.masked_fill_(hidden, -math.inf)
            out[r0:r1, h] = torch.softmax(sc, 1) @ v[:, h // G]
    return out.reshape(M, H * hd)


def _heads64(qkv, s, pos0, q_norm, k_norm, eps):
    """Prepared queries, keys and values of qkv rows [M, qkv_rows]."""
    M, hd = qkv.shape[0], s.head_dim
    x = qkv.view(M, s.heads + 2 * s.kv_heads, hd)
    q, k, v = x.split([s.heads, s.kv_heads, s.kv_heads], 1)
    if q_norm is not None:
        q, k = _rms64(q, q_norm, eps), _rms64(k, k_norm, eps)
    pos = pos0 + torch.arange(M, device=DEV)
    return _rope64(q, pos, s.rope_theta), _rope64(k, pos, s.rope_theta), v


def _exact_model(c, seed):
    s, f = _shape(c), _fmt(_shape(c))
    toks, pos = _tokens(c, s, seed), c.get("pos", 0)
    M, kvd = len(toks), s.kv_heads * s.head_dim
    (raw, N, K), final_norm = _embedding_parts(s, seed)
    emb = _dense(f, raw, N, K)
    h = emb[torch.tensor(toks, device=DEV)]
    out = []
    for i in range(s.layers):
        p = _layer_parts(s, i, seed)
        W = lambda name: _dense(f, *p[name]).T  # noqa: E731
        x = _rms64(h, p["op_norm"], s.eps)
        if s.layer_type(i) == "conv":
            B, C, xx = (x @ W("in_proj")).split(s.hidden, 1)
            st = _conv_parts(s, seed, i).double() if c["kind"] != "prompt" else \
                torch.zeros((s.conv_kernel - 1, s.hidden), dtype=torch.float64, device=DEV)
            y = torch.cat([st, B * xx])
            z = sum(p["taps"][:, t].double() * y[t:t + M] for t in range(s.conv_kernel))
            h = h + (C * z) @ W("out_proj")
            # random drafts: a verify keeps its first row only
            kept = 1 if c["kind"] == "verify" else M
            rows = [y[kept:kept + s.conv_kernel - 1]]
        else:
            q, k, v = _heads64(x @ W("qkv"), s, pos, p.get("q_norm"), p.get("k_norm"), s.eps)
            ks, vs = k, v
            if pos:
                ck, cv = (t.double().view(pos, s.kv_heads, s.head_dim)
                          for t in _cache_parts(s, pos, seed, i))
                ks, vs = torch.cat([ck, k]), torch.cat([cv, v])
            h = h + _attend64(q, ks, vs, pos, s.kv_heads) @ W("o")
            rows = [k.reshape(M, kvd), v.reshape(M, kvd)]
        out += rows if i in _shown(s) else []
        g, u = (_rms64(h, p["ffn_norm"], s.eps) @ W("gate_up")).split(s.intermediate, 1)
        h = h + (torch.nn.functional.silu(g) * u) @ W("down")
    if c["kind"] == "prompt":
        h = h[-(M % 8 or 8):]
    return [_rms64(h, final_norm, s.eps) @ emb.T] + out


# ------------------------------------------------------------------ blocks

def _ffn_parts(c, seed):
    g, D, F = _gen(seed), c["D"], c["F"]
    return {"h": torch.randn((c["rows"], D), generator=g, device=DEV), "w": _norm_w(D, g),
            "gate_up": (_raw(c["fmt"], 2 * F, D, g), 2 * F, D),
            "down": (_raw(c["fmt"], D, F, g), D, F)}


def _attn_parts(c, seed):
    s, g = MODELS[c["model"]], _gen(seed)
    M, n = c["rows"], c["pos"] + c["rows"]
    p = {"k": torch.randn((n, s.kv_heads * s.head_dim), generator=g, device=DEV).half(),
         "v": torch.randn((n, s.kv_heads * s.head_dim), generator=g, device=DEV).half()}
    if c["kind"] == "attn_decode":
        p["q"] = torch.randn((M, s.heads * s.head_dim), generator=g, device=DEV) \
            / math.sqrt(s.head_dim)
    else:
        p["qkv"] = torch.randn((M, s.qkv_rows), generator=g, device=DEV)
        if s.qk_norm:
            p["q_norm"], p["k_norm"] = _norm_w(s.head_dim, g), _norm_w(s.head_dim, g)
    return s, p


def _gdn_parts(c, seed):
    g, f = _gen(seed), c["fmt"]
    D, H, dk, dv, W = (GDN[k] for k in ("D", "H", "dk", "dv", "W"))
    C = 2 * H * dk + H * dv
    rn = lambda *n: torch.randn(n, generator=g, device=DEV)  # noqa: E731
    return {"x": rn(c["rows"], D).half(), "in": (_raw(f, C + H * dv, D, g), C + H * dv, D),
            "ba": (_raw(f, 2 * H, D, g), 2 * H, D),
            "out": (_raw(f, D, H * dv, g), D, H * dv), "taps": (rn(C, W) * 0.5).contiguous(),
            "A": -torch.exp(rn(H) * 0.5), "dt": rn(H) * 0.5, "norm": _norm_w(dv, g),
            "conv": rn(W - 1, C), "state": rn(H, dk, dv) * 0.1}


def _sample_parts(c, seed):
    g = _gen(seed)
    mask = torch.zeros(c["V"], dtype=torch.uint8, device=DEV)
    mask[torch.randint(0, c["V"], (64,), device=DEV, generator=g)] = 1
    return torch.randn((c["rows"], c["V"]), generator=g, device=DEV) * 3, mask


def _x16(c, seed):
    return torch.randn((c["rows"], c["K"]), generator=_gen(seed, 5), device=DEV).half()


def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind in ("decode", "verify", "prompt"):
        return _model_state(c, seed)
    st = {"case": c}
    if kind == "ffn":
        p = _ffn_parts(c, seed)
        st.update(h=p["h"], w=p["w"], down=_upload(c["fmt"], *p["down"]),
                  gate_up=_upload(c["fmt"], *p["gate_up"], order=E.gate_up_row_order(c["F"])),
                  x16=torch.empty((c["rows"], c["D"]), dtype=torch.float16, device=DEV),
                  rs=torch.empty(c["rows"], device=DEV))
    elif kind in ("attn_prompt", "attn_decode"):
        s, p = _attn_parts(c, seed)
        st.update(p, shape=ops.attn_shape(s.heads, s.kv_heads, s.head_dim, s.head_dim, s.eps,
                                          s.qk_norm),
                  pos0=torch.tensor([c["pos"]], dtype=torch.int32, device=DEV),
                  rope=E._rope_table(s.rope_theta, s.head_dim, c["pos"] + c["rows"]).to(DEV))
        if kind == "attn_decode":
            st["scratch"] = ops.attn_scratch(c["rows"], st["shape"], p["k"].shape[0])
    elif kind == "gdn":
        p, f = _gdn_parts(c, seed), c["fmt"]
        blk = LinearAttention(_upload(f, *p["in"]), _upload(f, *p["ba"]), _upload(f, *p["out"]),
                              p["taps"], p["A"], p["dt"], p["norm"], GDN["H"], GDN["dk"],
                              GDN["dv"])
        st.update(blk=blk, x=p["x"], conv=p["conv"], state=p["state"])
    elif kind == "gemv":
        st.update(x=_x16(c, seed),
                  m=_upload(c["fmt"], _raw(c["fmt"], c["N"], c["K"], _gen(seed)), c["N"], c["K"]))
    elif kind == "sample":
        st["logits"], st["mask"] = _sample_parts(c, seed)
    else:
        st["raw"] = _raw(c["fmt"], c["N"], c["K"], _gen(seed))
    return st


def run(state):
    st, c = state, state["case"]
    kind = c["kind"]
    if kind in ("decode", "verify", "prompt"):
        return _run_model(st)
    if kind == "ffn":
        ops.norm_to_h2(st["h"], st["w"], 1e-5, st["x16"], st["rs"])
        ff = ops.gemm_swiglu(st["gate_up"], st["x16"], row_scale=st["rs"])
        return ops.gemm(st["down"], ff, residual=st["h"])
    if kind == "attn_prompt":
        q = ops.head_prep(st["qkv"], st["shape"], st["rope"], st["pos0"], st["k"], st["v"],
                          st.get("q_norm"), st.get("k_norm"))
        att = ops.attn_prefill(q, st["shape"], st["k"], st["v"], st["pos0"])
        return [att, st["k"], st["v"]]
    if kind == "attn_decode":
        return ops.attn_decode(st["q"], st["shape"], st["k"], st["v"], st["pos0"],
                               scratch=st["scratch"])
    if kind == "gdn":
        blk = st["blk"]
        blk.state.copy_(st["state"])  # the sequence's states before these rows
        blk.conv_state[0].copy_(st["conv"])
        return [blk.forward(st["x"]), blk.state, blk.conv_state[0]]
    if kind == "gemv":
        return ops.gemv(st["m"], st["x"])
    if kind == "sample":
        return ops.pick_candidates(st["logits"], c["count"], mask=st["mask"], penalty=1.1,
                                   presence_penalty=0.2)
    m = _upload(c["fmt"], st["raw"], c["N"], c["K"])
    return [t for t in (m.quants, m.scales, m.zeros) if t is not None]


# ------------------------------------------------------------ exact results

def _exact_gdn(c, seed):
    p, f = _gdn_parts(c, seed), c["fmt"]
    H, dk, dv, W, M = GDN["H"], GDN["dk"], GDN["dv"], GDN["W"], c["rows"]
    C = 2 * H * dk + H * dv
    x = p["x"].double()
    proj, ba = x @ _dense(f, *p["in"]).T, x @ _dense(f, *p["ba"]).T
    rows = torch.cat([p["conv"].double(), proj[:, :C]])
    qkv = torch.nn.functional.silu(sum(p["taps"][:, t].double() * rows[t:t + M]
                                       for t in range(W)))
    q, k, v = qkv.split([H * dk, H * dk, H * dv], 1)
    q, k, v = q.view(M, H, dk), k.view(M, H, dk), v.view(M, H, dv)
    q = q / torch.sqrt(q.square().sum(-1, keepdim=True) + 1e-6) / math.sqrt(dk)
    k = k / torch.sqrt(k.square().sum(-1, keepdim=True) + 1e-6)
    beta = torch.sigmoid(ba[:, :H])
    decay = torch.exp(p["A"].double() * torch.nn.functional.softplus(ba[:, H:]
                                                                     + p["dt"].double()))
    S = p["state"].double()
    o = torch.empty((M, H, dv), dtype=torch.float64, device=DEV)
    for m in range(M):
        S = S * decay[m, :, None, None]
        d = beta[m, :, None] * (v[m] - (S * k[m, :, :, None]).sum(1))
        S = S + k[m, :, :, None] * d[:, None, :]
        o[m] = (S * q[m, :, :, None]).sum(1)
    z = torch.nn.functional.silu(proj[:, C:]).view(M, H, dv)
    y = (_rms64(o, p["norm"], 1e-6) * z).view(M, H * dv)
    return [y @ _dense(f, *p["out"]).T, S, rows[M:]]


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind in ("decode", "verify", "prompt"):
        return _exact_model(c, seed)
    if kind == "ffn":
        p, f = _ffn_parts(c, seed), c["fmt"]
        h = p["h"].double()
        g, u = (_rms64(h, p["w"], 1e-5) @ _dense(f, *p["gate_up"]).T).split(c["F"], 1)
        return h + (torch.nn.functional.silu(g) * u) @ _dense(f, *p["down"]).T
    if kind in ("attn_prompt", "attn_decode"):
        s, p = _attn_parts(c, seed)
        k, v = (p[t].double().view(-1, s.kv_heads, s.head_dim) for t in "kv")
        if kind == "attn_decode":  # queries come scaled
            q = p["q"].double().view(-1, s.heads, s.head_dim) * math.sqrt(s.head_dim)
            return _attend64(q, k, v, c["pos"], s.kv_heads)
        q, kn, vn = _heads64(p["qkv"].double(), s, c["pos"], p.get("q_norm"), p.get("k_norm"),
                             s.eps)
        k, v = torch.cat([k[:c["pos"]], kn]), torch.cat([v[:c["pos"]], vn])
        n = k.shape[0]
        return [_attend64(q, k, v, c["pos"], s.kv_heads), k.reshape(n, -1), v.reshape(n, -1)]
    if kind == "gdn":
        return _exact_gdn(c, seed)
    if kind == "gemv":
        raw = _raw(c["fmt"], c["N"], c["K"], _gen(seed))
        return _x16(c, seed).double() @ _dense(c["fmt"], raw, c["N"], c["K"]).T
    return None  # a pick of given logits, bytes: compared as they are


# ---------------------------------------------------------- work, tolerance

def work(case):
    c, kind = case, case["kind"]
    if kind in ("decode", "verify", "prompt"):
        s = _shape(c)
        M, pos = c.get("tokens") or c.get("rows") or 1, c.get("pos", 0)
        T = (M % 8 or 8) if kind == "prompt" else M
        bpw, D, A = BYTES_PER_WEIGHT[_fmt(s)], s.hidden, s.heads * s.head_dim
        per = flops = byts = 0
        for i in range(s.layers):
            n = 3 * s.intermediate * D
            if s.layer_type(i) == "conv":
                n += 4 * D * D
                byts += 2 * 4 * (s.conv_kernel - 1) * D
                flops += 2 * M * D * (s.conv_kernel + 2)
            else:
                n += s.qkv_rows * D + A * D
                byts += (pos + 2 * M) * 2 * s.kv_heads * s.head_dim * 2
                flops += 4 * A * (M * pos + M * (M + 1) // 2)
            per += n
        flops += 2 * M * per + 2 * T * s.vocab * D
        byts += (per + s.vocab * D) * bpw + 4 * T * s.vocab
        return {"bytes": int(byts), "flops": int(flops)}
    if kind == "ffn":
        n = 3 * c["D"] * c["F"]
        return {"bytes": int(n * BYTES_PER_WEIGHT[c["fmt"]] + 8 * c["rows"] * c["D"]),
                "flops": 2 * c["rows"] * n}
    if kind in ("attn_prompt", "attn_decode"):
        s, M, pos = MODELS[c["model"]], c["rows"], c["pos"]
        A, kv = s.heads * s.head_dim, s.kv_heads * s.head_dim
        if kind == "attn_decode":
            return {"bytes": (pos + M) * 2 * kv * 2 + M * A * 6, "flops": 4 * A * M * (pos + M)}
        return {"bytes": pos * 2 * kv * 2 + M * (4 * s.qkv_rows + 2 * 2 * kv + 2 * A),
                "flops": 4 * A * (M * pos + M * (M + 1) // 2)}
    if kind == "gdn":
        D, H, dk, dv = GDN["D"], GDN["H"], GDN["dk"], GDN["dv"]
        n = (2 * H * dk + 2 * H * dv + 2 * H + H * dv) * D
        return {"bytes": int(n * BYTES_PER_WEIGHT[c["fmt"]] + c["rows"] * D * 6
                             + 8 * H * dk * dv),
                "flops": c["rows"] * (2 * n + 6 * H * dk * dv)}
    if kind == "gemv":
        return {"bytes": int(c["N"] * c["K"] * BYTES_PER_WEIGHT[c["fmt"]]
                             + c["rows"] * (2 * c["K"] + 4 * c["N"])),
                "flops": 2 * c["rows"] * c["N"] * c["K"]}
    if kind == "sample":
        return {"bytes": c["rows"] * (4 * c["V"] + 1028 * c["count"]) + c["V"],
                "flops": c["rows"] * c["V"]}
    n = c["N"] * c["K"]
    return {"bytes": int(2 * n * BYTES_PER_WEIGHT[c["fmt"]]), "flops": n}


def tolerance(case):
    """Two to five times the distance from float64 measured over these sizes.
    Half activations and float32 sums: FFNs 1.5e-4 to 9.1e-4, DeltaNet blocks
    1.9e-4 to 4.9e-4, attention 2.0e-4 to 3.3e-4 (half outputs and caches),
    GEMVs 1e-7 to 6e-6 (exact products), with Q4_K's half-rounded block
    scales 4e-4 to 4.8e-4; a whole model carries each layer's rounding through the
    next: 3e-4 to 4e-3, 9.6e-3 after 32 layers of Q4_K."""
    kind = case["kind"]
    if kind in ("sample", "load"):
        return "exact"
    if kind in ("decode", "verify", "prompt"):
        return {"rel": 2e-2}
    if kind in ("attn_prompt", "attn_decode"):
        return {"rel": 1.2e-3}
    if kind == "gemv":
        return {"rel": 1.6e-3 if case["fmt"] == "q4_k" else 2.5e-5}
    return {"rel": 4e-3 if kind == "ffn" else 2e-3}
