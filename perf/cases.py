"""The decoder-layer calls of a serving program, as cases to time.

A case is one pass through public operators of `moa_amd.ops` on one model's shapes (hidden 3840, FFN
15360, 262144 vocabulary rows) and M token rows: M = 1 is a decode step, a few rows are a batched or
speculative step, hundreds are a prefill chunk. Kinds:

  layer      a sliding layer's projections: sliding_project_qkv, then O and the GeGLU FFN on one
             residual (sliding_attention_output_feedforward, in the weight format `fmt`). The
             attention output that feeds O is an input of its own, so each result is one block away
             from its inputs.
  full       a full-attention layer's projections: full_project_qkv and full_attention_output
  attention  sliding_attention over the 1024-slot ring cache
  pages      a full-attention layer's attention over `pages` 512-slot cache pages, by full_attention
             or page by page (`paged`) as the reference's runtime calls it
  logits     final_norm_and_logits over the whole vocabulary

Inputs follow the model: unit-variance activations, N(0, 0.02) weights quantised to their format
(FP8 per row, NVFP4 blocks of 16 under a global scale, MXFP4 blocks of 32), norm weights near one,
RoPE tables of both layer types, causal masks of consecutive positions.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "moa-workspace_amd"))
from moa_amd import ops  # noqa: E402

H, L, W = 3840, 15360, 262144
NS, DS, QS, PS, TS = 8, 256, 4096, 2048, 1024  # sliding layers: KV heads, head dim, Q and K/V columns, ring slots
GF, DF, QF, TF = 16, 512, 8192, 512            # full-attention layers: query heads, head dim, Q columns, page slots
E = 32768                                      # RoPE table rows
EPS = 1e-6
DEV = "cuda"


# ------------------------------------------------------------------------------------------ cases

def listed():
    return [
        # the smallest call: one decode token's attention over a partly filled ring
        {"name": "attention_m1", "kind": "attention", "m": 1, "pos": 700},
        # attention of a prefill chunk, the window filling up behind it
        {"name": "attention_m512", "kind": "attention", "m": 512, "pos": 300},
        # one decode token page by page, as the reference's runtime drives a full-attention layer
        {"name": "pages_m1_paged3", "kind": "pages", "m": 1, "pages": 3, "pos": 1300, "paged": True},
        # a prefill chunk's full attention at a few thousand tokens of context
        {"name": "pages_m200_p6", "kind": "pages", "m": 200, "pages": 6, "pos": 2700, "paged": False},
        # a short speculative step at the longest context
        {"name": "pages_m4_p64", "kind": "pages", "m": 4, "pages": 64, "pos": 32700, "paged": False},
        # the decode step's projections with FP8 weights
        {"name": "layer_m1_fp8", "kind": "layer", "m": 1, "fmt": "fp8", "pos": 5000},
        # a batched or speculative step with MXFP4 weights, rows not a multiple of anything
        {"name": "layer_m13_mxfp4", "kind": "layer", "m": 13, "fmt": "mxfp4", "pos": 777},
        # the 256-row prefill chunk with FP8 weights
        {"name": "layer_m256_fp8", "kind": "layer", "m": 256, "fmt": "fp8", "pos": 0},
        # a long ragged prefill chunk with the reference's own operand types (NVFP4, bf16 scales)
        {"name": "layer_m1000_nvfp4", "kind": "layer", "m": 1000, "fmt": "nvfp4", "pos": 24},
        # a prefill chunk's projections of a full-attention layer
        {"name": "full_m300", "kind": "full", "m": 300, "pos": 1124},
        # the decode step's logits
        {"name": "logits_m1", "kind": "logits", "m": 1},
        # logits of a batched or speculative step
        {"name": "logits_m24", "kind": "logits", "m": 24},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def draw(rng):
    kind = rng.choice(["layer", "layer", "full", "attention", "pages", "logits"])
    if kind == "layer":
        m = _log_int(rng, 1, 1000)
        return {"kind": kind, "m": m, "fmt": rng.choice(["fp8", "nvfp4", "mxfp4"]), "pos": rng.randrange(0, 8192)}
    if kind == "full":
        m = _log_int(rng, 1, 500)
        return {"kind": kind, "m": m, "pos": 512 * rng.randrange(0, 60) + rng.randrange(0, TF - m + 1)}
    if kind == "attention":
        return {"kind": kind, "m": _log_int(rng, 1, 512), "pos": rng.randrange(0, 8192)}
    if kind == "pages":
        pages = _log_int(rng, 1, 64)
        m = _log_int(rng, 1, max(1, min(256, 1200 // pages)))
        first = max(0, pages * TF - m - rng.randrange(0, TF))
        return {"kind": kind, "m": m, "pages": pages, "pos": first, "paged": pages <= 16 and m <= 16 and rng.random() < 0.4}
    return {"kind": kind, "m": _log_int(rng, 1, 32)}


# ----------------------------------------------------------------------------------------- inputs

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _normal(g, shape, std=1.0, mean=0.0):
    return torch.randn(shape, generator=g, device=DEV, dtype=torch.float32) * std + mean


def _bf16(g, shape, std=1.0):
    return _normal(g, shape, std).to(torch.bfloat16)


def _rms_weight(g, n):
    return _normal(g, (n,), 0.1, 1.0).to(torch.bfloat16)


def _i32(v):
    return torch.tensor([v], dtype=torch.int32, device=DEV)


def _fp8(g, rows, cols, bf16_scales):
    """E4M3 codes and the per-row scale of an N(0, 0.02) matrix."""
    w = _normal(g, (rows, cols), 0.02)
    s = w.abs().amax(1) / 448.0
    if bf16_scales:
        s = s.to(torch.bfloat16)
    q = (w / s.float()[:, None]).clamp_(-448.0, 448.0).to(torch.float8_e4m3fn)
    return q.view(torch.uint8), s


_E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0)


def _pack_e2m1(x):
    """Nearest E2M1 codes of x, two per byte, the lower element in the low nibble."""
    mids = torch.tensor([(a + b) / 2 for a, b in zip(_E2M1, _E2M1[1:])], device=DEV)
    c = torch.bucketize(x.abs(), mids).to(torch.uint8) | (x < 0).to(torch.uint8) << 3
    c = c.view(x.shape[0], -1, 2)
    return (c[:, :, 0] | c[:, :, 1] << 4).contiguous()


def _unpack_e2m1(p):
    c = torch.stack([p & 15, p >> 4], dim=2).view(p.shape[0], -1).long()
    v = torch.tensor(_E2M1, device=DEV, dtype=torch.float64)[c & 7]
    return torch.where(c >= 8, -v, v)


def _mxfp4(g, rows, cols):
    """E2M1 codes and E8M0 scales per 32 elements."""
    w = _normal(g, (rows, cols), 0.02)
    b = w.view(rows, cols // 32, 32)
    e = torch.floor(torch.log2(b.abs().amax(2).clamp_min(2.0 ** -100))) - 2.0
    packed = _pack_e2m1((b * torch.exp2(-e)[:, :, None]).view(rows, cols))
    return packed, (e + 127.0).to(torch.uint8)


def _nvfp4(g, rows, cols):
    """E2M1 codes, E4M3 scales per 16 elements and the reciprocal global scale."""
    w = _normal(g, (rows, cols), 0.02)
    b = w.view(rows, cols // 16, 16)
    amax = b.abs().amax(2)
    glob = 448.0 * 6.0 / amax.max()
    s = (amax * (glob / 6.0)).clamp_(2.0 ** -6, 448.0).to(torch.float8_e4m3fn)
    packed = _pack_e2m1((b * (glob / s.float())[:, :, None]).view(rows, cols))
    return packed, s.view(torch.uint8), (1.0 / glob).reshape(1).float()


def _rope(head, theta, rotated):
    """cos and sin [E, head] bf16; sin's low half is negated, dims past `rotated` of a head do not turn."""
    i = torch.arange(head // 2, device=DEV, dtype=torch.float64)
    inv = torch.where(i < rotated // 2, theta ** (-2.0 * i / head), torch.zeros_like(i))
    a = torch.arange(E, device=DEV, dtype=torch.float64)[:, None] * inv[None, :]
    cos, sin = torch.cos(a), torch.sin(a)
    return torch.cat([cos, cos], 1).to(torch.bfloat16), torch.cat([-sin, sin], 1).to(torch.bfloat16)


def prepare(case, seed):
    g, m, kind = _gen(seed), case["m"], case["kind"]
    s = {"kind": kind, "m": m}
    if kind == "layer":
        fmt, pos = case["fmt"], case["pos"]
        bf = fmt == "nvfp4"  # the reference's operand types: bf16 scales with NVFP4
        s["fmt"] = fmt
        s["x"], s["attn"], s["residual"] = _bf16(g, (m, H)), _bf16(g, (m, QS)), _bf16(g, (m, H))
        for n, rows, cols in (("q", QS, H), ("k", PS, H), ("v", PS, H), ("o", H, QS)):
            s[n + "_w"], s[n + "_s"] = _fp8(g, rows, cols, bf)
        for n, rows, cols in (("up", L, H), ("gate", L, H), ("down", H, L)):
            if fmt == "fp8":
                s[n + "_w"], s[n + "_s"] = _fp8(g, rows, cols, False)
            elif fmt == "mxfp4":
                s[n + "_w"], s[n + "_s"] = _mxfp4(g, rows, cols)
            else:
                s[n + "_w"], s[n + "_s"], s[n + "_g"] = _nvfp4(g, rows, cols)
        for n, d in (("in_rms", H), ("q_rms", DS), ("k_rms", DS), ("attn_rms", H), ("pre_rms", H), ("post_rms", H)):
            s[n] = _rms_weight(g, d)
        s["scalar"] = torch.full((8,), 0.375, dtype=torch.bfloat16, device=DEV)
        s["cos"], s["sin"] = _rope(DS, 10_000.0, DS)
        s["pos"], s["slot"] = pos, pos % TS
        s["rope_off"], s["kv_off"] = _i32(pos * DS * 2), _i32(pos % TS * NS * DS * 2)
        s["k_cache"], s["v_cache"] = _bf16(g, (TS, NS, DS)), _bf16(g, (TS, NS, DS))
        s["q_out"] = torch.empty((m, NS, 2, DS), dtype=torch.bfloat16, device=DEV)
    elif kind == "full":
        pos = case["pos"]
        s["x"], s["residual"] = _bf16(g, (m, H)), _bf16(g, (m, H))
        for n, rows, cols in (("q", QF, H), ("k", DF, H), ("o", H, QF)):
            s[n + "_w"], s[n + "_s"] = _fp8(g, rows, cols, True)
        for n, d in (("in_rms", H), ("q_rms", DF), ("k_rms", DF), ("attn_rms", H)):
            s[n] = _rms_weight(g, d)
        s["cos"], s["sin"] = _rope(DF, 1_000_000.0, 128)
        s["pos"], s["slot"] = pos, pos % TF
        s["rope_off"], s["kv_off"] = _i32(pos * DF * 2), _i32(pos % TF * DF * 2)
        s["k_page"], s["v_page"] = _bf16(g, (TF, DF)), _bf16(g, (TF, DF))
        s["q_out"] = torch.empty((m, GF, DF), dtype=torch.bfloat16, device=DEV)
        s["attn"] = _bf16(g, (m, GF, DF), 4.0)
        s["sum"] = torch.rand((m, GF), generator=g, device=DEV) * 49.0 + 1.0
    elif kind == "attention":
        pos = case["pos"]
        s["q"] = _bf16(g, (m, NS, 2, DS))
        s["k_cache"], s["v_cache"] = _bf16(g, (TS, NS, DS)), _bf16(g, (TS, NS, DS))
        # slot t holds the newest position p <= pos + m - 1 with p % TS == t; row i sees p <= pos + i
        last = pos + m - 1
        t = torch.arange(TS, device=DEV)
        held = last - (last - t) % TS
        row = pos + torch.arange(m, device=DEV)
        s["mask"] = ((held[None, :] <= row[:, None]) & (held >= 0)[None, :]).float()
        s["out"] = torch.empty((m, NS, 2, DS), dtype=torch.bfloat16, device=DEV)
    elif kind == "pages":
        pages, pos = case["pages"], case["pos"]
        s["paged"], s["pages"] = case["paged"], pages
        s["q"] = _bf16(g, (m, GF, DF))
        s["k_pages"], s["v_pages"] = _bf16(g, (pages, TF, DF)), _bf16(g, (pages, TF, DF))
        t = torch.arange(pages * TF, device=DEV).view(pages, 1, TF)
        s["masks"] = (t <= (pos + torch.arange(m, device=DEV))[None, :, None]).float().contiguous()
        s["max"] = torch.empty((m, GF), dtype=torch.float32, device=DEV)
        s["sum"] = torch.empty((m, GF), dtype=torch.float32, device=DEV)
        s["out"] = torch.empty((m, GF, DF), dtype=torch.bfloat16, device=DEV)
    else:
        s["input"], s["rms"] = _bf16(g, (m, H)), _rms_weight(g, H)
        # the norm's unit rows against a head of this spread give logits that bend under the softcap
        s["head"] = torch.empty((W, H), dtype=torch.bfloat16, device=DEV)
        for r in range(0, W, 32768):
            s["head"][r:r + 32768] = _bf16(g, (32768, H), 0.2)
        s["out"] = torch.empty((m, W), dtype=torch.bfloat16, device=DEV)
    return s


# ------------------------------------------------------------------------------------------- pass

def run(s):
    kind = s["kind"]
    if kind == "layer":
        ops.sliding_project_qkv(s["x"], s["q_w"], s["k_w"], s["v_w"], s["q_s"], s["k_s"], s["v_s"], s["in_rms"],
                                s["q_rms"], s["k_rms"], s["kv_off"], s["rope_off"], s["cos"], s["sin"], s["k_cache"],
                                s["v_cache"], s["q_out"])
        head = (s["attn"], s["attn_rms"], s["o_w"], s["o_s"], s["residual"], s["pre_rms"], s["up_w"], s["gate_w"],
                s["down_w"], s["up_s"], s["gate_s"], s["down_s"])
        if s["fmt"] == "fp8":
            ops.sliding_attention_output_feedforward_fp8(*head, s["post_rms"], s["scalar"])
        elif s["fmt"] == "mxfp4":
            ops.sliding_attention_output_feedforward_mxfp4(*head, s["post_rms"], s["scalar"])
        else:
            ops.sliding_attention_output_feedforward(*head, s["up_g"], s["gate_g"], s["down_g"], s["post_rms"], s["scalar"])
        return {"q": s["q_out"], "k_cache": s["k_cache"], "v_cache": s["v_cache"], "residual": s["residual"]}
    if kind == "full":
        ops.full_project_qkv(s["x"], s["q_w"], s["k_w"], s["q_s"], s["k_s"], s["in_rms"], s["q_rms"], s["k_rms"],
                             s["kv_off"], s["rope_off"], s["cos"], s["sin"], s["k_page"], s["v_page"], s["q_out"])
        ops.full_attention_output(s["attn"], s["sum"], s["attn_rms"], s["o_w"], s["o_s"], s["residual"])
        return {"q": s["q_out"], "k_page": s["k_page"], "v_page": s["v_page"], "residual": s["residual"]}
    if kind == "attention":
        ops.sliding_attention(s["q"], s["k_cache"], s["v_cache"], s["mask"], s["out"])
        return s["out"]
    if kind == "pages":
        if s["paged"]:
            for p in range(s["pages"]):
                call = ops.full_attention_page if p else ops.full_attention_first_page
                call(s["q"], s["k_pages"][p], s["v_pages"][p], s["masks"][p], s["max"], s["sum"], s["out"])
        else:
            ops.full_attention(s["q"], s["k_pages"], s["v_pages"], s["masks"], s["max"], s["sum"], s["out"])
        return {"max": s["max"], "sum": s["sum"], "out": s["out"]}
    ops.final_norm_and_logits(s["input"], s["rms"], s["head"], s["out"])
    return s["out"]


# ------------------------------------------------------------------------------------ what is due

def _ffn_bytes(fmt):
    n = 3 * L * H
    if fmt == "fp8":
        return n + 4 * (2 * L + H)
    return n // 2 + (n // 16 if fmt == "nvfp4" else n // 32)


def work(case):
    m, kind = case["m"], case["kind"]
    if kind == "layer":
        weights = (QS + 2 * PS) * H + H * QS
        scales = (QS + 2 * PS + H) * (2 if case["fmt"] == "nvfp4" else 4)
        rows = m * 2 * (H + QS + 2 * PS + 2 * DS + QS + 2 * H)  # x; q, K and V slots; cos, sin; attention; residual in, out
        return {"bytes": weights + scales + _ffn_bytes(case["fmt"]) + rows + 2 * (4 * H + 2 * DS),
                "flops": 2 * m * (weights + 3 * L * H)}
    if kind == "full":
        weights = (QF + DF) * H + H * QF
        rows = m * (2 * (H + QF + 2 * DF + 2 * DF + QF + 2 * H) + 4 * GF)
        return {"bytes": weights + 2 * (QF + DF + H) + rows + 2 * (2 * H + 2 * DF), "flops": 2 * m * weights}
    if kind == "attention":
        seen = sum(min(TS, case["pos"] + i + 1) for i in range(m))
        slots = min(TS, case["pos"] + m)
        return {"bytes": slots * 2 * 2 * PS + m * (2 * 2 * QS + 4 * TS), "flops": 4 * seen * QS}
    if kind == "pages":
        seen = sum(min(case["pages"] * TF, case["pos"] + i + 1) for i in range(m))
        slots = min(case["pages"] * TF, case["pos"] + m)
        return {"bytes": slots * 2 * 2 * DF + m * (2 * 2 * QF + 8 * GF + 4 * case["pages"] * TF), "flops": 4 * seen * QF}
    return {"bytes": 2 * W * H + m * 2 * (H + W) + 2 * H, "flops": 2 * m * W * H}


def tolerance(case):
    # About four times what the operators are from 64-bit results (layer 0.005, full 0.0037, attention
    # 0.0016, pages 0.0014, logits 0.0027): bf16 results, and the bf16 values a block rounds on its way.
    return {"layer": {"rel": 2e-2}, "full": {"rel": 1.5e-2}, "attention": {"rel": 6e-3}, "pages": {"rel": 6e-3},
            "logits": {"rel": 1.1e-2}}[case["kind"]]


# ---------------------------------------------------------------------------------- in 64 bits

def _d(t):
    return t.to(torch.float64)


def _norm(x):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS)


def _fp8_f64(s, n):
    return _d(s[n + "_w"].view(torch.float8_e4m3fn).float()) * _d(s[n + "_s"])[:, None]


def _ffn_f64(s, n):
    if s["fmt"] == "fp8":
        return _fp8_f64(s, n)
    v = _unpack_e2m1(s[n + "_w"])
    rows, cols = v.shape
    if s["fmt"] == "mxfp4":
        return (v.view(rows, cols // 32, 32) * torch.exp2(_d(s[n + "_s"]) - 127.0)[:, :, None]).view(rows, cols)
    scale = _d(s[n + "_s"].view(torch.float8_e4m3fn).float())
    return (v.view(rows, cols // 16, 16) * scale[:, :, None]).view(rows, cols) * _d(s[n + "_g"])


def _turn(n, cos, sin):
    """RoPE of heads n [m, heads, d] (sin's low half is negated already)."""
    d = n.shape[-1]
    return n * cos[:, None, :] + torch.roll(n, d // 2, -1) * sin[:, None, :]


def _masked(scores, valid):
    scores = scores.masked_fill(~valid, -math.inf)
    top = scores.amax(-1, keepdim=True)
    return top, torch.exp(scores - top)


def exact(case, seed):
    s, m, kind = prepare(case, seed), case["m"], case["kind"]
    if kind in ("layer", "full"):
        rows = s["pos"] + torch.arange(m, device=DEV)
        cos, sin = _d(s["cos"][rows]), _d(s["sin"][rows])
        h = _norm(_d(s["x"])) * _d(s["in_rms"])
        heads, dim = (NS * 2, DS) if kind == "layer" else (GF, DF)
        q = _turn(_norm((h @ _fp8_f64(s, "q").T).view(m, heads, dim)) * _d(s["q_rms"]), cos, sin)
        kv = (NS, DS) if kind == "layer" else (1, DF)
        raw = (h @ _fp8_f64(s, "k").T).view(m, *kv)
        k = _turn(_norm(raw) * _d(s["k_rms"]), cos, sin)
        v = _norm((h @ _fp8_f64(s, "v").T).view(m, *kv)) if kind == "layer" else _norm(raw)
        names = ("k_cache", "v_cache") if kind == "layer" else ("k_page", "v_page")
        out = {"q": q.view(s["q_out"].shape)}
        for n, new in zip(names, (k, v)):
            out[n] = _d(s[n])
            out[n][(s["slot"] + torch.arange(m, device=DEV)) % out[n].shape[0]] = new.view(m, *out[n].shape[1:])
        x = _d(s["attn"]) if kind == "layer" else (_d(s["attn"]) / _d(s["sum"])[:, :, None]).view(m, QF)
        r = _d(s["residual"]) + _norm(x @ _fp8_f64(s, "o").T) * _d(s["attn_rms"])
        if kind == "layer":
            h = _norm(r) * _d(s["pre_rms"])
            up, gate = h @ _ffn_f64(s, "up").T, h @ _ffn_f64(s, "gate").T
            p = torch.nn.functional.gelu(gate, approximate="tanh") * up
            r = (r + _norm(p @ _ffn_f64(s, "down").T) * _d(s["post_rms"])) * _d(s["scalar"][0])
        out["residual"] = r
        return out
    if kind == "attention":
        out = torch.empty(s["out"].shape, dtype=torch.float64, device=DEV)
        for n in range(NS):
            k, v = _d(s["k_cache"][:, n]), _d(s["v_cache"][:, n])
            for j in range(2):
                _, p = _masked(_d(s["q"][:, n, j]) @ k.T, s["mask"] != 0)
                out[:, n, j] = p @ v / p.sum(-1, keepdim=True)
        return out
    if kind == "pages":
        k, v = _d(s["k_pages"]).view(-1, DF), _d(s["v_pages"]).view(-1, DF)
        valid = s["masks"].transpose(0, 1).reshape(m, -1) != 0
        out = {n: torch.empty(s[n].shape, dtype=torch.float64, device=DEV) for n in ("max", "sum", "out")}
        for j in range(GF):
            top, p = _masked(_d(s["q"][:, j]) @ k.T, valid)
            out["max"][:, j], out["sum"][:, j], out["out"][:, j] = top[:, 0], p.sum(-1), p @ v
        return out
    x = _norm(_d(s["input"])) * _d(s["rms"])
    out = torch.empty((m, W), dtype=torch.float64, device=DEV)
    for r in range(0, W, 16384):
        out[:, r:r + 16384] = 30.0 * torch.tanh(x @ _d(s["head"][r:r + 16384]).T / 30.0)
    return out
