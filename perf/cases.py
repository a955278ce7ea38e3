"""The measured work of this framework: its linears, paged attention, Gated DeltaNet and MoE operators and one whole
layer, through the axk package, at the sizes of the repository's own configurations (axk/configs.py) and of the
ranges around them.

A case is a dict of plain values whose "kind" names the operator:
  linear        one MX / FP8 runtime-weight projection, 1 row (a decode step) to 4096 rows (a prefill chunk)
  paged_decode  one token per sequence over a paged KV cache (bf16, FP8 or INT8)
  paged_prefill a chunk of new tokens per sequence over its paged history and itself
  gdn_decode    the Gated DeltaNet recurrence, 1 token (decode) or a few (speculative drafts) per sequence
  gdn_prefill   the chunked Gated DeltaNet over a prompt
  moe           the MoE layer: router, top-k, shared expert, routed MXFP4 experts, combine
  attn_verify   a whole attention layer over speculative draft rows: norms, FP8 projections, RoPE, KV write, paged
                attention, output gate, MXFP4 MLP
"""
import math
import os
import random

import sys

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for _p in (_ROOT, os.path.join(_ROOT, "ax-dsl-kernels_amd")):
    if _p not in sys.path:
        sys.path.insert(0, _p)

import torch  # noqa: E402

import axk  # noqa: E402
from axk import layer  # noqa: E402

DEV = "cuda:0"
F64 = torch.float64
# The 35B's MoE block (hidden 2048, 256 routed experts of 512 and one shared expert of 512, top-8).
MOE = {"hidden": 2048, "experts": 256, "inter": 512, "top_k": 8}
# The hybrid decode group's attention layer (hidden 4096, 32 query / 4 KV heads of 256, MLP 12288, rotary 64).
LAYER = {"hidden": 4096, "inter": 12288, "hq": 32, "hkv": 4, "d": 256, "rot": 64, "page": 64, "theta": 1e7}


def listed():
    return [
        # The smallest call: one decode token through one MXFP4 projection, bound by launch and latency.
        {"name": "linear_decode1", "kind": "linear", "fmt": "mxfp4", "m": 1, "n": 4096, "k": 4096, "out": "bf16"},
        # The LM head over a decode batch of 32 sequences: the largest weight a step reads, fp32 logits.
        {"name": "lm_head_b32", "kind": "linear", "fmt": "mxfp4", "m": 32, "n": 248320, "k": 2048, "out": "f32"},
        # A projection over a full prefill chunk of 4096 tokens: a dense matrix product.
        {"name": "linear_prefill4096", "kind": "linear", "fmt": "mxfp4", "m": 4096, "n": 4096, "k": 4096,
         "out": "bf16"},
        # A serving step's decode attention: 16 sequences of 1024 to 16384 tokens, bf16 cache.
        {"name": "paged_decode_b16", "kind": "paged_decode", "kv": "bf16", "batch": 16, "lo": 1024, "hi": 16384,
         "hq": 16, "hkv": 2, "d": 256, "page": 64},
        # One 256-token prefill page of a long prompt: few query rows against 16000 tokens of history.
        {"name": "paged_prefill_page256", "kind": "paged_prefill", "batch": 1, "new": 256, "hist": 16000, "hq": 16,
         "hkv": 2, "d": 256, "page": 64},
        # The first 4096-token chunk of a prompt: causal attention with no history.
        {"name": "paged_prefill_4096", "kind": "paged_prefill", "batch": 1, "new": 4096, "hist": 0, "hq": 16,
         "hkv": 2, "d": 256, "page": 64},
        # The GDN state update of a decode step at 32 sequences.
        {"name": "gdn_decode_b32", "kind": "gdn_decode", "batch": 32, "tokens": 1, "nk": 16, "nv": 32},
        # The GDN scan over a 4096-token prompt chunk.
        {"name": "gdn_prefill_4096", "kind": "gdn_prefill", "batch": 1, "tokens": 4096, "nk": 16, "nv": 32},
        # The MoE layer at a decode batch of 32 sequences.
        {"name": "moe_decode32", "kind": "moe", "tokens": 32},
        # The MoE layer over one 256-token prefill page.
        {"name": "moe_page256", "kind": "moe", "tokens": 256},
        # The MoE layer over a 4096-token prefill chunk: the largest case.
        {"name": "moe_prefill4096", "kind": "moe", "tokens": 4096},
        # A whole attention layer verifying 4 draft rows for each of 4 sequences of uneven context.
        {"name": "attn_verify_b4t4", "kind": "attn_verify", "batch": 4, "tokens": 4, "lo": 1024, "hi": 16384},
    ]


def _log(rng, lo, hi):
    """An integer spread over [lo, hi] by its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "paged_decode", "paged_prefill", "gdn_decode", "gdn_prefill", "moe", "moe",
                       "attn_verify"])
    if kind == "linear":
        n, k = rng.choice([(4096, 4096), (8192, 2048), (2048, 4096), (16384, 4096), (12288, 4096), (4096, 12288),
                           (1024, 2048), (3080, 1504)])
        m = _log(rng, 1, min(4096, int(1.3e11 / (2 * n * k))))
        return {"kind": kind, "fmt": rng.choice(["mxfp4", "mxfp8", "fp8", "nvfp4"]), "m": m, "n": n, "k": k,
                "out": rng.choice(["bf16", "bf16", "f32"])}
    if kind == "paged_decode":
        hq, hkv, d = rng.choice([(16, 2, 256), (32, 4, 256), (8, 2, 128), (16, 4, 256)])
        batch = _log(rng, 1, 64)
        hi = _log(rng, 64, max(64, min(32768, 240000 // (batch * hkv))))
        return {"kind": kind, "kv": rng.choice(["bf16", "bf16", "fp8", "i8"]), "batch": batch, "lo": max(1, hi // 8),
                "hi": hi, "hq": hq, "hkv": hkv, "d": d, "page": rng.choice([16, 64, 256])}
    if kind == "paged_prefill":
        hq, hkv, d = rng.choice([(16, 2, 256), (32, 4, 256), (8, 2, 128)])
        batch = rng.choice([1, 1, 2, 4])
        hist = rng.choice([0, _log(rng, 16, 16000)])
        top = max(2, min(4096, int(6e10 / (4.0 * d * hq * (hist + 2048) * batch))))
        return {"kind": kind, "batch": batch, "new": _log(rng, 2, top), "hist": hist, "hq": hq, "hkv": hkv, "d": d,
                "page": rng.choice([16, 64])}
    if kind == "gdn_decode":
        tokens = rng.choice([1, 1, 2, 3, 4])
        return {"kind": kind, "batch": _log(rng, 1, 64), "tokens": tokens, "nk": 16, "nv": rng.choice([16, 32])}
    if kind == "gdn_prefill":
        batch = rng.choice([1, 1, 2, 4])
        return {"kind": kind, "batch": batch, "tokens": _log(rng, 17, 4096 // batch), "nk": 16,
                "nv": rng.choice([16, 32])}
    if kind == "moe":
        return {"kind": kind, "tokens": _log(rng, 1, 4000)}
    batch = _log(rng, 1, 8)
    hi = _log(rng, 64, 60000 // batch if batch > 3 else 16384)
    return {"kind": kind, "batch": batch, "tokens": rng.choice([1, 2, 3, 4, 5, 8, 16]), "lo": max(1, hi // 8),
            "hi": hi}


# ---- sizes that follow from a case alone ----
def _lens(case):
    """The context length of each sequence: spread over [lo, hi] by a generator of the case's own sizes."""
    rng = random.Random(case["batch"] * 1000003 + case["lo"] * 1009 + case["hi"])
    return [rng.randint(case["lo"], case["hi"]) for _ in range(case["batch"])]


def _weight_bytes(fmt, n, k):
    return {"mxfp4": n * k // 2 + n * k // 32, "nvfp4": n * k // 2 + n * k // 16 + 4, "mxfp8": n * k + n * k // 32,
            "fp8": n * k + 4 * n}[fmt]


def _active_experts(tokens):
    """The expected number of distinct experts that `tokens` tokens select."""
    e, k = MOE["experts"], MOE["top_k"]
    return e * (1.0 - (1.0 - k / e) ** tokens)


def work(case):
    kind = case["kind"]
    if kind == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        out = 4 if case["out"] == "f32" else 2
        return {"bytes": _weight_bytes(case["fmt"], n, k) + 2 * m * k + out * m * n, "flops": 2.0 * m * n * k}
    if kind == "paged_decode":
        toks = sum(_lens(case))
        row = case["hkv"] * (case["d"] * (2 if case["kv"] == "bf16" else 1) + (2 if case["kv"] == "i8" else 0))
        return {"bytes": 2 * toks * row + 4 * case["batch"] * case["hq"] * case["d"],
                "flops": 4.0 * toks * case["hq"] * case["d"]}
    if kind == "paged_prefill":
        b, n, h = case["batch"], case["new"], case["hist"]
        return {"bytes": b * (4 * (h + n) * case["hkv"] * case["d"] + 4 * n * case["hq"] * case["d"]),
                "flops": 4.0 * b * case["d"] * case["hq"] * (n * h + n * (n + 1) / 2)}
    if kind in ("gdn_decode", "gdn_prefill"):
        b, t, nk, nv = case["batch"], case["tokens"], case["nk"], case["nv"]
        io = b * t * (2 * nk * 256 + 2 * nv * 256 + 4 * nv)
        flops = 6.0 * b * t * nv * 128 * 128
        if kind == "gdn_prefill":  # the chunked form: per 64-token chunk five 64 x 64 x 128 and three 64 x 128 x 128
            flops = float(b * nv * ((t + 63) // 64)) * (5 * 2 * 64 * 64 * 128 + 3 * 2 * 64 * 128 * 128)
        return {"bytes": io + 2 * b * nv * 65536, "flops": flops}
    if kind == "moe":
        t, h, f = case["tokens"], MOE["hidden"], MOE["inter"]
        per = 3 * (f * h // 2 + f * h // 32)
        return {"bytes": int((_active_experts(t) + 1) * per) + 2 * MOE["experts"] * h + 6 * t * h
                + 4 * t * (MOE["experts"] + 2 * MOE["top_k"]),
                "flops": 2.0 * t * (h * MOE["experts"] + (MOE["top_k"] + 1) * 3 * h * f)}
    b, t, c = case["batch"], case["tokens"], LAYER
    hid, toks, rows = c["hidden"], sum(_lens(case)), case["batch"] * case["tokens"]
    proj = (3 * c["hq"] + 2 * c["hkv"]) * c["d"] * hid
    mlp = 3 * hid * c["inter"]
    return {"bytes": proj + mlp // 2 + mlp // 32 + 4 * (toks + rows) * c["hkv"] * c["d"] + 4 * rows * hid,
            "flops": 2.0 * rows * (proj + mlp) + 4.0 * c["d"] * c["hq"] * t * toks}


# ---- inputs, made on the device from the seed ----
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *shape, std=1.0, dtype=torch.bfloat16):
    x = torch.randn(*shape, generator=g, device=DEV, dtype=torch.float32)
    return (x if std == 1.0 else x * std).to(dtype)


def _bytes(g, lo, hi, *shape):
    return torch.randint(lo, hi, shape, generator=g, device=DEV, dtype=torch.uint8)


def _weight(g, fmt, n, k):
    """Weights of an RMS near 0.05 in each format, as axk/configs.py draws them."""
    if fmt == "mxfp4":
        return {"w": _bytes(g, 0, 256, n, k // 2), "s": _bytes(g, 119, 124, n, k // 32)}
    if fmt == "nvfp4":
        return {"w": _bytes(g, 0, 256, n, k // 2), "s": _bytes(g, 0x28, 0x38, n, k // 16),
                "s2": torch.tensor([0.05], device=DEV)}
    w = _randn(g, n, k, std=3.0 if fmt == "mxfp8" else 0.5, dtype=torch.float8_e4m3fn).view(torch.uint8)
    if fmt == "mxfp8":
        return {"w": w, "s": _bytes(g, 119, 124, n, k // 32)}
    return {"w": w, "s": (torch.rand(n, generator=g, device=DEV) * 2 + 1) / math.sqrt(k)}


def _pages(g, lens, page):
    """A page table over a pool of exactly enough pages, placed by a random permutation."""
    counts = [(n + page - 1) // page for n in lens]
    pool = sum(counts)
    indptr = torch.tensor([sum(counts[:i]) for i in range(len(counts) + 1)], dtype=torch.int32, device=DEV)
    last = torch.tensor([n - page * (c - 1) for n, c in zip(lens, counts)], dtype=torch.int32, device=DEV)
    return pool, indptr, torch.randperm(pool, generator=g, device=DEV).to(torch.int32), last


def _positions(table, lens, news, page):
    """(page id, slot) int32 [B, T, 2] of the last `news` tokens of each sequence."""
    _, indptr, indices, _ = table
    pos = torch.tensor([[n - news + t for t in range(news)] for n in lens], device=DEV)
    pid = indices[indptr[:-1].long()[:, None] + pos // page]
    return torch.stack([pid, (pos % page).to(torch.int32)], -1).contiguous(), pos


def _inputs(case, seed):
    """The case's inputs alone (no workspaces or outputs)."""
    g = _gen(seed)
    kind = case["kind"]
    if kind == "linear":
        s = _weight(g, case["fmt"], case["n"], case["k"])
        s["x"] = _randn(g, case["m"], case["k"])
        return s
    if kind == "paged_decode":
        lens = _lens(case)
        table = _pages(g, lens, case["page"])
        shape = (table[0], 2, case["page"], case["hkv"], case["d"])
        s = {"table": table, "q": _randn(g, case["batch"], case["hq"], case["d"])}
        if case["kv"] == "bf16":
            s["cache"] = _randn(g, *shape)
        elif case["kv"] == "fp8":
            s["cache"] = _randn(g, *shape, std=8.0, dtype=torch.float8_e4m3fn).view(torch.uint8)
        else:
            s["cache"] = _bytes(g, 1, 256, *shape).view(torch.int8)
            s["scales"] = (torch.rand(*shape[:4], generator=g, device=DEV) * 0.01 + 0.008).to(torch.bfloat16)
        return s
    if kind == "paged_prefill":
        b, n = case["batch"], case["new"]
        table = _pages(g, [case["hist"] + n] * b, case["page"])
        return {"table": table, "q": _randn(g, b * n, case["hq"], case["d"]),
                "cache": _randn(g, table[0], 2, case["page"], case["hkv"], case["d"]),
                "qo": torch.arange(b + 1, dtype=torch.int32, device=DEV) * n}
    if kind in ("gdn_decode", "gdn_prefill"):
        b, t, nk, nv = case["batch"], case["tokens"], case["nk"], case["nv"]
        s = {n: _randn(g, b, t, h, 128) for n, h in (("q", nk), ("k", nk), ("v", nv))}
        s["a"], s["b"] = _randn(g, b, t, nv), _randn(g, b, t, nv)
        s["a_log"], s["dt_bias"] = (_randn(g, nv, std=0.5, dtype=torch.float32) for _ in range(2))
        s["state"] = _randn(g, b, nv, 128, 128, std=0.02, dtype=torch.float32)
        return s
    if kind == "moe":
        h, e, f = MOE["hidden"], MOE["experts"], MOE["inter"]
        w = {"w_router": _randn(g, e, h, std=0.02), "w_shg": _randn(g, h, std=0.02)}
        for n, rows, cols in (("gate", f, h), ("up", f, h), ("down", h, f)):
            x = _weight(g, "mxfp4", rows, cols)
            w["w_" + n], w["s_" + n] = x["w"], x["s"]
        w["e_gw"], w["e_gs"] = _bytes(g, 0, 256, e, 2 * f, h // 2), _bytes(g, 119, 124, e, 2 * f, h // 32)
        w["e_dw"], w["e_ds"] = _bytes(g, 0, 256, e, h, f // 2), _bytes(g, 119, 124, e, h, f // 32)
        return {"w": w, "h2": _randn(g, case["tokens"], h), "x_res": _randn(g, case["tokens"], h)}
    c, b, t = LAYER, case["batch"], case["tokens"]
    hid = c["hidden"]
    w = {}
    for n, rows, cols in (("q", 2 * c["hq"] * c["d"], hid), ("k", c["hkv"] * c["d"], hid),
                          ("v", c["hkv"] * c["d"], hid), ("o", hid, c["hq"] * c["d"])):
        x = _weight(g, "fp8", rows, cols)
        w["w_" + n], w["s_" + n] = x["w"], x["s"]
    for n, rows, cols in (("gate", c["inter"], hid), ("up", c["inter"], hid), ("down", hid, c["inter"])):
        w["w_" + n], w["s_" + n] = _bytes(g, 0, 256, rows, cols // 2), _bytes(g, 116, 121, rows, cols // 32)
    for n, size in (("ln1", hid), ("q_norm", c["d"]), ("k_norm", c["d"]), ("ln2", hid)):
        w[n] = 1.0 + _randn(g, size, std=0.1, dtype=torch.float32)
    lens = [n + t for n in _lens(case)]
    table = _pages(g, lens, c["page"])
    loc, pos = _positions(table, lens, t, c["page"])
    inv = c["theta"] ** (-torch.arange(0, c["rot"], 2, dtype=torch.float32, device=DEV) / c["rot"])
    ang = pos.float()[..., None] * inv
    return {"w": w, "table": table, "loc": loc, "cos": ang.cos().to(torch.bfloat16), "x": _randn(g, b, t, hid),
            "sin": ang.sin().to(torch.bfloat16), "cache": _randn(g, table[0], 2, c["page"], c["hkv"], c["d"])}


def prepare(case, seed):
    """The inputs, with the outputs and workspaces that a serving program keeps from step to step."""
    s = _inputs(case, seed)
    kind = case["kind"]
    s["case"] = case
    if kind == "linear":
        s["dt"] = torch.float32 if case["out"] == "f32" else torch.bfloat16
        s["out"] = torch.empty(case["m"], case["n"], dtype=s["dt"], device=DEV)
    elif kind == "paged_decode":
        s["ws"] = axk.paged_decode_workspace(case["batch"], case["hq"], case["hkv"], case["d"], DEV)
        s["out"] = torch.empty_like(s["q"])
    elif kind == "paged_prefill":
        s["out"] = torch.empty_like(s["q"])
    elif kind in ("gdn_decode", "gdn_prefill"):
        s["state_out"], s["out"] = torch.empty_like(s["state"]), torch.empty_like(s["v"])
        if kind == "gdn_prefill":
            s["ws"] = axk.gdn_chunk_workspace(case["batch"], case["tokens"], case["nk"], case["nv"], DEV)
    elif kind == "moe":
        s["ws"] = axk.moe_workspace(case["tokens"], MOE["hidden"], MOE["experts"], MOE["top_k"], MOE["inter"],
                                    MOE["inter"], DEV)
        s["out"] = torch.empty_like(s["h2"])
    else:
        c = LAYER
        s["ws"] = layer.attn_verify_workspace(case["batch"], case["tokens"], c["hidden"], c["hq"], c["hkv"], c["d"],
                                              c["inter"], DEV)
        s["out"] = torch.empty_like(s["x"])
    return s


def run(state):
    s = state
    case = s["case"]
    kind = case["kind"]
    if kind == "linear":
        fmt = case["fmt"]
        if fmt == "mxfp4":
            return axk.mxfp4_gemm(s["x"], s["w"], s["s"], s["dt"], output=s["out"])
        if fmt == "nvfp4":
            return axk.nvfp4_gemm(s["x"], s["w"], s["s"], s["s2"], s["dt"], output=s["out"])
        if fmt == "mxfp8":
            return axk.mxfp8_gemm(s["x"], s["w"], s["s"], s["dt"], output=s["out"], fmt="e4m3")
        return axk.fp8_gemm(s["x"], s["w"], None, s["s"], s["dt"], output=s["out"])
    if kind == "paged_decode":
        _, indptr, indices, last = s["table"]
        if case["kv"] == "bf16":
            return axk.paged_decode(s["q"], s["cache"], indptr, indices, last, output=s["out"], workspace=s["ws"])
        if case["kv"] == "fp8":
            return axk.paged_decode_fp8(s["q"], s["cache"], indptr, indices, last, 8.0, output=s["out"],
                                        workspace=s["ws"])
        return axk.paged_decode_i8(s["q"], s["cache"], s["scales"], indptr, indices, last, output=s["out"],
                                   workspace=s["ws"])
    if kind == "paged_prefill":
        _, indptr, indices, last = s["table"]
        return axk.paged_prefill(s["q"], s["cache"], s["qo"], indptr, indices, last, output=s["out"])
    if kind == "gdn_decode":
        return axk.gdn_recurrent(s["q"], s["k"], s["v"], s["a"], s["b"], s["a_log"], s["dt_bias"], s["state"],
                                 s["state_out"], s["out"])
    if kind == "gdn_prefill":
        return axk.gdn_chunk_prefill(s["q"], s["k"], s["v"], s["a"], s["b"], s["a_log"], s["dt_bias"], s["state"],
                                     s["state_out"], s["out"], workspace=s["ws"])
    if kind == "moe":
        return axk.moe_decode(s["h2"], s["w"], MOE["top_k"], x_res=s["x_res"], output=s["out"], workspace=s["ws"])
    _, indptr, indices, last = s["table"]
    out = layer.attn_layer_verify(s["x"], s["w"], s["cos"], s["sin"], s["cache"], indptr, indices, last, s["loc"],
                                  LAYER["hq"], LAYER["rot"], workspace=s["ws"], out=s["out"])
    return out, s["cache"]


def tolerance(case):
    # Four times the distance to the 64-bit result that bf16 inputs to the matrix products, bf16 intermediates and
    # bf16 outputs give (linears 1.7e-3, attention 2.3e-3, recurrence 1.7e-3, chunked form 4.7e-3, MoE 3.5e-3, layer
    # 3.0e-3); fp32 outputs 2.7e-7. Expert ids: two neighbours of almost equal logits may change places.
    kind = case["kind"]
    if kind == "linear":
        return {"rel": 2e-6 if case["out"] == "f32" else 7e-3}
    if kind == "moe":
        return {"rel": 1.4e-2, "differ": max(1e-3, 2.5 / (MOE["top_k"] * case["tokens"]))}
    return {"rel": {"paged_decode": 9e-3, "paged_prefill": 9e-3, "gdn_decode": 7e-3, "gdn_prefill": 2e-2,
                    "attn_verify": 1.2e-2}[kind]}


# ---- what run returns, in 64 bits and plain torch ----
_E2M1 = [0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0]


def _fp4(codes):
    lut = torch.tensor(_E2M1 + [-v for v in _E2M1], dtype=F64, device=codes.device)
    return torch.stack([lut[(codes & 15).long()], lut[(codes >> 4).long()]], -1).flatten(-2)


def _dequant(fmt, w, s, s2=None):
    """[N, K] in 64 bits."""
    n = w.shape[0]
    if fmt == "fp8":
        return w.view(torch.float8_e4m3fn).to(F64) * s.to(F64)[:, None]
    v = w.view(torch.float8_e4m3fn).to(F64) if fmt == "mxfp8" else _fp4(w)
    scale = torch.exp2(s.to(F64) - 127) if fmt != "nvfp4" else s.view(torch.float8_e4m3fn).to(F64) * s2.to(F64)
    return (v.reshape(n, scale.shape[1], -1) * scale[..., None]).reshape(n, -1)


def _linear64(x, fmt, w, s, s2=None, rows=32768):
    """x @ dequant(w).T in 64 bits, `rows` weight rows at a time."""
    return torch.cat([x @ _dequant(fmt, w[i:i + rows], s[i:i + rows], s2).T for i in range(0, w.shape[0], rows)], 1)


def _attend(q, keys, values, first):
    """q [T, HQ, D] (row t sees the first + t + 1 leading tokens), keys / values [L, HKV, D], all in 64 bits."""
    t, hq, d = q.shape
    length, hkv = keys.shape[:2]
    g = hq // hkv
    hide = torch.arange(length, device=q.device)[None] > first + torch.arange(t, device=q.device)[:, None]
    out = torch.empty_like(q)
    for h in range(hq):
        s = (q[:, h] @ keys[:, h // g].T * d ** -0.5).masked_fill_(hide, float("-inf"))
        out[:, h] = torch.softmax(s, -1) @ values[:, h // g]
    return out


def _tokens(cache, table, b, scale=None):
    """Sequence b's keys and values [L, HKV, D] in 64 bits."""
    _, indptr, indices, last = table
    lo, hi = int(indptr[b]), int(indptr[b + 1])
    page = cache.shape[2]
    pages = cache[indices[lo:hi].long()].to(F64)
    if scale is not None:
        pages = pages * scale[indices[lo:hi].long()].to(F64)[..., None]
    n = (hi - lo - 1) * page + int(last[b])
    return tuple(pages[:, i].reshape(-1, *cache.shape[3:])[:n] for i in (0, 1))


def _swiglu(x, gate, up, down):
    a = x @ gate.T
    return (a * torch.sigmoid(a) * (x @ up.T)) @ down.T


def _norm(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6) * w.to(F64)


def _exact_gdn(s):
    q, k, v, a, b = (s[n].to(F64) for n in ("q", "k", "v", "a", "b"))
    per = v.shape[2] // q.shape[2]
    q, k = (x / torch.sqrt(x.square().sum(-1, keepdim=True) + 1e-6) for x in (q, k))
    q, k = (q * 128 ** -0.5).repeat_interleave(per, 2), k.repeat_interleave(per, 2)
    decay = torch.exp(-torch.exp(s["a_log"].to(F64)) * torch.nn.functional.softplus(a + s["dt_bias"].to(F64)))
    beta = torch.sigmoid(b)
    state, out = s["state"].to(F64), torch.empty_like(v)
    for t in range(q.shape[1]):
        state = state * decay[:, t, :, None, None]
        err = (v[:, t] - (k[:, t, :, :, None] * state).sum(2)) * beta[:, t, :, None]
        state = state + k[:, t, :, :, None] * err[:, :, None, :]
        out[:, t] = (q[:, t, :, :, None] * state).sum(2)
    return out, state


def _exact_moe(s):
    w, h, res = s["w"], s["h2"].to(F64), s["x_res"].to(F64)
    logits = h @ w["w_router"].to(F64).T
    order = torch.sort(logits, dim=-1, descending=True, stable=True)[1][:, :MOE["top_k"]]
    prob = torch.gather(torch.softmax(logits, -1), 1, order)
    prob = prob / prob.sum(-1, keepdim=True)
    shared = [_dequant("mxfp4", w["w_" + n], w["s_" + n]) for n in ("gate", "up", "down")]
    out = res + torch.sigmoid(h @ w["w_shg"].to(F64))[:, None] * _swiglu(h, *shared)
    for e in range(MOE["experts"]):
        rows, slots = torch.nonzero(order == e, as_tuple=True)
        if rows.numel():
            gu = _dequant("mxfp4", w["e_gw"][e], w["e_gs"][e])
            y = _swiglu(h[rows], gu[:MOE["inter"]], gu[MOE["inter"]:], _dequant("mxfp4", w["e_dw"][e], w["e_ds"][e]))
            out.index_add_(0, rows, y * prob[rows, slots][:, None])
    return out, logits, order.to(torch.int32), prob


def _rope(x, cos, sin, rot):
    half = rot // 2
    x1, x2 = x[..., :half], x[..., half:rot]
    c, s = cos.to(F64)[:, :, None], sin.to(F64)[:, :, None]
    return torch.cat([x1 * c - x2 * s, x2 * c + x1 * s, x[..., rot:]], -1)


def _exact_layer(s):
    c, w = LAYER, s["w"]
    b, t, hid = s["x"].shape
    x = s["x"].to(F64).reshape(b * t, hid)
    h = _norm(x, w["ln1"])
    qg, k, v = (_linear64(h, "fp8", w["w_" + n], w["s_" + n]).reshape(b, t, -1, width)
                for n, width in (("q", 2 * c["d"]), ("k", c["d"]), ("v", c["d"])))
    q = _rope(_norm(qg[..., :c["d"]], w["q_norm"]), s["cos"], s["sin"], c["rot"])
    k = _rope(_norm(k, w["k_norm"]), s["cos"], s["sin"], c["rot"])
    cache = s["cache"].to(F64)
    loc = s["loc"].long()
    cache[loc[..., 0], 0, loc[..., 1]] = k
    cache[loc[..., 0], 1, loc[..., 1]] = v
    rows = []
    for i in range(b):
        keys, values = _tokens(cache, s["table"], i)
        rows.append(_attend(q[i], keys, values, keys.shape[0] - t))
    attn = torch.stack(rows) * torch.sigmoid(qg[..., c["d"]:])
    x = x + _linear64(attn.reshape(b * t, -1), "fp8", w["w_o"], w["s_o"])
    mlp = [_dequant("mxfp4", w["w_" + n], w["s_" + n]) for n in ("gate", "up", "down")]
    return (x + _swiglu(_norm(x, w["ln2"]), *mlp)).reshape(b, t, hid), cache


def exact(case, seed):
    s = _inputs(case, seed)
    kind = case["kind"]
    if kind == "linear":
        return _linear64(s["x"].to(F64), case["fmt"], s["w"], s["s"], s.get("s2"))
    if kind == "paged_decode":
        cache = s["cache"]
        scale = s.get("scales")
        if case["kv"] == "fp8":
            cache = cache.view(torch.float8_e4m3fn).to(torch.float32) / 8.0
        rows = []
        for b in range(case["batch"]):
            keys, values = _tokens(cache, s["table"], b, scale)
            rows.append(_attend(s["q"][b:b + 1].to(F64), keys, values, keys.shape[0] - 1))
        return torch.cat(rows)
    if kind == "paged_prefill":
        n = case["new"]
        rows = []
        for b in range(case["batch"]):
            keys, values = _tokens(s["cache"], s["table"], b)
            rows.append(_attend(s["q"][b * n:(b + 1) * n].to(F64), keys, values, case["hist"]))
        return torch.cat(rows)
    if kind in ("gdn_decode", "gdn_prefill"):
        return _exact_gdn(s)
    if kind == "moe":
        return _exact_moe(s)
    return _exact_layer(s)
