"""Performance cases of the fused decode-attention path, over the range it is used in.

Each case is one call (or one serving step) through the public entry points of ``fqkv_decode``:
single-block MHA / GQA decode, split-K decode with the caller's scratch, strided, token-major and
paged KV caches with ragged lengths, the on-GPU KV quantizers that fill the caches, and a decode
step of a static quantized cache (quantize the new token, attend). ``draw`` gives further cases of
the same operations, formats and size ranges.
"""

import math
import os
import sys

import torch

# the package lives one folder below the repository's root, which is the working folder
sys.path.insert(0, os.path.join(os.getcwd(), "fused-quantized-kv-decode-attention_amd"))

import fqkv_decode as fq  # noqa: E402

DEV = "cuda"
QMAX = {"int8": 127.0, "int4": 7.0, "fp8": 448.0}
SRC = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
MAX_BYTES = 1.0e9  # of a drawn case; the largest listed ones read 1.1 GB


def listed():
    """The listed cases; D 64 / 128 and 32 query heads over 8 KV heads are the geometries of the
    repository's benchmark (Llama-3 shapes)."""
    return [
        # two short chat turns: latency and launches count
        dict(name="gqa_fp16_b2_n1200_d128", op="gqa", fmt="fp16", B=2, Hq=32, Hkv=8, N=1200, D=128, W=8),
        # the headline: batch-1 long context, split-K with the caller's scratch
        dict(name="splitk_fp16_n16384_d128", op="splitk", fmt="fp16", B=1, Hq=32, Hkv=8, N=16384, D=128, S=32, W=8),
        # sustained long-context decode, batch 8
        dict(name="splitk_fp16_b8_n32768_d128", op="splitk", fmt="fp16", B=8, Hq=32, Hkv=8, N=32768, D=128, S=8, W=8),
        # a serving batch whose size and length are no powers of two
        dict(name="gqa_fp16_b40_n1777_d128", op="gqa", fmt="fp16", B=40, Hq=32, Hkv=8, N=1777, D=128, W=8),
        # the precision benchmark's MHA shapes: int8 at batch x heads 256, int4 at 2048
        dict(name="mha_int8_b256_n4096_d128", op="mha", fmt="int8", B=256, N=4096, D=128, W=8),
        dict(name="mha_int4_b2048_n4096_d128", op="mha", fmt="int4", B=2048, N=4096, D=128, W=8),
        # a bf16 model's growing cache read in place: the filled part of a larger allocation
        dict(name="strided_bf16_b6_n3001_d128", op="strided", fmt="bf16", B=6, Hq=32, Hkv=8, N=3001, cap=4096, D=128,
             W=8),
        # a token-major (NHD) int8 cache, few sequences
        dict(name="nhd_int8_b12_n2500_d128", op="nhd", fmt="int8", B=12, Hq=32, Hkv=8, N=2500, D=128, W=8),
        # continuous batching over 16-token fp16 pages, lengths from 120 to 7700 tokens
        dict(name="paged_fp16_b32_ragged_d128", op="paged", fmt="fp16", B=32, Hq=32, Hkv=8, N=7700, nmin=120, page=16,
             order="nhd", D=128, W=8),
        # the same over head-major fp8 pages of 64, a larger batch and longer contexts
        dict(name="paged_fp8_b64_ragged_d128", op="paged", fmt="fp8", B=64, Hq=32, Hkv=8, N=12000, nmin=300, page=64,
             order="hnd", D=128, W=8),
        # prefill: a chunk of prompt tokens quantized into shuffled pages
        dict(name="to_pages_int8_bf16_t8190_d128", op="to_pages", fmt="int8", src="bf16", T=8190, Hkv=8, page=16,
             order="hnd", D=128),
        # one layer of a graph-style decode step over a static int4 cache that is partly filled
        dict(name="step_int4_b16_n1100_d64", op="step", fmt="int4", src="fp16", B=16, Hq=32, Hkv=8, N=1100, cap=2048,
             D=64, W=8),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def draw(rng):
    """One more case: operation, format, head geometry and sizes over the ranges above."""
    while True:
        op = rng.choice(["gqa", "gqa", "splitk", "splitk", "mha", "strided", "nhd", "paged", "paged", "paged",
                         "to_pages", "append", "quantize", "step"])
        D = rng.choice([64, 128, 128])
        Hkv = rng.choice([2, 4, 8, 8])
        Hq = Hkv * rng.choice([1, 3, 4, 4, 7, 8])
        B = _log_int(rng, 1, 128)
        N = _log_int(rng, 256, 40000)
        quant = rng.choice(["int8", "int4", "fp8"])
        any_fmt = rng.choice(["fp16", "bf16", "int8", "int4", "fp8"])
        order = rng.choice(["nhd", "hnd"])
        page = rng.choice([16, 32, 64, 256])
        src = rng.choice(["fp16", "bf16", "fp32"])
        if op == "gqa":
            c = dict(op=op, fmt=rng.choice(["fp16", "int8", "int4", "fp8"]), B=B, Hq=Hq, Hkv=Hkv, N=N, D=D, W=8)
        elif op == "splitk":
            # the caller's split count: about one workgroup per compute unit of a 256-CU card
            S = max(1, min(64, -(-256 // (B * Hkv)), N // 32))
            S = -(-N // -(-N // S))  # no empty split
            c = dict(op=op, fmt=any_fmt, B=B, Hq=Hq, Hkv=Hkv, N=N, D=D, S=S, W=8)
        elif op == "mha":
            c = dict(op=op, fmt=rng.choice(["fp16", "int8", "int4"]), B=_log_int(rng, 8, 2048), N=_log_int(rng, 256, 8192),
                     D=D, W=8)
        elif op == "strided":
            c = dict(op=op, fmt=any_fmt, B=min(B, 32), Hq=Hq, Hkv=Hkv, N=N, cap=N + rng.randrange(1, 600), D=D, W=8)
        elif op == "nhd":
            c = dict(op=op, fmt=any_fmt, B=min(B, 64), Hq=Hq, Hkv=Hkv, N=N, D=D, W=8)
        elif op == "paged":
            c = dict(op=op, fmt=any_fmt, B=B, Hq=Hq, Hkv=Hkv, N=N, nmin=max(16, N // rng.choice([1, 8, 40])), page=page,
                     order=order, D=D, W=8)
        elif op == "to_pages":
            c = dict(op=op, fmt=quant, src=src, T=_log_int(rng, 16, 60000), Hkv=Hkv, page=page, order=order, D=D)
        elif op == "append":
            c = dict(op=op, fmt=quant, src=src, B=min(B, 16), Hkv=Hkv, n=_log_int(rng, 16, 16000), D=D)
        elif op == "quantize":
            c = dict(op=op, fmt=quant, src=src, T=_log_int(rng, 64, 800000), D=D)
        else:
            n = min(N, 8000)
            c = dict(op=op, fmt=quant, src=rng.choice(["fp16", "bf16"]), B=min(B, 64), Hq=Hq, Hkv=Hkv, N=n,
                     cap=1 << n.bit_length(), D=D, W=8)
        if work(c)["bytes"] <= MAX_BYTES:
            return c


# ---------------------------------------------------------------- inputs ----
def _lengths(c):
    """Sequence lengths of a paged case: evenly spread in log length from nmin to N (the longest is N)."""
    B, lo, hi = c["B"], c["nmin"], c["N"]
    if B == 1:
        return [hi]
    return [int(round(lo * (hi / lo) ** (i / (B - 1)))) for i in range(B)]


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) & 0x7FFFFFFFFFFF)


def _quantize(x, fmt):
    """Per-token codes and fp16 scales of fp32 rows x[..., D] (plain torch)."""
    s = (x.abs().amax(-1, keepdim=True) / QMAX[fmt]).clamp_(min=1e-8)
    y = x / s
    s = s.squeeze(-1).half()
    if fmt == "fp8":
        return y.clamp_(-448.0, 448.0).to(torch.float8_e4m3fn), s
    y = y.round_().clamp_(-QMAX[fmt], QMAX[fmt])
    if fmt == "int8":
        return y.to(torch.int8), s
    n = y.to(torch.int16)
    return ((n[..., 0::2] & 15) | ((n[..., 1::2] & 15) << 4)).to(torch.uint8), s


def _rows(shape, fmt, g, key):
    """K or V rows of a format: normal values, keys with a few large channels (as rotary keys have).
    Returns (codes, scales or None)."""
    D = shape[-1]
    out, scales = [], []
    lead = shape[0]
    per = max(1, int((1 << 27) // max(1, math.prod(shape[1:]))))
    boost = torch.ones(D, device=DEV)
    if key:
        boost[:: D // 8] = 2.0
    for i in range(0, lead, per):
        x = torch.randn((min(per, lead - i),) + tuple(shape[1:]), generator=g, device=DEV) * boost
        if fmt in SRC:
            out.append(x.to(SRC[fmt]))
        else:
            q, s = _quantize(x, fmt)
            out.append(q)
            scales.append(s)
        del x
    cat = lambda v: v[0] if len(v) == 1 else torch.cat([t.view(torch.uint8) for t in v]).view(v[0].dtype)  # noqa: E731
    return cat(out), (torch.cat(scales) if scales else None)


def _decode(codes, s):
    """Codes (and scales) back to 64-bit values [..., D]."""
    if codes.dtype == torch.uint8:
        lo, hi = (codes & 15).to(torch.int8), (codes >> 4).to(torch.int8)
        v = torch.stack((lo, hi), -1).flatten(-2)
        x = torch.where(v >= 8, v - 16, v).double()
    elif codes.dtype == torch.float8_e4m3fn:
        x = codes.float().double()
    else:
        x = codes.double()
    return x if s is None else x * s.double().unsqueeze(-1)


def prepare(case, seed):
    c, g = case, _gen(seed)
    op, D = c["op"], c["D"]
    st = {"c": c}
    if op in ("to_pages", "append", "quantize"):
        dt = SRC[c["src"]]
        cd = {"int8": torch.int8, "int4": torch.uint8, "fp8": torch.float8_e4m3fn}[c["fmt"]]
        w = D // 2 if c["fmt"] == "int4" else D
        if op == "quantize":
            st["x"] = torch.randn(c["T"], D, generator=g, device=DEV).to(dt)
            return st
        if op == "append":
            B, H, n = c["B"], c["Hkv"], c["n"]
            st["k"] = torch.randn(B, H, n, D, generator=g, device=DEV).to(dt)
            st["v"] = torch.randn(B, H, n, D, generator=g, device=DEV).to(dt)
            cap = n + 300
            st["pos"] = 37
            caches = lambda: torch.zeros(B, H, cap, w, dtype=torch.uint8, device=DEV).view(cd)  # noqa: E731
            st["kc"], st["vc"] = caches(), caches()
            st["ks"] = torch.zeros(B, H, cap, dtype=torch.float16, device=DEV)
            st["vs"] = torch.zeros_like(st["ks"])
            return st
        T, H, page = c["T"], c["Hkv"], c["page"]
        st["k"] = torch.randn(T, H, D, generator=g, device=DEV).to(dt)
        st["v"] = torch.randn(T, H, D, generator=g, device=DEV).to(dt)
        need = -(-T // page)
        P = need + max(1, need // 8)
        ids = torch.randperm(P, generator=g, device=DEV)[:need]
        t = torch.arange(T, device=DEV)
        st["slots"] = (ids[t // page] * page + t % page).to(torch.int32)
        st["kc"], st["vc"], st["ks"], st["vs"] = _page_buffers(P, page, H, w, cd, c["order"])
        return st

    fmt = c["fmt"]
    if op == "mha":
        B, N = c["B"], c["N"]
        st["q"] = torch.randn(B, D, generator=g, device=DEV).half()
        st["k"], st["ks"] = _rows((B, N, D), fmt, g, True)
        st["v"], st["vs"] = _rows((B, N, D), fmt, g, False)
        return st
    B, Hq, Hkv, N = c["B"], c["Hq"], c["Hkv"], c["N"]
    st["q"] = torch.randn(B, Hq, D, generator=g, device=DEV).half()
    if op == "gqa":
        st["k"], st["ks"] = _rows((B, Hkv, N, D), fmt, g, True)
        st["v"], st["vs"] = _rows((B, Hkv, N, D), fmt, g, False)
    elif op == "splitk":
        S = c["S"]
        st["q"] = st["q"].view(B * Hq, D)
        st["k"], st["ks"] = _rows((B * Hkv, N, D), fmt, g, True)
        st["v"], st["vs"] = _rows((B * Hkv, N, D), fmt, g, False)
        st["m"] = torch.empty(B * Hq, S, device=DEV)
        st["l"] = torch.empty(B * Hq, S, device=DEV)
        st["p"] = torch.empty(B * Hq, S, D, device=DEV)
        st["o"] = torch.empty(B * Hq, D, dtype=torch.float16, device=DEV)
    elif op == "strided":
        st["k"], st["ks"] = (None if t is None else t[:, :, :N] for t in _rows((B, Hkv, c["cap"], D), fmt, g, True))
        st["v"], st["vs"] = (None if t is None else t[:, :, :N] for t in _rows((B, Hkv, c["cap"], D), fmt, g, False))
    elif op == "nhd":
        st["k"], st["ks"] = _rows((B, N, Hkv, D), fmt, g, True)
        st["v"], st["vs"] = _rows((B, N, Hkv, D), fmt, g, False)
    elif op == "paged":
        page = c["page"]
        lens = _lengths(c)
        order = torch.randperm(B, generator=torch.Generator().manual_seed(int(seed))).tolist()
        lens = [lens[i] for i in order]
        npg = [-(-n // page) for n in lens]
        P = sum(npg) + max(1, sum(npg) // 16)
        mp = max(npg)
        ids = torch.randperm(P, generator=g, device=DEV).to(torch.int32)
        table = torch.zeros(B, mp, dtype=torch.int32, device=DEV)
        at = 0
        for b, k in enumerate(npg):
            table[b, :k] = ids[at:at + k]
            at += k
        shape = (P, page, Hkv, D) if c["order"] == "nhd" else (P, Hkv, page, D)
        view = (lambda t: t) if c["order"] == "nhd" else (  # noqa: E731
            lambda t: None if t is None else t.transpose(1, 2))
        st["k"], st["ks"] = (view(t) for t in _rows(shape, fmt, g, True))
        st["v"], st["vs"] = (view(t) for t in _rows(shape, fmt, g, False))
        st["table"], st["lens"] = table, torch.tensor(lens, dtype=torch.int32, device=DEV)
    else:  # step: N - 1 tokens cached, the new one at position N - 1
        cap, dt = c["cap"], SRC[c["src"]]
        st["kc"], st["ks"] = _rows((B, Hkv, cap, D), fmt, g, True)
        st["vc"], st["vs"] = _rows((B, Hkv, cap, D), fmt, g, False)
        st["k"] = torch.randn(B, Hkv, 1, D, generator=g, device=DEV).to(dt)
        st["v"] = torch.randn(B, Hkv, 1, D, generator=g, device=DEV).to(dt)
        lens = torch.full((B,), N, dtype=torch.int32, device=DEV)
        st["lens"], st["pos"] = lens, lens - 1
        st["table"] = torch.arange(B, dtype=torch.int32, device=DEV).view(B, 1)
    return st


def _page_buffers(P, page, H, w, cd, order):
    shape = (P, page, H, w) if order == "nhd" else (P, H, page, w)
    out = []
    for dtype, sh in ((cd, shape), (cd, shape), (torch.float16, shape[:3]), (torch.float16, shape[:3])):
        t = torch.zeros(sh, dtype=torch.uint8, device=DEV).view(dtype) if dtype == cd else torch.zeros(
            sh, dtype=dtype, device=DEV)
        out.append(t if order == "nhd" else t.transpose(1, 2))
    return out


# ------------------------------------------------------------------ pass ----
def run(st):
    c = st["c"]
    op, fmt = c["op"], c["fmt"]
    if op == "gqa":
        if fmt == "fp16":
            return fq.decode_attn_gqa(st["q"], st["k"], st["v"], c["W"])
        fn = {"int8": fq.decode_attn_gqa_int8, "int4": fq.decode_attn_gqa_int4, "fp8": fq.decode_attn_gqa_fp8}[fmt]
        return fn(st["q"], st["k"], st["v"], st["ks"], st["vs"], c["W"])
    if op == "mha":
        if fmt == "fp16":
            return fq.decode_attn_fp16_mw(st["q"], st["k"], st["v"], c["W"])
        fn = fq.decode_attn_int8_mw if fmt == "int8" else fq.decode_attn_int4
        return fn(st["q"], st["k"], st["v"], st["ks"], st["vs"], c["W"])
    if op == "splitk":
        if fmt in ("fp16", "bf16"):
            fn = fq.gqa_sk_fast if fmt == "fp16" else fq.gqa_sk_fast_bf16
            fn(st["q"], st["k"], st["v"], st["m"], st["l"], st["p"], st["o"], c["S"], c["W"], 8)
        else:
            fn = {"int8": fq.gqa_sk_fast_int8, "int4": fq.gqa_sk_fast_int4, "fp8": fq.gqa_sk_fast_fp8}[fmt]
            fn(st["q"], st["k"], st["v"], st["ks"], st["vs"], st["m"], st["l"], st["p"], st["o"], c["S"], c["W"], 8)
        return st["o"], st["m"], st["l"], st["p"]
    if op == "strided":
        return fq.decode_attn_gqa_strided(st["q"], st["k"], st["v"], c["W"], st["ks"], st["vs"])
    if op == "nhd":
        return fq.decode_attn_gqa_nhd(st["q"], st["k"], st["v"], c["W"], st["ks"], st["vs"])
    if op == "paged":
        return fq.decode_attn_gqa_paged(st["q"], st["k"], st["v"], st["table"], st["lens"], c["N"], c["W"], st["ks"],
                                        st["vs"])
    if op == "quantize":
        fn = {"int8": fq.quantize_int8_per_token, "int4": fq.quantize_int4_per_token,
              "fp8": fq.quantize_fp8_per_token}[fmt]
        return _codes(fn(st["x"]))
    if op == "append":
        fq.quantize_kv_append_(st["k"], st["v"], st["kc"], st["vc"], st["ks"], st["vs"], st["pos"])
        return _codes((st["kc"], st["vc"], st["ks"], st["vs"]))
    if op == "to_pages":
        fq.quantize_kv_to_pages_(st["k"], st["v"], st["slots"], st["kc"], st["vc"], st["ks"], st["vs"])
        return _codes((st["kc"], st["vc"], st["ks"], st["vs"]))
    # step: the static cache's [B, Hkv, cap, .] buffers are one page per sequence
    fq.quantize_kv_append_at_(st["k"], st["v"], st["kc"], st["vc"], st["ks"], st["vs"], st["pos"])
    return fq.decode_attn_gqa_paged(st["q"], st["kc"].permute(0, 2, 1, 3), st["vc"].permute(0, 2, 1, 3), st["table"],
                                    st["lens"], c["cap"], c["W"], st["ks"].permute(0, 2, 1), st["vs"].permute(0, 2, 1))


def _codes(ts):
    """Quantizer outputs as integers (fp8 codes as their bytes)."""
    return tuple(t.view(torch.uint8) if t.dtype == torch.float8_e4m3fn else t for t in ts)


# ------------------------------------------------------------------ work ----
def _row_bytes(fmt, D):
    return {"fp16": 2 * D, "bf16": 2 * D, "int8": D + 2, "fp8": D + 2, "int4": D // 2 + 2}[fmt]  # scale included


def work(case):
    c = case
    op, D, rb = c["op"], c["D"], _row_bytes(c["fmt"], c["D"])
    if op in ("to_pages", "append", "quantize"):
        rows = {"to_pages": lambda: 2 * c["T"] * c["Hkv"], "append": lambda: 2 * c["B"] * c["Hkv"] * c["n"],
                "quantize": lambda: c["T"]}[op]()
        src = 4 if c["src"] == "fp32" else 2
        return {"bytes": rows * (D * src + rb) + (4 * c["T"] if op == "to_pages" else 0), "flops": 4 * rows * D}
    if op == "mha":
        return {"bytes": c["B"] * (2 * c["N"] * rb + 4 * D), "flops": 4 * c["B"] * c["N"] * D}
    heads = c["B"] * c["Hq"]
    tokens = sum(_lengths(c)) if op == "paged" else c["B"] * c["N"]
    b = tokens * c["Hkv"] * 2 * rb + heads * 4 * D
    if op == "splitk":
        b += heads * c["S"] * (D + 2) * 4  # the caller's scratch is an output
    if op == "paged":
        b += sum(-(-n // c["page"]) for n in _lengths(c)) * 4 + 4 * c["B"]
    if op == "step":
        b += 2 * c["B"] * c["Hkv"] * 2 * D
    return {"bytes": b, "flops": 4 * tokens * c["Hq"] * D}


def tolerance(case):
    """Quantizers: bit for bit. Attention: about four times the distance of the fp16 outputs from ``exact``,
    2.0e-4 to 2.6e-4 over the listed and two dozen drawn cases (split-K's fp32 partials: below 1e-5)."""
    if case["op"] in ("to_pages", "append", "quantize"):
        return "exact"
    return {"rel": 1e-3}


# ----------------------------------------------------------------- exact ----
def _attend(q, k, v):
    """softmax(q k^T / sqrt(D)) v for q [R,G,D], k, v [R,N,D] in 64 bits."""
    x = torch.matmul(k, q.transpose(1, 2).contiguous()) / math.sqrt(q.shape[-1])  # [R,N,G]
    p = torch.softmax(x, 1)
    return torch.matmul(p.transpose(1, 2).contiguous(), v)


def exact(case, seed):
    c = case
    op = c["op"]
    if op in ("to_pages", "append", "quantize"):
        return None  # whole codes, compared bit for bit
    st = prepare(c, seed)
    D = c["D"]
    if op == "mha":
        q, rows = st["q"].double().view(c["B"], 1, D), c["B"]
    else:
        rows = c["B"] * c["Hkv"]
        q = st["q"].double().view(rows, c["Hq"] // c["Hkv"], D)
    out = torch.empty_like(q)

    if op in ("mha", "gqa", "splitk", "strided"):
        lead = 2 if op in ("gqa", "strided") else 1  # dims before the tokens
        flat = lambda t: None if t is None else t.reshape((rows, c["N"]) + tuple(t.shape[lead + 1:]))  # noqa: E731
        k, v, ks, vs = flat(st["k"]), flat(st["v"]), flat(st["ks"]), flat(st["vs"])
        cut = lambda t, a, b: None if t is None else t[a:b]  # noqa: E731
        per = max(1, (1 << 26) // (c["N"] * D))
        parts = None
        if op == "splitk":
            parts = [torch.empty(rows * q.shape[1], c["S"], dtype=torch.float64, device=DEV) for _ in range(2)]
            parts.append(torch.empty(rows * q.shape[1], c["S"], D, dtype=torch.float64, device=DEV))
        for a in range(0, rows, per):
            b = min(rows, a + per)
            kd, vd = _decode(cut(k, a, b), cut(ks, a, b)), _decode(cut(v, a, b), cut(vs, a, b))
            out[a:b] = _attend(q[a:b], kd, vd)
            if parts is not None:
                _partials(c, q[a:b], kd, vd, a * q.shape[1], parts)
        if op == "splitk":
            return (out.view(rows * q.shape[1], D),) + tuple(parts)
        return out.view(c["B"], D) if op == "mha" else out.view(c["B"], c["Hq"], D)

    if op == "step":
        # the new token's row as the quantizer's format stores it
        for new, cache, sc in (("k", "kc", "ks"), ("v", "vc", "vs")):
            x = st[new][:, :, 0]
            q1, s1 = _quantize_as_stored(x, c["fmt"])
            st[cache].view(torch.uint8)[:, :, c["N"] - 1] = q1.view(torch.uint8)
            st[sc][:, :, c["N"] - 1] = s1
    for b in range(c["B"]):
        if op == "paged":
            n = int(st["lens"][b])
            ids = st["table"][b, : -(-n // c["page"])].long()
            take = lambda t: None if t is None else _index(t, ids)[:n].transpose(0, 1)  # noqa: E731
            k, v, ks, vs = take(st["k"]), take(st["v"]), take(st["ks"]), take(st["vs"])
        elif op == "nhd":
            take = lambda t: None if t is None else t[b].transpose(0, 1)  # noqa: E731
            k, v, ks, vs = take(st["k"]), take(st["v"]), take(st["ks"]), take(st["vs"])
        else:
            n = c["N"]
            k, v, ks, vs = st["kc"][b, :, :n], st["vc"][b, :, :n], st["ks"][b, :, :n], st["vs"][b, :, :n]
        r = slice(b * c["Hkv"], (b + 1) * c["Hkv"])
        out[r] = _attend(q[r], _decode(k, ks).contiguous(), _decode(v, vs).contiguous())
    return out.view(c["B"], c["Hq"], D)


def _index(t, ids):
    """Pages ids of t [P, page, H, ...] as tokens [len(ids) * page, H, ...]."""
    if t.dtype == torch.float8_e4m3fn:
        return t.view(torch.uint8)[ids].flatten(0, 1).contiguous().view(torch.float8_e4m3fn)
    return t[ids].flatten(0, 1)


def _quantize_as_stored(x, fmt):
    """The library's stated quantizer in plain torch: fp32 expressions (bf16 widened; fp8 always), or fp16
    ones for fp16 rows."""
    f16 = x.dtype == torch.float16 and fmt != "fp8"
    y = x if f16 else x.float()
    a = y.abs().amax(-1, keepdim=True)
    inv = torch.tensor(1.0, dtype=torch.float32, device=x.device) / QMAX[fmt]
    s = (a.float() * inv).half() if f16 else (a * inv).clamp(min=1e-8)
    r = y / s
    if fmt == "fp8":
        return r.clamp(-448.0, 448.0).to(torch.float8_e4m3fn), s.squeeze(-1).half()
    n = r.float().round().clamp(-QMAX[fmt], QMAX[fmt]).to(torch.int16)
    if fmt == "int8":
        return n.to(torch.int8), s.squeeze(-1).half()
    return ((n[..., 0::2] & 15) | ((n[..., 1::2] & 15) << 4)).to(torch.uint8), s.squeeze(-1).half()


def _partials(c, q, k, v, h0, parts):
    """Each split's maximum, sum of weights and weighted values (scores in natural-log units)."""
    S, N, D = c["S"], c["N"], c["D"]
    chunk = -(-N // S)
    x = torch.matmul(k, q.transpose(1, 2).contiguous()) / math.sqrt(D)  # [R,N,G]
    R, G = q.shape[:2]
    h = slice(h0, h0 + R * G)
    for s in range(S):
        a, b = s * chunk, min(N, (s + 1) * chunk)
        if a >= b:
            parts[0][h, s], parts[1][h, s], parts[2][h, s] = -math.inf, 0.0, 0.0
            continue
        m = x[:, a:b].amax(1, keepdim=True)
        p = torch.exp(x[:, a:b] - m)
        parts[0][h, s] = m.reshape(R * G)
        parts[1][h, s] = p.sum(1).reshape(R * G)
        parts[2][h, s] = torch.matmul(p.transpose(1, 2).contiguous(), v[:, a:b].contiguous()).reshape(R * G, D)
