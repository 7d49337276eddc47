"""Contiguous single-block calls at the sizes where their split count changes: one round of
workgroups below the CU count (rounded down), three splits with 4 waves up to 4/3 rows per CU, one
split elsewhere, against the float64 oracle.

Tolerance: fp16 output of values below 4 (half a unit: 2e-3) and weights held to 2^-22."""

import numpy as np
import pytest
import torch

import fqkv_decode as fq
import oracle
from fqkv_decode import quant

TOL = 2e-3
CODE = {"fp16": 0, "int8": 1, "int4": 2}


def split_model(rows, N, D, fmt, W, cus):
    rowb = {"fp16": 2 * D, "int8": D, "int4": D // 2}[fmt]
    if rows >= cus:
        thirds = W >= 4 and rows > cus and 3 * rows <= 4 * cus
        return 3 if thirds and (N >= 1536 if rowb >= 128 else fmt == "int4" and N >= 4096) else 1
    down = W == 8 or (W == 4 and not (fmt == "int4" and cus // rows == 1))
    return max(1, min(cus // rows if down else -(-cus // rows), N // 32))


@pytest.mark.parametrize("fmt", ["fp16", "int8", "int4"])
@pytest.mark.parametrize("W", [2, 4, 8])
def test_split_choice(fmt, W):
    try:
        cus = fq.cu_count()
    except RuntimeError:
        cus = 256  # what the library assumes without a device
    for D in (64, 128):
        for N in (1, 31, 63, 64, 1535, 1536, 4095, 4096, 100000):
            for rows in (1, 3, 17, 48, 127, 128, 129, 255, 256, 257, 341, 342, 512, 2048):
                S = fq.choose_splits(rows, 1, N, D, CODE[fmt], W)
                assert S == split_model(rows, N, D, fmt, W, cus), (D, N, rows)
                if rows < cus and S > 1 and W == 8:
                    assert rows * S <= cus


def make(fmt, g, B, N, D):
    q = torch.randn(B, D, generator=g).half()
    K, V = torch.randn(B, N, D, generator=g), torch.randn(B, N, D, generator=g)
    if fmt == "fp16":
        K, V = K.half(), V.half()
        return q, (K, V), (K.numpy(), V.numpy())
    f = quant.quant_int8_per_token if fmt == "int8" else quant.quant_int4_per_token
    back = oracle.dequant_int8 if fmt == "int8" else oracle.dequant_int4
    (Kq, Ks), (Vq, Vs) = f(K), f(V)
    return q, (Kq, Vq, Ks, Vs), (back(Kq.numpy(), Ks.numpy()), back(Vq.numpy(), Vs.numpy()))


@pytest.mark.gpu
@pytest.mark.parametrize("fmt,B,N,D,W", [
    ("fp16", 48, 333, 64, 8),    # 6 -> 5 splits of 67
    ("int8", 129, 200, 128, 8),  # unsplit just above half the CUs
    ("int4", 129, 200, 64, 4),   # two splits: 4 waves of int4
    ("fp16", 255, 65, 128, 8),
    ("fp16", 257, 1536, 64, 8),  # thirds, first row count and length
    ("fp16", 257, 1535, 64, 8),  # one token short of them
    ("int8", 341, 1537, 128, 8),  # last row count, ragged thirds
    ("int8", 342, 1537, 128, 4),
    ("int4", 300, 4097, 64, 8),
])
def test_gpu_calls_around_the_split_rule(fmt, B, N, D, W):
    g = torch.Generator().manual_seed(B + N)
    q, dev, (K, V) = make(fmt, g, B, N, D)
    fn = {"fp16": fq.decode_attn_fp16_mw, "int8": fq.decode_attn_int8_mw, "int4": fq.decode_attn_int4}[fmt]
    args = [t.cuda() for t in dev]
    pick = [0, 1, B // 2, B - 2, B - 1]  # rows of both ends and the middle
    want = oracle.attention(q.numpy()[pick], K[pick], V[pick])
    out = fn(q.cuda(), *args, W)
    assert float(np.abs(out.float().cpu().numpy()[pick] - want).max()) <= TOL
    # every other row: the same rows alone, whose split count differs
    for a in (0, B - 7):
        sub = fn(q[a:a + 7].cuda(), *[t[a:a + 7].contiguous() for t in args], W)
        assert float((out[a:a + 7].float() - sub.float()).abs().max()) <= TOL
