"""The work-balanced paged kernel (one line of 16-token tiles over all sequences, cut into equal
spans) against the float64 oracle at max-abs 2e-3, the tolerance of every paged test: sequence
lengths at the edges of tiles, of a wave's part and of a workgroup's span, empty sequences, lengths
that cut every row alike, lines shorter than the grid, more sequences than one scan block holds,
and lengths that change between graph replays. A large max_seq_len (what the call could hold)
selects the kernel, whatever the sequences hold; unsplit calls of the other kernel report no merge."""

import numpy as np
import pytest
import torch

import oracle
import fqkv_decode as fq

pytestmark = pytest.mark.gpu

TOL = 2e-3


def draw(g, *shape):
    return torch.randn(*shape, generator=g, dtype=torch.float32)


def quantize(fmt, X):
    if fmt == "int8":
        q, s = fq.quantize_int8_per_token(X.cuda())
        return q, s, oracle.dequant_int8(q.cpu().numpy(), s.cpu().numpy())
    if fmt == "fp8":
        q, s = fq.quantize_fp8_per_token(X.cuda())
        return q, s, oracle.dequant_fp8(q.view(torch.uint8).cpu().numpy(), s.cpu().numpy())
    q, s = fq.quantize_int4_per_token(X.cuda())
    return q, s, oracle.dequant_int4(q.cpu().numpy(), s.cpu().numpy())


class Cache:
    """Shuffled pages holding `lens` tokens per sequence; unused slots hold NaN scales (or values)."""

    def __init__(self, g, lens, Hkv, D, page, fmt, hnd, max_seq):
        npages = [-(-n // page) for n in lens]
        P = sum(npages) + 2
        ids = torch.randperm(P, generator=g).to(torch.int32)
        self.table = torch.full((len(lens), -(-max_seq // page)), -1, dtype=torch.int32)
        k = 0
        for b, n in enumerate(npages):
            self.table[b, :n] = ids[k:k + n]
            k += n
        X = draw(g, 2, P, page, Hkv, D)
        used = torch.zeros(P, page, dtype=torch.bool)
        for b, n in enumerate(lens):
            for j in range(npages[b]):
                used[self.table[b, j], :min(page, n - j * page)] = True
        if fmt in ("fp16", "bf16"):
            X = X.to(torch.float16 if fmt == "fp16" else torch.bfloat16)
            self.f = [x.float().numpy() for x in X]
            self.kv, self.sc = [x.cuda() for x in X], [None, None]
        else:
            parts = [quantize(fmt, x) for x in X]
            self.kv, self.f = [p[0] for p in parts], [p[2] for p in parts]
            self.sc = [p[1].masked_fill(~used.cuda()[:, :, None], float("nan")) for p in parts]
        if hnd:
            self.kv = [x.transpose(1, 2).contiguous().transpose(1, 2) for x in self.kv]
            self.sc = [None if x is None else x.transpose(1, 2).contiguous().transpose(1, 2) for x in self.sc]
        self.lens, self.page, self.max_seq = lens, page, max_seq

    def run(self, q, lens=None, W=8):
        sl = torch.tensor(self.lens if lens is None else lens, dtype=torch.int32).cuda()
        return fq.decode_attn_gqa_paged(q.cuda(), self.kv[0], self.kv[1], self.table.cuda(), sl, self.max_seq, W,
                                        self.sc[0], self.sc[1])

    def check(self, q, out, lens=None):
        out = out.float().cpu().numpy().astype(np.float64)
        for b, n in enumerate(self.lens if lens is None else lens):
            if n == 0:
                assert not out[b].any(), b
                continue
            t = np.arange(n)
            pid, pos = self.table[b, t // self.page].numpy(), t % self.page
            K, V = (f[pid, pos].transpose(1, 0, 2) for f in self.f)
            ref = oracle.gqa_attention(q.numpy()[b:b + 1], K[None], V[None])[0]
            err = np.abs(out[b] - ref).max()
            assert err <= TOL, (b, n, err)


def ragged(seed, B, most):
    edges = [0, 1, 15, 16, 17, 63, 64, 65, 255, 256, 257, 0, 511, 512, 513]
    r = np.random.RandomState(seed)
    lens = (edges + [int(most ** r.rand()) for _ in range(B)])[:B]
    lens[-1] = most
    return [int(x) for x in r.permutation(lens)]


CASES = [  # fmt, D, Hq, Hkv, page, hnd, B: head groups of 1, 4, 8 (7 used) and 16 (two groups: 24 heads)
    ("fp16", 128, 32, 8, 16, False, 33), ("fp16", 64, 8, 8, 64, True, 33), ("fp16", 128, 96, 4, 32, True, 40),
    ("bf16", 128, 32, 8, 32, True, 33), ("bf16", 64, 56, 8, 16, False, 33),
    ("int8", 128, 32, 8, 64, True, 33), ("int8", 64, 64, 4, 16, False, 65), ("int8", 128, 7, 1, 32, False, 260),
    ("fp8", 128, 32, 8, 64, True, 33), ("fp8", 128, 96, 6, 16, False, 45),
    ("int4", 128, 32, 8, 32, False, 33), ("int4", 64, 32, 8, 16, False, 33), ("int4", 128, 8, 8, 64, True, 33),
]


@pytest.mark.parametrize("fmt,D,Hq,Hkv,page,hnd,B", CASES)
def test_ragged_lengths(fmt, D, Hq, Hkv, page, hnd, B, merge_mode):
    g = torch.Generator().manual_seed(71)
    c = Cache(g, ragged(B + D, B, 3000), Hkv, D, page, fmt, hnd, 16384)
    q = draw(g, B, Hq, D).half()
    for W in (8, 2):
        out = c.run(q, W=W)
        assert fq._ext._last_merge_protocol() == (1 if merge_mode == "two_kernel" else 2) or (
            merge_mode == "fused" and fq._ext._last_merge_protocol() == 3)
        c.check(q, out)
        assert torch.equal(out, c.run(q, W=W))  # the arrival counters are back at zero


@pytest.mark.parametrize("fmt,D", [("fp16", 128), ("int8", 128), ("int4", 64)])
@pytest.mark.parametrize("n", [1, 16, 100, 1040, 2000])
def test_equal_lengths(fmt, D, n):
    """Every row cut alike (or, short, one span per row), and the same batch with one sequence a tile longer."""
    g = torch.Generator().manual_seed(72)
    B, Hq, Hkv = 32, 32, 8
    for lens in ([n] * B, [n] * (B - 1) + [n + 16]):
        c = Cache(g, lens, Hkv, D, 32, fmt, True, 16384)
        q = draw(g, B, Hq, D).half()
        c.check(q, c.run(q))


@pytest.mark.parametrize("B", [255, 256, 257, 600])
def test_many_sequences(B):
    """The scan over the lengths takes 256 sequences a block; most are a few tokens long."""
    g = torch.Generator().manual_seed(73)
    lens = [int(x) for x in np.random.RandomState(B).randint(0, 40, B)]
    lens[B // 2], lens[-1] = 1500, 700
    c = Cache(g, lens, 2, 64, 16, "fp16", False, 16384)
    q = draw(g, B, 8, 64).half()
    c.check(q, c.run(q))


def test_one_long_sequence_among_short_ones():
    g = torch.Generator().manual_seed(74)
    lens = [20000] + [3] * 31
    c = Cache(g, lens, 8, 128, 64, "int8", True, 32768)
    q = draw(g, 32, 32, 128).half()
    c.check(q, c.run(q))


def test_lengths_change_between_graph_replays():
    """A captured call finds its spans from the lengths at each replay."""
    g = torch.Generator().manual_seed(75)
    B, Hq, Hkv, D = 33, 32, 8, 128
    full = ragged(5, B, 2500)
    c = Cache(g, full, Hkv, D, 16, "fp16", False, 16384)
    q = draw(g, B, Hq, D).half()
    qd, table = q.cuda(), c.table.cuda()
    sl = torch.tensor(full, dtype=torch.int32).cuda()
    call = lambda: fq.decode_attn_gqa_paged(qd, c.kv[0], c.kv[1], table, sl, c.max_seq, 8)  # noqa: E731
    call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call()
    r = np.random.RandomState(9)
    for step in range(4):
        lens = [int(r.randint(0, n + 1)) for n in full] if step else full
        sl.copy_(torch.tensor(lens, dtype=torch.int32))
        eager = call().clone()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager), step
        c.check(q, out, lens)
