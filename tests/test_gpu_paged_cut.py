"""Length-balanced paged decode (SsqCut, ssq_decode_paged.h): batches of at least as many (sequence, KV
head) pairs as CUs and block tables of at least 4,096 tokens on the 4x4-MFMA kernel, against the same
call with one workgroup per pair (num_splits 1), whose results test_gpu_decode*.py compares with the
oracle.

Lengths sit at the edges of pages, tiles and shares; sequences span several shares, share one, or are
empty.  Short or like lengths are not cut: each sequence is then one workgroup's, bit for bit as with
num_splits 1.  Cut, both runs round their probabilities to 16 bits against their own running maxima (2^-9 of each,
so 2^-9 of the p-weighted mean of |v| per run: at most 1 for long sequences of N(0, 1) values, at most
the largest output for short ones) and their outputs (2^-9 of each): |a - b| <= 2^-8 (1 + 2 max|b|).
lse and raw scores agree within fp32 rounding.
"""

import math

import pytest
import torch

from sunshape_amd import hip_ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _problem(lens, Hq, Hkv, D, bd, nc, heavy=0, dtype=torch.bfloat16, seed=0):
    g = torch.Generator().manual_seed(seed)
    nb, B = D // bd, len(lens)
    T = max(max(lens), 4096)
    perm = torch.randperm(D, generator=g).to(DEV)
    cent = torch.randn(Hkv, nb, nc, bd, generator=g).to(DEV)
    width = (T + 15) // 16
    pages = [(n + 15) // 16 for n in lens]
    pool = torch.randperm(sum(pages), generator=g).to(torch.int32)
    table = torch.zeros(B, width, dtype=torch.int32)
    at = 0
    for b, n in enumerate(pages):
        table[b, :n] = pool[at:at + n]
        at += n
    gd = torch.Generator(device=DEV).manual_seed(seed)
    codes = torch.randint(0, nc, (at, Hkv, 16, nb), generator=gd, device=DEV, dtype=torch.uint8)
    v = torch.randn(at, Hkv, D, 16, generator=gd, device=DEV, dtype=dtype)
    q = torch.randn(B, Hq, 1, D, generator=gd, device=DEV, dtype=dtype)
    kw = dict(scale=1 / math.sqrt(D), block_table=table.to(DEV),
              seq_lens=torch.tensor(lens, dtype=torch.int32, device=DEV), return_lse=True)
    if heavy:
        kw["heavy"] = [b < heavy for b in range(nb)]
        kw["pt"] = torch.randn(at, Hkv, 16, heavy, bd, generator=gd, device=DEV, dtype=dtype)
    return (q, codes, v, perm, cent), kw


def _compare(args, kw, scores=False, cut=True):
    got = hip_ops.decode(*args, **kw, return_scores=scores)
    ref = hip_ops.decode(*args, **kw, return_scores=scores, num_splits=1)
    assert torch.equal(got[0].nan_to_num(7), ref[0].nan_to_num(7)) != cut
    for name, a, b in zip(("out", "lse", "scores"), got, ref):
        assert torch.equal(torch.isfinite(a), torch.isfinite(b)), name
        a, b = a.float().nan_to_num(0, 0, 0), b.float().nan_to_num(0, 0, 0)
        top = float(b.abs().max())
        tol = 2.0 ** -8 * (1 + 2 * top) if name == "out" else 1e-6 * top
        assert float((a - b).abs().max()) <= tol, (name, float((a - b).abs().max()))


EDGES = [1, 15, 16, 17, 63, 64, 65, 127, 448, 511, 512, 513, 896, 897, 1025]


@pytest.mark.parametrize("case", ["one_long", "edges", "many", "equal", "empty", "short_edges", "short_many",
                                  "short_equal", "short_empty"])
def test_cut_lengths(case):
    g = torch.Generator().manual_seed(3)
    lens = {"one_long": [9000] + [3] * 39,                     # one sequence over almost every share
            "edges": (EDGES * 3)[:40] + [6001],
            "many": torch.randint(1, 700, (131,), generator=g).tolist() + [9000],  # three chunks of 64 lengths
            "equal": [5000] * 48,
            "empty": [0, 700, 0, 5] * 10 + [5100],
            "short_edges": [n for n in EDGES if n < 600] * 4,
            "short_many": torch.randint(1, 300, (131,), generator=g).tolist(),
            "short_equal": [1500] * 48,
            "short_empty": [0, 70, 0, 5] * 10 + [210]}[case]
    args, kw = _problem(lens, 32, 8, 128, 2, 256)
    _compare(args, kw, scores=case in ("edges", "one_long", "short_edges"), cut=not case.startswith("short"))


@pytest.mark.parametrize("Hq,Hkv,D,bd,nc,heavy,dtype", [
    (6, 2, 128, 2, 256, 0, torch.bfloat16),   # 3 rows per KV head
    (32, 8, 128, 4, 256, 4, torch.bfloat16),  # passthrough values as vectors
    (32, 8, 128, 8, 100, 0, torch.float16),
    (16, 8, 128, 2, 64, 0, torch.float16),
])
def test_cut_variants(Hq, Hkv, D, bd, nc, heavy, dtype):
    g = torch.Generator().manual_seed(Hq + bd)
    B = -(-264 // Hkv)
    lens = torch.exp(torch.rand(B, generator=g) * 8).int().clamp(1, 2900).tolist()
    lens[1] = 5900
    _compare(*_problem(lens, Hq, Hkv, D, bd, nc, heavy, dtype, seed=5))


def test_cut_graph_replay():
    """Captured and replayed with eager calls between, the lengths changed in place: each replay follows
    the lengths it finds."""
    args, kw = _problem([6000] + [1200] * 39, 32, 8, 128, 2, 256)
    hip_ops.decode(*args, **kw)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out, lse = hip_ops.decode(*args, **kw)
    for lens in ([1200] * 40, [5900] + [1, 1200] * 19 + [1], [700] + [64] * 39, [6000] + [1200] * 39):
        kw["seq_lens"].copy_(torch.tensor(lens, dtype=torch.int32))
        graph.replay()
        torch.cuda.synchronize()
        ref, ref_lse = hip_ops.decode(*args, **kw)
        assert torch.equal(out, ref) and torch.equal(lse, ref_lse)


def test_cut_infinite_values():
    """An infinite value under a probability that underflows makes its output NaN (0 times infinity), whichever
    workgroups the sequence is cut between."""
    args, kw = _problem([9000] + [3] * 39, 32, 8, 128, 2, 256)
    args[2][kw["block_table"][0, ::97].long(), :, 5, 3] = float("inf")
    kw["scale"] = 30.0  # the shares' maxima lie hundreds apart
    got, ref = hip_ops.decode(*args, **kw), hip_ops.decode(*args, **kw, num_splits=1)
    assert not torch.isfinite(ref[0][0, :, :, 5]).any()
    assert torch.equal(torch.isfinite(got[0]), torch.isfinite(ref[0]))
