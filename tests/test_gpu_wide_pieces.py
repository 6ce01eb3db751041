"""Staged-codebook decode (ssq_decode_wide.hip) at the edges of its register and tile sizes: rows of 8 to
64 blocks (at most 32 blocks' codes are in registers at a time), splits of 2,048 tokens (2 per thread)
and more (4 per thread), tails of one token, 64 and 128 value dims, 1 and up to 4 query rows, pages.

Against the same call split into 256-token splits, which gathers codewords per token (k_decode_generic,
compared with the oracle in test_gpu_wide_codes.py).  Raw scores are equal bit for bit.  Both outputs
are fp32 sums rounded once to 16 bits (2^-9 of each, bf16), so they differ by at most 2^-8 of the largest
plus the fp32 sums' own error, far below that."""

import math

import pytest
import torch

from sunshape_amd import hip_ops

from _util import time_us

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("T,splits", [(2048, 1), (2049, 1), (4096, 1), (4097, 1), (8193, 2)])
@pytest.mark.parametrize("D,bd,nc,Dv,Hq,paged,dtype", [
    (128, 2, 1024, 128, 4, False, torch.bfloat16),  # 64 blocks: the row in two parts
    (80, 2, 512, 64, 3, True, torch.float16),       # 40 blocks: the second part has one piece
    (96, 4, 4096, 128, 1, True, torch.bfloat16),    # 24 blocks, one query row
    (32, 4, 2048, 64, 2, False, torch.float16),     # 8 blocks
    (64, 4, 512, 64, 4, True, torch.bfloat16),      # 16 blocks, pages of 64 value dims: two 16-token runs
    (64, 4, 512, 64, 2, False, torch.bfloat16),     # at a time, as contiguous rows of 64 dims
    (32, 2, 512, 64, 2, True, torch.float16),       # two query rows
])
def test_row_pieces_and_tails(D, bd, nc, Dv, Hq, paged, dtype, T, splits):
    g = torch.Generator().manual_seed(T + D)
    gd = torch.Generator(device=DEV).manual_seed(T + D)
    nb = D // bd
    perm = torch.randperm(D, generator=g).to(DEV)
    cent = torch.randn(1, nb, nc, bd, generator=gd, device=DEV)
    q = torch.randn(1, Hq, 1, D, generator=gd, device=DEV, dtype=dtype)
    codes = torch.randint(0, nc, (1, 1, T, nb), generator=gd, device=DEV, dtype=torch.int16)
    v = torch.randn(1, 1, T, Dv, generator=gd, device=DEV, dtype=dtype)
    v[0, 0, T - 1, 5] = float("inf")  # the last token's, read again for the slots past it
    kw = dict(scale=1 / math.sqrt(D), return_lse=True, return_scores=True)
    if paged:
        n = (T + 15) // 16
        pool = torch.randperm(n, generator=g).to(DEV)
        cp = torch.zeros(n, 1, 16, nb, dtype=codes.dtype, device=DEV)
        vp = torch.zeros(n, 1, Dv, 16, dtype=dtype, device=DEV)
        pad = n * 16 - T
        cp[pool] = torch.nn.functional.pad(codes[0, 0], (0, 0, 0, pad)).view(n, 1, 16, nb)
        vp[pool] = torch.nn.functional.pad(v[0, 0], (0, 0, 0, pad)).view(n, 16, Dv).transpose(1, 2).unsqueeze(1)
        args = (q, cp, vp, perm, cent)
        kw.update(block_table=pool.view(1, n).to(torch.int32),
                  seq_lens=torch.tensor([T], dtype=torch.int32, device=DEV))
    else:
        args = (q, codes, v, perm, cent)
    out, lse, sc = hip_ops.decode(*args, num_splits=splits, **kw)
    ref, lse_r, sc_r = hip_ops.decode(*args, num_splits=(T + 255) // 256, **kw)
    assert torch.equal(sc[..., :T], sc_r[..., :T])
    assert torch.isinf(out[..., 5]).all() and torch.isinf(ref[..., 5]).all()
    out[..., 5] = ref[..., 5] = 0
    assert torch.isfinite(out).all()
    assert float((out.float() - ref.float()).abs().max()) <= 2.0 ** -8 * float(ref.float().abs().max())
    assert float((lse - lse_r).abs().max()) <= 1e-6 * float(lse_r.abs().max())


@pytest.mark.parametrize("Hq", [8, 32])
def test_pages_time_at_64_dims(Hq):
    """Pages of 64 value dims take at most 1.25 times the contiguous rows' time (1.08 to 1.13; with one 16-token run
    loaded at a time, 1.35 to 1.42)."""
    B, Hkv, T, D, bd, nc = 16, 8, 8192, 64, 4, 512
    gd = torch.Generator(device=DEV).manual_seed(5)
    perm = torch.randperm(D, generator=gd, device=DEV)
    cent = torch.randn(Hkv, D // bd, nc, bd, generator=gd, device=DEV)
    q = torch.randn(B, Hq, 1, D, generator=gd, device=DEV, dtype=torch.bfloat16)
    codes = torch.randint(0, nc, (B, Hkv, T, D // bd), generator=gd, device=DEV, dtype=torch.int16)
    v = torch.randn(B, Hkv, T, D, generator=gd, device=DEV, dtype=torch.bfloat16)
    table = torch.randperm(B * T // 16, generator=gd, device=DEV).view(B, T // 16).to(torch.int32)
    lens = torch.full((B,), T, dtype=torch.int32, device=DEV)
    rows = time_us(lambda: hip_ops.decode(q, codes, v, perm, cent, scale=0.125))
    cp, vp = codes.view(B * T // 16, Hkv, 16, D // bd), v.view(B * T // 16, Hkv, D, 16)
    pages = time_us(lambda: hip_ops.decode(q, cp, vp, perm, cent, scale=0.125, block_table=table, seq_lens=lens))
    assert pages < 1.25 * rows, (pages, rows)
