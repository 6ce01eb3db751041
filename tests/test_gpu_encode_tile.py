"""The matrix-core screen encode (ssq_encode_tile.hip) against the exact scan (kernel 1, pinned to the
oracle in test_gpu_encode.py and test_gpu_wide_codes.py), bit for bit, at the sizes where its tiles,
stages, chunks and lists end: key counts around 32 and 512, padded block dims, codebooks around a
stage's end, every key type, aligned and odd key rows, folded and paged outputs, metrics, and
codebooks whose ties put every pair on the full scan.
"""

import pytest
import torch

from sunshape_amd import hip_ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _codec(D, bd, nc, heads, seed):
    g = torch.Generator().manual_seed(seed)
    sig = torch.exp(torch.rand(D, generator=g) * 3.4 - 2.3)
    perm = torch.randperm(D, generator=g)
    cent = torch.randn(heads, D // bd, nc, bd, generator=g) * sig[perm].view(D // bd, 1, bd)
    return sig, perm.to(DEV), cent.to(DEV)


def _both(keys, perm, cent, **kw):
    got = hip_ops.encode(keys, perm, cent, **kw)
    ref = hip_ops.encode(keys, perm, cent, kernel=1, **kw)
    assert torch.equal(got[0], ref[0]), int((got[0] != ref[0]).sum())
    if ref[1] is not None:
        assert torch.equal(got[1], ref[1])


@pytest.mark.parametrize("bd,D", [(1, 48), (2, 64), (3, 48), (4, 128), (5, 40), (8, 64), (10, 60)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_tile_key_counts_and_block_dims(bd, D, dtype):
    """Key counts at the edges of a wave's 32 and a workgroup's 512, in one long and in folded short
    sequences; block dims 1, 3, 5 and 10 are padded."""
    sig, perm, cent = _codec(D, bd, 256, 2, bd)
    for B, S in ((1, 1), (3, 11), (1, 33), (2, 511), (1, 513), (1, 1057)):
        g = torch.Generator().manual_seed(S)
        keys = (torch.randn(B, 2, S, D, generator=g) * sig).to(dtype).to(DEV)
        _both(keys, perm, cent)
    odd = torch.empty(1, 2, 300, D + 1, dtype=dtype, device=DEV)[..., :D]  # rows off 16-byte alignment
    odd.copy_((torch.randn(1, 2, 300, D) * sig).to(dtype))
    _both(odd, perm, cent)


@pytest.mark.parametrize("bd", [2, 3, 4, 8])
@pytest.mark.parametrize("nc", [257, 512, 1023, 1025, 2500])
def test_tile_codebooks_past_256(bd, nc):
    """Codebooks that end inside, at and just past a 1,024- or 512-codeword stage, and one codeword
    into a tile; bf16 keys (exact in one part), fp32 keys (two parts) and fp32 keys that hold bf16
    values; 16-bit codes."""
    D = 48
    sig, perm, cent = _codec(D, bd, nc, 1, nc)
    keys = torch.randn(1, 1, 11000, D) * sig  # more than 2^24 (key, block, codeword) triples: the screen
    for k in (keys.bfloat16(), keys, keys.bfloat16().float(), keys.half()):
        _both(k.to(DEV), perm, cent[0])
        _both(k[:, :, :700].to(DEV), perm, cent[0])  # the screen or, up to 2^24, the scan
    _both(keys[:, :, :5].to(DEV), perm, cent[0])


@pytest.mark.parametrize("nc", [256, 700])
@pytest.mark.parametrize("ties", ["equal", "pairs", "nan", "huge"])
def test_tile_ties_and_extreme_codebooks(nc, ties):
    """Every pair on the full scan: equal codewords overflow the workgroup's list, duplicated ones fill
    it partly, a NaN codeword is the reference's first minimum, squares past 2^120 have no bound."""
    D, bd = 64, 4
    sig, perm, cent = _codec(D, bd, nc, 1, 7)
    cent = cent[0]
    if ties == "equal":
        cent[:] = cent[:, :1]
    elif ties == "pairs":
        cent[:, 1::2] = cent[:, 0::2][:, :cent[:, 1::2].shape[1]]
    elif ties == "nan":
        cent[3, 77, 1] = float("nan")
        cent[5, 200] = float("inf")
    else:
        cent[2] *= 1e19
    keys = torch.randn(1, 1, 700, D) * sig
    keys[0, 0, 5] = 1e25
    keys[0, 0, 6, 3] = float("nan")
    keys[0, 0, 7] = 0
    _both(keys.bfloat16().to(DEV), perm, cent)


@pytest.mark.parametrize("nc", [256, 600])
def test_tile_heavy_pages_metric_and_repeated_dims(nc):
    """Passthrough blocks (compact and dense, their dims outside the staged chunk), paged outputs, a
    block metric, and a permutation that repeats a dim (gathered, not inverted)."""
    D, bd, B, S = 128, 4, 5, 130
    sig, perm, cent = _codec(D, bd, nc, 2, 11)
    keys = (torch.randn(B, 2, S, D) * sig).bfloat16().to(DEV)
    heavy = [b in (0, 9, 31) for b in range(D // bd)]
    _both(keys, perm, cent, heavy=heavy)
    _both(keys, perm, cent, heavy=heavy, pt_dense=True, pt_dtype=torch.float32)
    E = (torch.eye(D) + 0.2 * torch.randn(D, D)).to(DEV)
    _both(keys, perm, cent, metric=E)
    rep = perm.clone()
    rep[3] = rep[90]
    _both(keys, rep, cent)
    slots = torch.randperm(B * S, device=DEV).view(B, S)
    pages = [torch.zeros((B * S + 15) // 16, 2, 16, D // bd, dtype=hip_ops.index_dtype(nc), device=DEV) for _ in range(2)]
    for out, kernel in zip(pages, (0, 1)):
        hip_ops.encode(keys, perm, cent, codes_out=out, slot_mapping=slots, kernel=kernel)
    assert torch.equal(pages[0], pages[1])
