"""The matrix-core screen encode (ssq_encode_tile.hip) against the exact scan (kernel 1, pinned to the
oracle in test_gpu_encode.py and test_gpu_wide_codes.py), bit for bit, at the sizes where its tiles,
stages, chunks and lists end: key counts around 32 and 512, padded block dims, codebooks around a
stage's end, every key type, aligned and odd key rows, folded and paged outputs, metrics, and
codebooks whose ties put every pair on the full scan.
"""

import pytest
import torch

from sunshape_amd import hip_ops

from _util import time_us

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _codec(D, bd, nc, heads, seed):
    g = torch.Generator().manual_seed(seed)
    sig = torch.exp(torch.rand(D, generator=g) * 3.4 - 2.3)
    perm = torch.randperm(D, generator=g)
    cent = torch.randn(heads, D // bd, nc, bd, generator=g) * sig[perm].view(D // bd, 1, bd)
    return sig, perm.to(DEV), cent.to(DEV)


def _screened(keys, cent):
    """Whether a call past 256 codewords takes the screen: block dims 3 to 8, at least 32 keys per KV head and
    more than 2^24 (key, block, codeword) triples."""
    n = keys.shape[0] * keys.shape[2]
    return cent.shape[-1] >= 3 and n >= 32 and n * keys.shape[1] * cent.shape[-3] * cent.shape[-2] > 1 << 24


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
    odd.copy_((torch.randn(1, 2, 300, D, generator=g) * sig).to(dtype))
    _both(odd, perm, cent)


@pytest.mark.parametrize("bd", [3, 4, 8])
@pytest.mark.parametrize("nc", [257, 512, 1023, 1025, 2500])
def test_tile_codebooks_past_256(bd, nc):
    """Codebooks that end inside, at and just past a 1,024- or 512-codeword stage, and one codeword
    into a tile; bf16 keys (exact in one part), fp32 keys (two parts) and fp32 keys that hold bf16
    values; 16-bit codes."""
    D = 48
    sig, perm, cent = _codec(D, bd, nc, 1, nc)
    keys = torch.randn(1, 1, 11000, D, generator=torch.Generator().manual_seed(nc + bd)) * sig
    least = (1 << 24) // (D // bd * nc) + 1  # the smallest call on the screen
    for k in (keys.bfloat16(), keys, keys.bfloat16().float(), keys.half()):
        for n in (11000, least):
            assert _screened(k[:, :, :n], cent)
            _both(k[:, :, :n].to(DEV), perm, cent[0])
    assert not _screened(keys[:, :, :least - 1], cent)  # the last call on the scan, split over lanes
    _both(keys[:, :, :least - 1].to(DEV), perm, cent[0])


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
    n = 700 if nc == 256 else 1600  # past 256 codewords: enough for the screen
    keys = torch.randn(1, 1, n, D, generator=torch.Generator().manual_seed(n)) * sig
    assert nc == 256 or _screened(keys, cent)
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
    g = torch.Generator().manual_seed(nc)
    keys = (torch.randn(B, 2, S, D, generator=g) * sig).bfloat16().to(DEV)
    assert nc == 256 or _screened(keys, cent)
    heavy = [b in (0, 9, 31) for b in range(D // bd)]
    _both(keys, perm, cent, heavy=heavy)
    _both(keys, perm, cent, heavy=heavy, pt_dense=True, pt_dtype=torch.float32)
    E = (torch.eye(D) + 0.2 * torch.randn(D, D, generator=g)).to(DEV)
    _both(keys, perm, cent, metric=E)
    rep = perm.clone()
    rep[3] = rep[90]
    _both(keys, rep, cent)
    slots = torch.randperm(B * S, generator=g).view(B, S).to(DEV)
    pages = [torch.zeros((B * S + 15) // 16, 2, 16, D // bd, dtype=hip_ops.index_dtype(nc), device=DEV) for _ in range(2)]
    for out, kernel in zip(pages, (0, 1)):
        hip_ops.encode(keys, perm, cent, codes_out=out, slot_mapping=slots, kernel=kernel)
    assert torch.equal(pages[0], pages[1])


@pytest.mark.parametrize("nc,bd", [(256, 4), (256, 1), (256, 10), (700, 4), (1500, 3), (600, 8)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_tile_offsets(nc, bd, dtype):
    """Keys and codewords that share an offset per dim, up to where rounding hides the differences (every
    pair on the list, which fills at each block), one that only the keys have, and one that only half
    of the codewords have."""
    D = {3: 48, 10: 80}.get(bd, 64)
    _, perm, cent = _codec(D, bd, nc, 2, nc + bd)
    n = 1111 if nc == 256 else 2000
    for i, (off, cut) in enumerate(((0.7, 1.0), (10.0, 1.0), (300.0, 1.0), (5.0, 0.0), (20.0, 0.5))):
        g = torch.Generator().manual_seed(i)
        ch = torch.randn(D, generator=g).sign() * off * (1 + torch.rand(D, generator=g))
        keys = torch.randn(1, 2, n, D, generator=g) + ch
        c = cent.clone()
        c[:, :, :int(nc * cut)] += ch.to(DEV)[perm].view(D // bd, 1, bd)
        assert nc == 256 or _screened(keys, c)
        _both(keys.to(dtype).to(DEV), perm, c)
        if nc == 256:  # few keys: chunks of one or two blocks, whose codewords are still in LDS
            _both(keys[:, :, :90].to(dtype).to(DEV), perm, c)
    E = (torch.eye(D) + 0.2 * torch.randn(D, D, generator=g)).to(DEV)
    _both(keys.to(dtype).to(DEV), perm, c, metric=E)


def _offset_problem(n, H, D, bd, nc, dtype, off):
    g = torch.Generator(device=DEV).manual_seed(1)
    perm = torch.randperm(D, generator=g, device=DEV)
    cent = torch.randn(H, D // bd, nc, bd, generator=g, device=DEV) + off
    return (torch.randn(1, H, n, D, generator=g, device=DEV) + off).to(dtype), perm, cent


@pytest.mark.parametrize("nc,dtype,n", [(256, torch.float16, 4096), (256, torch.bfloat16, 4096),
                                        (4096, torch.float32, 2048), (4096, torch.bfloat16, 2048)])
def test_tile_time_at_an_offset(nc, dtype, n):
    """An offset of ten standard deviations that keys and codewords share costs at most twice the centred
    call (1.05 to 1.5 times; a screen whose bound grows with |x|^2, 1.8 to 13 times), and 30 no more than
    twice the exact scan past 256 codewords, five times the centred call at 256 (1.3; 10 to 17)."""
    base = time_us(lambda a=_offset_problem(n, 8, 128, 4, nc, dtype, 0.0): hip_ops.encode(*a))
    ten = time_us(lambda a=_offset_problem(n, 8, 128, 4, nc, dtype, 10.0): hip_ops.encode(*a))
    far = _offset_problem(n, 8, 128, 4, nc, dtype, 30.0)
    thirty = time_us(lambda: hip_ops.encode(*far))
    limit = 5 * base if nc == 256 else 2 * time_us(lambda: hip_ops.encode(*far, kernel=1))
    assert ten < 2 * base and thirty < limit, (base, ten, thirty, limit)


@pytest.mark.parametrize("n,H,D,bd,nc", [(1024, 1, 128, 2, 300), (2048, 8, 128, 1, 1024), (8, 8, 128, 4, 65535)])
def test_wide_calls_that_stay_on_the_scan(n, H, D, bd, nc):
    """Few keys, and codebooks of dims 1 and 2: the exact scan serves them faster than the screen (2 to 6 times)."""
    a = _offset_problem(n, H, D, bd, nc, torch.bfloat16, 0.0)
    assert time_us(lambda: hip_ops.encode(*a)) < 1.3 * time_us(lambda: hip_ops.encode(*a, kernel=1))


@pytest.mark.parametrize("bd", [4, 8])
def test_tile_metric_time(bd):
    """A step's keys under a block metric: at most three times the call without one (1.7 to 2; with E_b read from
    memory for each codeword, more than 3)."""
    a = _offset_problem(8, 8, 128, bd, 256, torch.bfloat16, 0.0)
    E = torch.eye(128, device=DEV) + 0.2 * torch.randn(128, 128, generator=torch.Generator().manual_seed(2)).to(DEV)
    plain, metric = time_us(lambda: hip_ops.encode(*a)), time_us(lambda: hip_ops.encode(*a, metric=E))
    assert metric < 3 * plain, (plain, metric)
