"""The work a program gives this library, as cases that can be timed and checked.

Each case is one call of a serving program: scoring a query against quantized keys, a decode step
over contiguous or paged codes, the short multi-token step of speculative verification, appending
a step's keys to code pages, quantizing a prompt's keys, and the dequantizing cache's round trip.
``prepare`` makes what the program holds before the call, ``run`` is the call, ``exact`` the same
result in 64 bits from plain torch.
"""

from __future__ import annotations

import math

import torch

from sunshape_amd import hip_ops
from sunshape_amd import vllm_attn_backend as backend
from sunshape_amd.cache import SunShapeCodedKeys, sunshape_attention_forward
from sunshape_amd.codec import SunShapeBlockCodec, SunShapeQuantized
from sunshape_amd.hf import SunShapeBundle
from sunshape_amd.integration.vllm import SunShapeVLLMRuntimeState
from sunshape_amd.kernels import sunshape_attention_scores

PAGE = 16
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}

# kind: what is called (see run).  B sequences, Hq / Hkv query and KV heads, head_dim D, block_dim
# bd, nc codewords per block, T tokens (the longest sequence's), Lq new tokens, heavy passthrough
# blocks (SunShape-Mixed), per_head: a codebook per KV head (else one per layer), pro: a SunShape-Pro
# block metric.
DEFAULTS = {"B": 1, "Hq": 32, "Hkv": 8, "D": 128, "bd": 2, "nc": 256, "T": 1, "Lq": 1, "heavy": 0, "ragged": False,
            "per_head": True, "pro": False, "dtype": "bf16"}


def _case(kind, **kw):
    return {**DEFAULTS, "kind": kind, **kw}


def listed():
    return [
        # the reference's own scoring call: one KV head's query group against 4,096 quantized keys
        _case("scores", name="scores_4k", Hq=7, Hkv=1, D=64, T=4096, per_head=False),
        # a chat's first tokens: one short sequence, where launches and host time are the cost
        _case("attend", name="attend_short", Hq=14, Hkv=2, D=64, T=517, per_head=False),
        # the small GQA layer (14/2 heads, head_dim 64) at the default 4 bits/dim, a full batch
        _case("attend", name="attend_8k", B=16, Hq=14, Hkv=2, D=64, T=8192),
        # the same layer as SunShape-Mixed (4 blocks kept in bf16) after a 16k prompt
        _case("attend", name="attend_mixed_16k", B=16, Hq=14, Hkv=2, D=64, T=16384, heavy=4),
        # speculative verification through the HF attention function: 8 new tokens over an odd length
        _case("verify", name="verify_8", B=4, T=4099, Lq=8, per_head=False),
        # continuous batching: 48 sequences of every length up to 8k in pages, 4 bits/dim, with lse
        _case("paged", name="paged_ragged_8k", B=48, T=8192, ragged=True),
        # the large decode step: 64 sequences of 32k in pages at 2 bits/dim
        _case("paged", name="paged_32k", B=64, T=32768, bd=4),
        # 3 bits/dim at block_dim 4 (4,096 codewords, 16-bit codes), contiguous, long contexts
        _case("attend", name="attend_3bit_16k", B=32, T=16384, bd=4, nc=4096),
        # one decode step's keys of 64 sequences into the code pages
        _case("append", name="append_64", B=64, T=32, bd=4),
        # prompts of the Mixed layer, quantized in one call
        _case("prefill", name="prefill_mixed_16k", B=16, Hq=14, Hkv=2, D=64, T=16384, heavy=4),
        # one long prompt at 2 bits/dim, block_dim 4
        _case("prefill", name="prefill_32k", T=32768, bd=4),
        # the dequantizing cache layer's update (fp32 keys -> codes -> fp32 keys) at 3 bits/dim
        _case("roundtrip", name="roundtrip_3bit_8k", T=8192, bd=4, nc=4096, per_head=False),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["scores", "attend", "attend", "verify", "paged", "paged", "append", "prefill", "prefill", "roundtrip"])
    hq, hkv, d = rng.choice([(14, 2, 64), (32, 8, 128), (32, 8, 128), (64, 8, 128)])
    # bits/dim x block_dim of the fitted codecs: 4, 2, 1, 3 (bd 2), 3 (bd 4), 5
    bd, nc = rng.choice([(2, 256), (2, 256), (4, 256), (4, 256), (8, 256), (2, 64), (4, 4096), (2, 1024)])
    c = {"Hq": hq, "Hkv": hkv, "D": d, "bd": bd, "nc": nc, "per_head": rng.random() < 0.5,
         "dtype": rng.choice(["bf16", "bf16", "f16"])}
    mixed = bd <= 4 and nc <= 256 and rng.random() < 0.25
    budget = 1 << 21  # keys of one call
    if kind == "scores":
        c.update(Hq=rng.choice([4, 7, 8, 32]), Hkv=1, T=_log(rng, 500, 131072), per_head=False)
    elif kind == "attend":
        c["B"] = _log(rng, 1, 64)
        c["T"] = _log(rng, 60, min(32768, budget // (c["B"] * hkv)))
        c["heavy"] = 4 if mixed else 0
    elif kind == "verify":
        c["B"] = _log(rng, 1, 16)
        c["Lq"] = rng.choice([2, 3, 4, 5, 8])
        c["T"] = _log(rng, 200, 16384)
    elif kind == "paged":
        c["B"] = _log(rng, 1, 128)
        c["T"] = _log(rng, 60, min(32768, budget // (c["B"] * hkv)))
        c["ragged"] = rng.random() < 0.6
        c["heavy"] = 4 if mixed else 0
    elif kind == "append":
        c["B"] = _log(rng, 1, 256)
        c["Lq"] = rng.choice([1, 1, 1, 2, 4])
        c["T"] = 32
    elif kind == "prefill":
        c["B"] = _log(rng, 1, 16)
        c["T"] = _log(rng, 30, min(32768, (1 << 18) // (c["B"] * hkv)))
        c["heavy"] = 4 if mixed else 0
        c["pro"] = not mixed and rng.random() < 0.15
    else:
        c["T"] = _log(rng, 30, 8192)
        c["per_head"] = False
    return _case(kind, **c)


# ------------------------------------------------------------------------------------- inputs
def _codec(c, g, dev):
    """Codec of the fitted form: one spread per dim, codewords drawn with it in the permuted basis."""
    D, bd, nc = c["D"], c["bd"], c["nc"]
    nb = D // bd
    heads = c["Hkv"] if c["per_head"] else 1
    sigma = torch.exp(torch.rand(D, generator=g, device=dev) * math.log(30.0) + math.log(0.1))
    perm = torch.randperm(D, generator=g, device=dev)
    spread = sigma[perm].view(nb, 1, bd)
    cent = torch.randn(heads, nb, nc, bd, generator=g, device=dev) * spread
    heavy = None
    mode = "profileperm_baseline"
    if c["heavy"]:
        mass = spread.square().sum((1, 2))
        heavy = torch.zeros(nb, dtype=torch.bool, device=dev)
        heavy[torch.topk(mass, c["heavy"]).indices] = True
        cent[:, heavy] = 0.0
        mode = "profileperm_mixed_precision"
    metric = None
    if c["pro"]:
        mode = "profileperm_localmetric_dsq"
        metric = torch.eye(D, device=dev) + 0.2 * torch.randn(D, D, generator=g, device=dev)
    codec = SunShapeBlockCodec.from_buffers(perm, cent if c["per_head"] else cent[0], mode=mode, metric=metric,
                                            mixed_high_precision_blocks=heavy, device=dev)
    return codec, sigma


def _codes(c, shape, g, dev):
    idx = torch.randint(0, c["nc"], shape, generator=g, device=dev, dtype=torch.int32)
    return idx.to(hip_ops.index_dtype(c["nc"]))


def _lengths(c, g, dev):
    if not c["ragged"]:
        return torch.full((c["B"],), c["T"], dtype=torch.int32, device=dev)
    # log-spread lengths, the longest one at T
    u = torch.rand(c["B"], generator=g, device=dev)
    lens = torch.exp(u * math.log(max(c["T"], 2))).round().to(torch.int32).clamp_(1, c["T"])
    lens[0] = c["T"]
    return lens


def prepare(case, seed):
    c = {**DEFAULTS, **case}
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(int(seed) * 7919 + 13)
    dt = DTYPES[c["dtype"]]
    codec, sigma = _codec(c, g, dev)
    B, Hq, Hkv, D, T, Lq = (c[k] for k in ("B", "Hq", "Hkv", "D", "T", "Lq"))
    nb, bd = D // c["bd"], c["bd"]
    s = {"case": c, "codec": codec, "scale": 1.0 / math.sqrt(D), "heavy": codec.heavy_blocks()}

    def randn(*shape):
        return torch.randn(*shape, generator=g, device=dev, dtype=dt)

    if c["kind"] == "scores":
        s["q"] = randn(Hq, D)
        s["key"] = SunShapeQuantized(indices=_codes(c, (T, nb), g, dev), head_dim=D, block_dim=bd, n_blocks=nb)
    elif c["kind"] in ("attend", "verify"):
        s["q"] = randn(B, Hq, Lq, D)
        # the HF cache layer's buffers grow in steps of 256 tokens; attention gets views of them
        cap = T if c["kind"] == "attend" else (T + 255) // 256 * 256
        codes = _codes(c, (B, Hkv, cap, nb), g, dev)
        pt = None
        if c["heavy"]:
            codes[..., codec.mixed_high_precision_blocks] = 0
            spread = sigma[codec.effective_permutation()[0] if c["per_head"] else codec.effective_permutation()]
            pt = (torch.randn(B, Hkv, T, c["heavy"], bd, generator=g, device=dev)
                  * spread.view(nb, bd)[codec.mixed_high_precision_blocks]).to(dt)
        s["v"] = randn(B, Hkv, cap, D)[:, :, :T]
        s["pt"] = pt
        s["codes"] = codes[:, :, :T]
        if c["kind"] == "attend":
            s["impl"] = backend.SunShapeAttentionImpl(layer_idx=0, runtime_state=_runtime(codec, bd))
            s["key"] = backend.SunShapeQuantizedKeys(quantized_heads=(), batch_size=B, num_kv_heads=Hkv, seq_len=T,
                                                     codes=s["codes"], passthrough=pt)
        else:
            s["key"] = SunShapeCodedKeys(s["codes"], None, codec, D, dt)
            s["module"] = torch.nn.Module()
            s["module"].is_causal = True
    elif c["kind"] == "paged":
        s["q"] = randn(B, Hq, Lq, D)
        lens = _lengths(c, g, dev)
        per = (lens.to(torch.int64) + PAGE - 1) // PAGE
        width, total = (T + PAGE - 1) // PAGE, int(per.sum())
        pool = torch.randperm(total, generator=g, device=dev).to(torch.int32)
        col = torch.arange(width, device=dev)
        first = torch.cumsum(per, 0) - per
        table = torch.where(col[None] < per[:, None], pool[(first[:, None] + col[None]).clamp_(max=total - 1)], 0)
        s["table"], s["lens"] = table.to(torch.int32).contiguous(), lens
        s["codes"] = _codes(c, (total, Hkv, PAGE, nb), g, dev)
        s["v"] = randn(total, Hkv, D, PAGE)
        s["pt"] = None
        if c["heavy"]:
            s["codes"][..., codec.mixed_high_precision_blocks] = 0
            spread = sigma[codec.effective_permutation()[0] if c["per_head"] else codec.effective_permutation()]
            s["pt"] = (torch.randn(total, Hkv, PAGE, c["heavy"], bd, generator=g, device=dev)
                       * spread.view(nb, bd)[codec.mixed_high_precision_blocks]).to(dt)
    else:
        n = Lq if c["kind"] == "append" else T
        keys = (torch.randn(B, Hkv, n, D, generator=g, device=dev) * sigma).to(dt)
        s["keys"] = keys
        codec.encode_search_grid(codec.codebook())  # kept by the codec from its first use on
        if c["kind"] == "append":
            pages = B * 2 + 64
            s["codes"] = torch.zeros(pages, Hkv, PAGE, nb, dtype=hip_ops.index_dtype(c["nc"]), device=dev)
            slots = torch.randperm(pages * PAGE // n, generator=g, device=dev)[:B] * n
            s["slots"] = slots[:, None] + torch.arange(n, device=dev)[None]
        elif c["kind"] == "prefill":
            s["runtime"] = _runtime(codec, bd)
        else:  # the cache layer hands the codec its keys in fp32, flattened
            s["keys"] = keys.reshape(-1, D).float()
    return s


def _runtime(codec, bd):
    bundle = SunShapeBundle("perf", [0], 0.0, bd, codec.mode, 0, 0, 0, {0: codec})
    return SunShapeVLLMRuntimeState("perf", "perf", codec.mode, 0.0, bd, [0], bundle, "cuda")


# ------------------------------------------------------------------------------------- the calls
def run(s):
    kind, codec = s["case"]["kind"], s["codec"]
    if kind == "scores":
        return sunshape_attention_scores(codec, s["q"], s["key"])
    if kind == "attend":
        return s["impl"](s["q"], s["key"], s["v"], scale=s["scale"])
    if kind == "verify":
        return sunshape_attention_forward(s["module"], s["q"], s["key"], s["v"], None, scaling=s["scale"])[0]
    if kind == "paged":
        out, lse = hip_ops.decode(s["q"], s["codes"], s["v"], codec.effective_permutation(), codec.codebook(),
                                  scale=s["scale"], heavy=s["heavy"], pt=s["pt"], block_table=s["table"],
                                  seq_lens=s["lens"], return_lse=True)
        return {"out": out, "lse": lse}
    if kind == "append":
        codes, _ = hip_ops.encode(s["keys"], codec.effective_permutation(), codec.codebook(), codes_out=s["codes"],
                                  slot_mapping=s["slots"], grid=codec.encode_search_grid(codec.codebook()),
                                  direct=hip_ops.cdist_direct(s["keys"].shape[2], codec.n_centroids))
        return codes
    if kind == "prefill":
        backend.register_runtime_state(s["runtime"])
        keys = backend.quantize_key_states(0, s["keys"])
        return {"codes": keys.codes, "passthrough": keys.passthrough}
    return codec(s["keys"])


# ------------------------------------------------------------------------------------- what it takes
def work(case):
    c = {**DEFAULTS, **case}
    D, nb, bd, B, Hkv = c["D"], c["D"] // c["bd"], c["bd"], c["B"], c["Hkv"]
    width = 1 if c["nc"] <= 256 else 2
    book = (Hkv if c["per_head"] else 1) * (nb * c["nc"] * bd * 4 + D * 8)
    if c["kind"] == "scores":
        keys = c["T"]
        return {"bytes": keys * (nb * width + 4 * c["Hq"]) + book + c["Hq"] * D * 2, "flops": float(c["Hq"] * keys * nb)}
    rows = B * c["Hq"] * c["Lq"]
    if c["kind"] in ("attend", "verify", "paged"):
        # a log-spread length's mean, over the sequences beside the longest
        mean = c["T"] if not c["ragged"] else (c["T"] + (B - 1) * (c["T"] - 1) / math.log(max(c["T"], 2))) / B
        keys = B * Hkv * mean
        return {"bytes": keys * (nb * width + 2 * D + 2 * c["heavy"] * bd) + 4 * rows * D + book,
                "flops": rows * mean * (2.0 * D + nb)}
    keys = B * Hkv * (c["Lq"] if c["kind"] == "append" else c["T"])
    flops = 3.0 * keys * D  # one distance per block
    if c["kind"] == "roundtrip":
        return {"bytes": keys * (8 * D + 2 * nb * width) + book, "flops": flops}
    return {"bytes": keys * (2 * D + nb * width + 2 * c["heavy"] * bd) + book, "flops": flops}


def tolerance(case):
    kind = case["kind"]
    if kind in ("append", "prefill", "roundtrip"):
        return "exact"  # indices, and values copied or looked up by them
    if kind == "scores":
        return {"rel": 1e-6}  # fp32 sums over the blocks in another order: 1.3e-7 to 3e-7 against 64 bits
    # 16-bit outputs, and probabilities rounded to 16 bits before P.V: 2.3e-3 (bf16) and 2e-4 (f16)
    return {"rel": 1e-2, "max": 1e-1} if case.get("dtype", "bf16") == "bf16" else {"rel": 1e-3, "max": 2e-2}


def _keys64(codec, codes, pt, heavy, head):
    """Keys of one KV head in the codec's basis, [T, D] in 64 bits."""
    cent = codec.codebook(head).double()
    nb, nc, bd = cent.shape
    idx = codes.to(torch.int64) % 65536
    k = cent.reshape(nb * nc, bd)[idx + torch.arange(nb, device=idx.device) * nc]
    if heavy is not None:
        k[:, torch.tensor(heavy, device=idx.device)] = pt.double()
    return k.reshape(k.shape[0], nb * bd)


def exact(case, seed):
    s = prepare(case, seed)
    c, codec, heavy = s["case"], s["codec"], s["heavy"]
    perm = codec.effective_permutation()
    kind = c["kind"]
    if kind == "scores":
        return s["q"].double()[:, perm] @ _keys64(codec, s["key"].indices, None, None, None).T
    if kind in ("attend", "verify", "paged"):
        return _attention64(s, c, codec, heavy, perm)
    if kind == "roundtrip":
        x = s["keys"].double()[:, perm].reshape(-1, codec.n_blocks, codec.block_dim)
        out = torch.empty_like(x)
        for b in range(codec.n_blocks):
            cb = codec.codebook()[b].double()
            for lo in range(0, x.shape[0], 16384):
                out[lo:lo + 16384, b] = cb[torch.cdist(x[lo:lo + 16384, b], cb).argmin(1)]
        res = torch.empty(x.shape[0], c["D"], dtype=torch.float64, device=x.device)
        res[:, perm] = out.reshape(x.shape[0], -1)
        return res
    if kind == "prefill" and heavy is not None:  # indices have no 64-bit value; the kept blocks do
        x = s["keys"].double()
        p = perm if perm.ndim == 1 else perm[0]
        x = x[..., p].reshape(*x.shape[:-1], codec.n_blocks, codec.block_dim)
        return {"codes": None, "passthrough": x[..., torch.tensor(heavy, device=x.device), :]}
    return None


def _attention64(s, c, codec, heavy, perm):
    B, Hq, Hkv, D, Lq = (c[k] for k in ("B", "Hq", "Hkv", "D", "Lq"))
    G = Hq // Hkv
    q = (s["q"] * s["scale"]).double()  # the query is scaled in its own type
    out = torch.empty(B, Hq, Lq, D, dtype=torch.float64, device=q.device)
    lse = torch.empty(B, Hq, Lq, dtype=torch.float64, device=q.device)
    lens = s["lens"].tolist() if c["kind"] == "paged" else [c["T"]] * B
    for b in range(B):
        T = lens[b]
        pages = s["table"][b, :(T + PAGE - 1) // PAGE].long() if c["kind"] == "paged" else None
        for h in range(Hkv):
            if pages is None:
                codes, v = s["codes"][b, h], s["v"][b, h]
                pt = None if s["pt"] is None else s["pt"][b, h]
            else:
                codes = s["codes"][pages, h].reshape(-1, codec.n_blocks)[:T]
                v = s["v"][pages, h].transpose(1, 2).reshape(-1, D)[:T]
                pt = None if s["pt"] is None else s["pt"][pages, h].reshape(-1, c["heavy"], codec.block_dim)[:T]
            head = h if c["per_head"] else None
            k = _keys64(codec, codes, pt, heavy, head)
            p = perm if perm.ndim == 1 else perm[h]
            rows = q[b, h * G:(h + 1) * G].reshape(G * Lq, D)[:, p]
            x = (rows @ k.T).view(G, Lq, T)
            if Lq > 1:  # the new tokens are the last Lq positions
                pos = torch.arange(T, device=q.device)
                x = x.masked_fill(pos[None, None] > (T - Lq + torch.arange(Lq, device=q.device))[None, :, None], -math.inf)
            x = x.reshape(G * Lq, T)
            lse[b, h * G:(h + 1) * G] = torch.logsumexp(x, -1).view(G, Lq)
            out[b, h * G:(h + 1) * G] = (torch.softmax(x, -1) @ v.double()).view(G, Lq, D)
    if c["kind"] == "paged":
        return {"out": out, "lse": lse}
    return out.transpose(1, 2).contiguous() if c["kind"] == "verify" else out
