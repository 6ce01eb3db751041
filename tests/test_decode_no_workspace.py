"""A batch that ssq_decode balances by length also runs without a workspace, unbalanced: callers that bring
none are not refused, and ssq_decode_noalloc does not put such a batch's partials into the scratch
that every call on the device shares."""

import math
import os
import subprocess
import sys

import pytest
import torch

from sunshape_amd import _native as N
from sunshape_amd import hip_ops

HERE = os.path.dirname(os.path.abspath(__file__))

# fake, aligned addresses: the plan and its checks only look at them, and without a GPU the launch
# fails at the runtime
CHILD = """
import ctypes, importlib.util, sys
spec = importlib.util.spec_from_file_location("ssq_abi", sys.argv[2])
abi = importlib.util.module_from_spec(spec)
spec.loader.exec_module(abi)
lib = ctypes.CDLL(sys.argv[1])
lib.ssq_decode_workspace_size.restype = ctypes.c_size_t
lib.ssq_last_error.restype = ctypes.c_char_p
lib.ssq_decode.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_void_p]
A = 1 << 32
a = abi.DecodeArgs(q=A, q_dtype=1, q_sb=4096, q_sh=128, q_sl=128, batch=48, num_q_heads=32, q_len=1, head_dim=128,
                   num_kv_heads=8, perm=A, cent=A, block_dim=2, n_blocks=64, n_centroids=256, layout=1, seq_len=8192,
                   codes=A, c_sb=8192, c_sh=1024, c_st=64, block_table=A, bt_sb=512, seq_lens=A, page_size=16,
                   v=A, v_dtype=1, value_dim=128, v_sb=16384, v_sh=2048, v_st=16, out=A, o_sb=4096, o_sh=128, o_sl=128)
assert lib.ssq_decode_workspace_size(ctypes.byref(a)) > 0
rc = lib.ssq_decode(ctypes.byref(a), None, 0, None)
assert rc != 0  # no GPU
assert b"workspace" not in lib.ssq_last_error(), lib.ssq_last_error()
print("runs without a workspace")
"""


# calls that one workgroup per pair serves as fast or faster: no workspace asked for
UNBALANCED = """
a.seq_len = 4095
assert lib.ssq_decode_workspace_size(ctypes.byref(a)) == 0
a.seq_len = 8192
a.batch, a.num_q_heads, a.num_kv_heads = 3, 129 * 4, 129  # one workgroup per KV head: half of the CUs
assert lib.ssq_decode_workspace_size(ctypes.byref(a)) == 0
a.batch, a.num_q_heads, a.num_kv_heads, a.head_dim, a.n_blocks, a.value_dim = 160, 14, 2, 64, 32, 64
assert lib.ssq_decode_workspace_size(ctypes.byref(a)) == 0
print("unbalanced")
"""


def test_calls_that_are_not_balanced():
    env = dict(os.environ, HIP_VISIBLE_DEVICES="-1", ROCR_VISIBLE_DEVICES="-1", CUDA_VISIBLE_DEVICES="-1")
    abi = os.path.join(HERE, "..", "sunshape_amd", "_abi.py")
    child = CHILD.split("rc = lib.ssq_decode(")[0] + UNBALANCED
    r = subprocess.run([sys.executable, "-c", child, N.LIB_PATH, abi], env=env, capture_output=True, text=True, timeout=300)
    assert "unbalanced" in r.stdout, (r.stdout[-500:], r.stderr[-2000:])


def test_balanced_batch_is_not_refused_without_a_workspace():
    env = dict(os.environ, HIP_VISIBLE_DEVICES="-1", ROCR_VISIBLE_DEVICES="-1", CUDA_VISIBLE_DEVICES="-1")
    abi = os.path.join(HERE, "..", "sunshape_amd", "_abi.py")
    r = subprocess.run([sys.executable, "-c", CHILD, N.LIB_PATH, abi], env=env, capture_output=True, text=True, timeout=300)
    assert "runs without a workspace" in r.stdout, (r.stdout[-500:], r.stderr[-2000:])


@pytest.mark.gpu
def test_noalloc_batch_runs_one_workgroup_per_pair():
    """Bit for bit the call with num_splits 1, which has one workgroup per (sequence, KV head) and no
    workspace.  Balanced, sequences cut between workgroups round their probabilities differently."""
    dev, g = "cuda", torch.Generator().manual_seed(1)
    lens = [5000] + torch.randint(1, 900, (47,), generator=g).tolist()
    perm = torch.randperm(128, generator=g).to(dev)
    cent = torch.randn(8, 64, 256, 2, generator=g).to(dev)
    pages = [(n + 15) // 16 for n in lens]
    pool = torch.randperm(sum(pages), generator=g).to(torch.int32)
    table = torch.zeros(48, max(pages), dtype=torch.int32)
    at = 0
    for b, n in enumerate(pages):
        table[b, :n] = pool[at:at + n]
        at += n
    gd = torch.Generator(device=dev).manual_seed(1)
    codes = torch.randint(0, 256, (at, 8, 16, 64), generator=gd, device=dev, dtype=torch.uint8)
    v = torch.randn(at, 8, 128, 16, generator=gd, device=dev, dtype=torch.bfloat16)
    q = torch.randn(48, 32, 1, 128, generator=gd, device=dev, dtype=torch.bfloat16)
    kw = dict(scale=1 / math.sqrt(128), block_table=table.to(dev),
              seq_lens=torch.tensor(lens, dtype=torch.int32, device=dev), return_lse=True)
    ref = hip_ops.decode(q, codes, v, perm, cent, num_splits=1, **kw)
    got = hip_ops.decode(q, codes, v, perm, cent, no_alloc=True, **kw)
    balanced = hip_ops.decode(q, codes, v, perm, cent, **kw)
    assert torch.equal(got[0], ref[0]) and torch.equal(got[1], ref[1])
    assert not torch.equal(balanced[0], ref[0])  # the batch is one that is balanced otherwise
