"""The split the kernels choose from a batch's lengths (kv_split = 0, up to
64 requests), against the oracle: the status word also shows a partial row
past the workspace, so every batch checks the sizing bounds."""
import math

import numpy as np
import pytest
import torch

from cast_amd import _lib
from cast_amd import scenarios as SC
from cast_amd.tree import TreeNode
from test_gpu_attn import _run_and_check, _words

pytestmark = pytest.mark.gpu


def _chain(n):
    return [TreeNode(i, i + 1, i - 1, 0.0) for i in range(n)]


def _batch(name, prefix, packs, Hq, Hkv, D, dtype="bf16"):
    return SC._make(name, [_chain(p - 1) for p in packs], prefix, dict(Hq=Hq, Hkv=Hkv, D=D, vocab=1000), dtype, 3,
                    1 / math.sqrt(D))


BATCHES = {
    # one long request among short ones; packs on both sides of a row block
    "long-among-short": ([9000] + [5, 64, 63, 130, 700], [33, 1, 32, 64, 31, 16], 16, 4, 128),
    # as many items as the device holds, exactly and one request more
    "items-fit": ([2048] * 8, [8] * 8, 32, 8, 128),
    "items-over": ([2048] * 8 + [2049], [8] * 9, 32, 8, 128),
    # the largest batch of the wave-wide schedule; many row blocks (one KV head)
    "batch-64": ([i * 17 % 900 for i in range(64)], [1 + i % 7 for i in range(64)], 8, 4, 64),
    "one-kv-head": ([6000, 300, 64], [128, 127, 2], 32, 1, 64),
    # averages that would not split, lengths that do
    "skewed": ([12000] + [40] * 39, [4] * 40, 32, 8, 128),
    "head-dim-256": ([3000, 65, 2000], [64, 1, 33], 8, 4, 256),
}


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("case", list(BATCHES))
def test_split_from_lengths(gpu, case, dtype):
    prefix, packs, Hq, Hkv, D = BATCHES[case]
    _run_and_check(_batch(case, prefix, packs, Hq, Hkv, D, dtype), gpu, label=f"split-from-lengths-{case}-{dtype}")


def test_missing_workspace_runs_unsplit(gpu):
    # calls whose averages ask for no split need no workspace: without one
    # they run as kv_split = -1 does, bit for bit, in both entry points
    prefix, packs, Hq, Hkv, D = BATCHES["skewed"]
    wl = _batch("no-workspace", prefix, packs, Hq, Hkv, D)
    print(f"case no-workspace: B={wl.B} total_q={wl.total_q} total_kv={wl.total_kv}", flush=True)
    lib = _lib.load()
    q, k, v = wl.qkv(device=gpu)
    meta = wl.meta_tensors(gpu)
    mask = torch.from_numpy(_words(wl).view(np.int64).copy()).to(gpu)
    outs = []
    for split, entry in ((-1, "ws"), (0, "ws"), (0, "noalloc")):
        out = torch.empty_like(q)
        lse = torch.empty(q.shape[:2], device=gpu)
        args = [_lib.ptr(q), _lib.ptr(k), _lib.ptr(v), _lib.ptr(out), _lib.ptr(lse), _lib.ptr(meta["cu_q"]),
                _lib.ptr(meta["cu_kv"]), _lib.ptr(meta["prefix_len"]), _lib.ptr(meta["pack_len"]), _lib.ptr(mask), 2,
                wl.B, wl.total_q, wl.total_kv, Hq, Hkv, D, q.stride(0), q.stride(1), k.stride(0), k.stride(1),
                v.stride(0), v.stride(1), out.stride(0), out.stride(1), _lib.BF16, float(D ** -0.5), split]
        with torch.cuda.device(gpu):
            if entry == "ws":
                st = lib.cast_tree_attn_fwd(*args, None, 0, None, _lib.stream_of(q))
            else:
                st = lib.cast_tree_attn_fwd_noalloc(*args, None, _lib.stream_of(q))
        assert st == 0, _lib.status_string(st)
        torch.cuda.synchronize()
        outs.append((out, lse))
    for out, lse in outs[1:]:
        assert torch.equal(out, outs[0][0]) and torch.equal(lse, outs[0][1])


def test_kv_split_from_a_tensor(gpu):
    # the workspace size is remembered by value, also where the caller keeps
    # kv_split in a tensor and changes it in place
    from cast_amd import varlen_tree_attention
    wl = _batch("split-tensor", [700, 300], [8, 5], 8, 4, 64)
    print("case split-tensor", flush=True)
    q, k, v = wl.qkv(device=gpu)
    meta = wl.meta_tensors(gpu)
    mask = torch.from_numpy(_words(wl).view(np.int64).copy()).to(gpu)
    args = (q, k, v, meta["cu_q"], meta["cu_kv"], meta["prefix_len"], meta["pack_len"], mask)
    split = torch.tensor(-1)
    assert torch.equal(varlen_tree_attention(*args, kv_split=split), varlen_tree_attention(*args, kv_split=-1))
    split.fill_(64)
    assert torch.equal(varlen_tree_attention(*args, kv_split=split), varlen_tree_attention(*args, kv_split=64))
    with pytest.raises(TypeError):
        varlen_tree_attention(*args, kv_split=0.5)
