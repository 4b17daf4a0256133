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
from cast_amd.tree_attn import plan
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
    # as many items as the device holds (512 of 4 waves), exactly and a few more
    "items-fit": ([4088] * 8, [8] * 8, 32, 8, 128),
    "items-over": ([4088] * 8 + [56], [8] * 9, 32, 8, 128),
    # the largest batch of the wave-wide schedule; averages that ask for no split
    "batch-64": ([i * 37 % 1900 for i in range(64)], [1 + i % 7 for i in range(64)], 8, 4, 64),
    # many row blocks (one KV head)
    "one-kv-head": ([6000, 300, 64], [128, 127, 2], 32, 1, 64),
    # averages that would not split, lengths that do
    "skewed": ([12000] + [400] * 39, [4] * 40, 32, 8, 128),
    "head-dim-256": ([3000, 65, 2000], [64, 1, 33], 8, 4, 256),
}


def _slots(packs, Hq, Hkv, D):
    """Query rows of a workgroup and the workgroups the device holds at once
    (256 CUs; per CU two of 4 waves at D = 128, three at 64, else one)."""
    G = Hq // Hkv
    most = 192 if D == 64 else 144 if sum(packs) % len(packs) else 128
    four = D == 256 or -(-sum(packs) // len(packs)) * G <= most
    return (128, 256 * {256: 1, 128: 2, 64: 3}[D]) if four else (256, 256)


def _choice(prefix, packs, Hq, Hkv, D):
    """The split of a 16-bit batch from its lengths: the candidate taken (None:
    no candidate's items fit the slots, "whole": no split) and its tiles of 64
    keys."""
    rows_wg, slots = _slots(packs, Hq, Hkv, D)
    tiles = [-(-(s + p) // 64) if p else 0 for s, p in zip(prefix, packs)]
    rb = [-(-p * (Hq // Hkv) // rows_wg) for p in packs]
    total = Hkv * sum(t * r for t, r in zip(tiles, rb))
    B, G = len(packs), Hq // Hkv
    t_avg, rows_avg = -(-(sum(prefix) + sum(packs)) // B), min(-(-sum(packs) // B), 128) * G
    p = plan(B, sum(packs), sum(prefix) + sum(packs), Hq, Hkv, D)
    if p.kv_split == -1 and D == 128 and max(tiles) * sum(rb) * Hkv <= (0.9 + 4 * rows_avg / t_avg) * total:
        return "whole", max(tiles)
    start = max(-(-total // slots), 1, 8 if total >= 8 * 192 else max(total // 192, 2))
    sizes = [(start * w + 7) // 8 for w in (8, 9, 10, 12)]
    fits = [Hkv * sum(r * -(-t // c) for t, r in zip(tiles, rb)) <= slots for c in sizes]
    taken = fits.index(True) if any(fits) else None
    return taken, sizes[2 if taken is None else taken]


def _run(wl, gpu, kv_split, ws=None):
    from cast_amd import varlen_tree_attention
    q, k, v = wl.qkv(device=gpu)
    meta = wl.meta_tensors(gpu)
    mask = torch.from_numpy(_words(wl).view(np.int64).copy()).to(gpu)
    return varlen_tree_attention(q, k, v, meta["cu_q"], meta["cu_kv"], meta["prefix_len"], meta["pack_len"], mask,
                                 return_lse=True, kv_split=kv_split, check=True, workspace=ws)


def _one_long(first, rest, n, pack, Hq, Hkv, D):
    return [first] + [rest] * n, [pack] * (n + 1), Hq, Hkv, D


# candidate (None: none fits) -> one long request and n alike; 3 and 5 KV heads
# are no multiple of the 8 XCDs
CHOICES = [
    (0, _one_long(1000, 60, 9, 8, 32, 8, 128)), (1, _one_long(9000, 700, 24, 8, 32, 8, 128)),
    (2, _one_long(5000, 700, 28, 8, 32, 8, 128)), (3, _one_long(1000, 700, 32, 8, 32, 8, 128)),
    (None, _one_long(1200, 800, 32, 8, 32, 8, 128)), ("whole", _one_long(1000, 900, 32, 24, 32, 8, 128)),
    ("whole", _one_long(700, 700, 31, 16, 32, 8, 128)),
    (0, _one_long(1000, 10, 9, 100, 20, 5, 128)), (1, _one_long(1000, 60, 9, 100, 20, 5, 128)),
    (2, _one_long(2000, 100, 20, 100, 20, 5, 128)), (3, _one_long(2000, 10, 17, 100, 20, 5, 128)),
    (None, _one_long(2000, 10, 19, 100, 20, 5, 128)),
    (0, _one_long(1000, 10, 23, 120, 12, 3, 64)), (1, _one_long(1000, 10, 17, 120, 12, 3, 64)),
    (2, _one_long(5000, 10, 29, 120, 12, 3, 64)), (3, _one_long(3000, 10, 33, 120, 12, 3, 64)),
    (None, _one_long(3000, 10, 34, 120, 12, 3, 64)),
    (0, _one_long(1000, 10, 7, 16, 16, 8, 256)), (1, _one_long(2000, 10, 17, 16, 16, 8, 256)),
    (2, _one_long(2000, 200, 27, 16, 16, 8, 256)), (3, _one_long(3000, 10, 21, 16, 16, 8, 256)),
    (None, _one_long(3000, 10, 23, 16, 16, 8, 256)),
    (0, BATCHES["items-fit"]), (1, BATCHES["items-over"]),
]


@pytest.mark.parametrize("i", range(len(CHOICES)))
def test_every_candidate(gpu, i):
    # the kernels' choice is the one the lengths ask for, and every item of it
    # is worked off: bit for bit the forced chunk of that size
    want, batch = CHOICES[i]
    taken, tiles = _choice(*batch)
    assert taken == want
    wl = _batch(f"choice-{i}", *batch)
    print(f"case choice {i}: candidate {want}, {tiles} tiles, B={wl.B} D={wl.D} Hkv={wl.Hkv}", flush=True)
    n = plan(wl.B, wl.total_q, wl.total_kv, wl.Hq, wl.Hkv, wl.D).workspace_bytes
    ws = torch.zeros(n, dtype=torch.uint8, device=gpu)
    out, lse = _run(wl, gpu, 0, ws)
    # the first workgroup leaves the choice in the last 256 bytes
    assert int(ws[n - 256:n - 252].view(torch.int32)[0]) == tiles
    forced = _run(wl, gpu, 64 * tiles)
    assert torch.equal(out, forced[0]) and torch.equal(lse, forced[1])


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
    # with one they split: the averages ask for none, the lengths do
    p = plan(wl.B, wl.total_q, wl.total_kv, Hq, Hkv, D)
    assert p.kv_split == -1 and p.workspace_bytes > 0
    cut = _run(wl, gpu, 0)
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
    assert not torch.equal(cut[0], outs[0][0]) and (cut[0].float() - outs[0][0].float()).abs().max() <= 2e-2


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
