"""Head dims without an instance of their own (multiples of 8 up to 256) on
the padded MFMA kernels: against float64, against the scalar kernel (which
takes what the padded kernels cannot: here an output that is not 16-byte
aligned), and rows that hold infinities."""
import math

import numpy as np
import pytest
import torch

from cast_amd import scenarios as SC
from cast_amd import varlen_tree_attention
from cast_amd.tree import TreeNode
from cast_amd.tree_attn import store_tree_attention
from oracle import bitmask as OB

pytestmark = pytest.mark.gpu

# the spacing just above 1 (8, 11 and 24 significant bits): rounding is within half of it, relatively
EPS = {"bf16": 2.0 ** -7, "fp16": 2.0 ** -10, "fp32": 2.0 ** -23}


def _case(gpu, D, dtype, seed, prefix, packs, Hq=8, Hkv=2):
    rng = np.random.default_rng(seed)
    trees = [[TreeNode(i, 1, int(rng.integers(-1, i)) if i else -1, 0.0) for i in range(p - 1)] for p in packs]
    wl = SC._make(f"d{D}", trees, prefix, dict(Hq=Hq, Hkv=Hkv, D=D, vocab=100), dtype, seed, 0.5)
    q, k, v = wl.qkv(device=gpu)
    words = OB.chain_walk_words(wl.packed.parent, wl.cu_q)
    return wl, q, k, v, wl.meta_tensors(gpu), torch.from_numpy(words.view(np.int64).copy()).to(gpu), words


def _exact(wl, q, k, v, words):
    """out, lse in float64 (the visibility bits unpacked to a dense mask)."""
    G = wl.Hq // wl.Hkv
    out = torch.zeros(q.shape, dtype=torch.float64)
    lse = torch.zeros(q.shape[:2], dtype=torch.float64)
    q, k, v = (x.double().cpu() for x in (q, k, v))
    for b in range(wl.B):
        r0, r1, S = int(wl.cu_q[b]), int(wl.cu_q[b + 1]), int(wl.prefix_len[b])
        kb, vb = (x[int(wl.cu_kv[b]):int(wl.cu_kv[b + 1])].repeat_interleave(G, dim=1) for x in (k, v))
        bits = np.unpackbits(words[r0:r1].view(np.uint8), axis=1, bitorder="little")[:, :r1 - r0].astype(bool)
        vis = torch.cat([torch.ones(r1 - r0, S, dtype=torch.bool), torch.from_numpy(bits)], dim=1)
        s = torch.matmul(q[r0:r1].transpose(0, 1), kb.permute(1, 2, 0).contiguous()) / math.sqrt(wl.D)
        s = s.masked_fill(~vis[None], -math.inf)
        lse[r0:r1] = torch.logsumexp(s, -1).T
        out[r0:r1] = torch.matmul(torch.softmax(s, -1), vb.transpose(0, 1).contiguous()).transpose(0, 1)
    return out, lse


@pytest.mark.parametrize("dtype", ["bf16", "fp16", "fp32"])
@pytest.mark.parametrize("D", [8, 56, 72, 80, 96, 104, 120, 136, 192, 200, 248])
def test_padded_head_dims(gpu, D, dtype):
    # 700 keys split by the automatic choice; packs around the 32-row block
    wl, q, k, v, meta, mask, words = _case(gpu, D, dtype, D, [700, 0, 65], [64, 9, 33])
    print(f"case padded D={D} {dtype}", flush=True)
    want, want_l = _exact(wl, q, k, v, words)
    for split in (0, -1):
        out, lse = varlen_tree_attention(q, k, v, meta["cu_q"], meta["cu_kv"], meta["prefix_len"], meta["pack_len"],
                                         mask, return_lse=True, kv_split=split, check=True)
        # P and every sum are fp32: what is left is the output's own rounding
        # (EPS / 2), twice where a split's fp32 partial rounds first, and fp32
        # sums of up to 764 terms (2^-24 * sqrt(764) * 8 < 2e-5 of the rows' scale)
        err = (out.double().cpu() - want).abs()
        assert (err <= 0.51 * EPS[dtype] * want.abs() + 2e-5).all(), f"{err.max()}"
        assert ((lse.double().cpu() - want_l).abs() <= 2e-5).all()


@pytest.mark.parametrize("D", [80, 192])
def test_padded_store_layout_and_scalar_fallback(gpu, D):
    wl, q, k, v, meta, mask, _ = _case(gpu, D, "bf16", 1, [300, 129], [20, 64])
    print(f"case padded-store D={D}", flush=True)
    cap = 320
    ks = torch.zeros((wl.B, wl.Hkv, cap, D), dtype=q.dtype, device=gpu)
    vs, kp = torch.zeros_like(ks), torch.empty((wl.Hkv, wl.total_q, D), dtype=q.dtype, device=gpu)
    vp = torch.empty_like(kp)
    for b in range(wl.B):
        a, S, e = int(wl.cu_kv[b]), int(wl.prefix_len[b]), int(wl.cu_kv[b + 1])
        r = slice(int(wl.cu_q[b]), int(wl.cu_q[b + 1]))
        for src, st, pk in ((k, ks, kp), (v, vs, vp)):
            st[b, :, :S] = src[a:a + S].transpose(0, 1)
            pk[:, r] = src[a + S:e].transpose(0, 1)
    args = (meta["cu_q"], meta["cu_kv"], meta["prefix_len"], meta["pack_len"], mask)
    o1, l1 = varlen_tree_attention(q, k, v, *args, return_lse=True, check=True)
    o2, l2 = store_tree_attention(q, ks, vs, kp, vp, meta["cu_q"], meta["prefix_len"], meta["pack_len"], mask,
                                  total_kv=wl.total_kv, return_lse=True, check=True)
    assert torch.equal(o1, o2) and torch.equal(l1, l2)
    # an output 8 bytes off: the scalar kernel, as before; both are the fp32
    # result rounded once, so at most a rounding apart
    buf = torch.empty(q.numel() + 4, dtype=q.dtype, device=gpu)
    o3, l3 = varlen_tree_attention(q, k, v, *args, return_lse=True, check=True, out=buf[4:].view(q.shape))
    assert ((o3.float() - o1.float()).abs() <= EPS["bf16"] * o1.float().abs() + 2e-5).all()
    assert ((l3 - l1).abs() <= 2e-5).all()


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("what", ["v-inf", "k-minus-inf", "k-nan", "q-inf", "score-overflow"])
def test_padded_rows_with_infinities(gpu, dtype, what):
    # rows whose products meet an infinity or a NaN come out as the scalar
    # kernel gives them; all others keep their bits
    wl, q, k, v, meta, mask, _ = _case(gpu, 96, dtype, 2, [200, 90], [10, 40])
    print(f"case padded-nonfinite {what} {dtype}", flush=True)
    args = (meta["cu_q"], meta["cu_kv"], meta["prefix_len"], meta["pack_len"], mask)
    clean = varlen_tree_attention(q, k, v, *args)
    q, k, v = q.clone(), k.clone(), v.clone()
    if what == "v-inf":
        v[5, 0, 17] = math.inf
    elif what == "k-minus-inf":
        k[70, 1, 3] = -math.inf
    elif what == "k-nan":
        k[12, 0, 95] = math.nan
    elif what == "q-inf":
        q[3, 2, 40] = math.inf
    else:
        q[4] *= 1e4
        k[:200, 0] *= 1e4
    got, lse = varlen_tree_attention(q, k, v, *args, return_lse=True, check=True)
    buf = torch.empty(q.numel() + 4, dtype=q.dtype, device=gpu)
    ref, ref_l = varlen_tree_attention(q, k, v, *args, return_lse=True, out=buf[4:].view(q.shape))
    assert torch.equal(torch.isnan(got), torch.isnan(ref)) and torch.equal(torch.isnan(lse), torch.isnan(ref_l))
    fin = torch.isfinite(ref)
    assert torch.equal(got[~fin & ~torch.isnan(ref)], ref[~fin & ~torch.isnan(ref)])
    if what != "score-overflow":
        assert not fin.all()
        assert ((got.float() - ref.float()).abs()[fin] <= EPS[dtype] * ref.float().abs()[fin] + 2e-5).all()
        assert torch.equal(got[10:], clean[10:]) or what == "k-minus-inf"


@pytest.mark.parametrize("what", ["v-inf", "k-minus-inf", "k-nan", "q-inf", "huge", "scaled"])
@pytest.mark.parametrize("D,packs", [(128, [10, 40]), (128, [120, 90]), (64, [10, 40]), (256, [10, 40])])
def test_fp32_terms_keep_floats(gpu, D, packs, what):
    # fp32 operands enter the products as three bf16 terms: infinities, NaN
    # and floats next to the largest (whose leading term rounds to infinity)
    # give what float products give, and powers of two pass through exactly
    wl, q, k, v, meta, mask, words = _case(gpu, D, "fp32", 2, [200, 90], packs)
    print(f"case fp32-terms D={D} packs={packs} {what}", flush=True)
    args = (meta["cu_q"], meta["cu_kv"], meta["prefix_len"], meta["pack_len"], mask)
    clean = varlen_tree_attention(q, k, v, *args, kv_split=-1)
    q, k, v = q.clone(), k.clone(), v.clone()
    if what == "v-inf":
        v[5, 0, 17] = math.inf
    elif what == "k-minus-inf":
        k[70, 1, 3] = -math.inf
    elif what == "k-nan":
        k[12, 0, D - 1] = math.nan
    elif what == "q-inf":
        q[3, 2, 40] = math.inf
    elif what == "huge":
        v[7, 1, 5] = 3.4e38      # rounds to infinity in bf16
    else:
        v *= 2.0 ** -90
    out, lse = varlen_tree_attention(q, k, v, *args, return_lse=True, kv_split=-1, check=True)
    if what == "scaled":
        assert torch.equal(out, clean * 2.0 ** -90)
        return
    assert torch.equal(out[packs[0]:], clean[packs[0]:])       # request 1 is untouched
    want, want_l = _exact(wl, q, k, v, words)
    hot = {"v-inf": (slice(None), slice(0, 4)), "k-minus-inf": (slice(None), slice(4, 8)),
           "k-nan": (slice(None), slice(0, 4)), "q-inf": (slice(3, 4), slice(2, 3)),
           "huge": (slice(None), slice(4, 8))}[what]
    rows = torch.zeros(out.shape[:2], dtype=torch.bool)
    rows[:packs[0]][hot] = True
    got = out.cpu()
    assert torch.equal(got[~rows], clean.cpu()[~rows])
    if what == "v-inf":
        assert torch.isposinf(got[:packs[0], :4, 17]).all()
        keep = [d for d in range(D) if d != 17]
        assert torch.isfinite(got[:packs[0], :4, keep]).all()
    elif what in ("k-nan", "q-inf"):
        assert torch.isnan(got[rows]).any(dim=-1).all()
    elif what == "huge":
        assert ((got.double() - want).abs()[rows] <= 2e-5 * want.abs()[rows].clamp(min=1.0)).all()
    else:                        # a score of -inf (q > 0) is a key that is not there; one of +inf makes NaN
        assert torch.equal(torch.isnan(got), torch.isnan(want))
        fin = rows[..., None] & torch.isfinite(want)
        assert fin.any() and ((got.double() - want).abs()[fin] <= 2e-5).all()


@pytest.mark.parametrize("layout", ["concat", "store"])
@pytest.mark.parametrize("split", [-1, 0, 128])
@pytest.mark.parametrize("D,dtype", [(64, "fp32"), (128, "fp32"), (256, "fp32"), (40, "fp32"), (200, "fp32"), (8, "bf16"),
                                     (96, "fp16"), (120, "bf16"), (192, "fp16"), (248, "bf16")])
def test_rows_again_with_float_products(gpu, D, dtype, split, layout):
    # one infinity in every (request, head)'s values, in the prefix or the
    # pack: every row that sees it is computed again, and its other elements
    # have to match float64 as if nothing had happened
    wl, q, k, v, meta, mask, words = _case(gpu, D, dtype, 5, [333, 0, 64], [64, 41, 5])
    print(f"case rows-again D={D} {dtype} split={split} {layout}", flush=True)
    for b in range(wl.B):
        for h in range(wl.Hkv):
            # an inner prefix key, or the pack's root, which every row sees
            key = 100 if h and wl.prefix_len[b] > 100 else int(wl.prefix_len[b])
            v[int(wl.cu_kv[b]) + key, h, 3] = math.inf
    if layout == "concat":
        out, lse = varlen_tree_attention(q, k, v, meta["cu_q"], meta["cu_kv"], meta["prefix_len"], meta["pack_len"],
                                         mask, return_lse=True, kv_split=split, check=True)
    else:
        ks = torch.zeros((wl.B, wl.Hkv, 384, D), dtype=q.dtype, device=gpu)
        vs, kp = torch.zeros_like(ks), torch.empty((wl.Hkv, wl.total_q, D), dtype=q.dtype, device=gpu)
        vp = torch.empty_like(kp)
        for b in range(wl.B):
            a, S, e = int(wl.cu_kv[b]), int(wl.prefix_len[b]), int(wl.cu_kv[b + 1])
            r = slice(int(wl.cu_q[b]), int(wl.cu_q[b + 1]))
            for src, st, pk in ((k, ks, kp), (v, vs, vp)):
                st[b, :, :S] = src[a:a + S].transpose(0, 1)
                pk[:, r] = src[a + S:e].transpose(0, 1)
        out, lse = store_tree_attention(q, ks, vs, kp, vp, meta["cu_q"], meta["prefix_len"], meta["pack_len"], mask,
                                        total_kv=wl.total_kv, return_lse=True, kv_split=split, check=True)
    want, want_l = _exact(wl, q, k, v.masked_fill(torch.isinf(v), 0.0), words)
    got = out.double().cpu()
    assert torch.isposinf(got[:, :, 3]).all()
    keep = [d for d in range(D) if d != 3]
    err = (got - want).abs()[..., keep]
    assert (err <= 0.51 * EPS[dtype] * want.abs()[..., keep] + 2e-5).all(), f"{err.max()}"
    assert ((lse.double().cpu() - want_l).abs() <= 2e-5).all()


@pytest.mark.parametrize("D,dtype", [(128, "fp32"), (96, "fp16")])
def test_one_nan_costs_little(gpu, D, dtype):
    # rows that meet a NaN go through float products 32 at a time: measured 2
    # to 4 times the clean call (row by row it was 30 to 200 times)
    wl, q, k, v, meta, mask, _ = _case(gpu, D, dtype, 6, [4000] * 4, [64] * 4, Hq=32, Hkv=8)
    print(f"case nan-cost D={D} {dtype}", flush=True)

    def best():
        times = []
        for _ in range(6):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            varlen_tree_attention(q, k, v, meta["cu_q"], meta["cu_kv"], meta["prefix_len"], meta["pack_len"], mask)
            b.record()
            b.synchronize()
            times.append(a.elapsed_time(b))
        return min(times)

    clean = best()
    v[5, 0, 7] = math.nan
    assert best() < 12 * clean


@pytest.mark.parametrize("n", [40, 900])
@pytest.mark.parametrize("D", [64, 96, 128, 256])
def test_fp32_products_left_out_are_unbiased(gpu, D, n):
    # values just above 1 whose second and third terms are the largest there
    # are, the same for every key: the output is the value, whatever the
    # weights, and what is left out of the products would push all outputs to
    # one side if the weights' terms had one sign
    wl, q, k, v, meta, mask, words = _case(gpu, D, "fp32", 7, [n] * 8, [16] * 8)
    print(f"case fp32-unbiased D={D} keys={n}", flush=True)
    g = torch.Generator(gpu).manual_seed(D)
    step = torch.randint(0, 30, (1, 1, D), generator=g, device=gpu)
    v.copy_((1 + 2.0 ** -8 - 2.0 ** -17 + 2.0 ** -23 * step).expand_as(v))
    out = varlen_tree_attention(q, k, v, meta["cu_q"], meta["cu_kv"], meta["prefix_len"], meta["pack_len"], mask,
                                check=True).double()
    err = out / v[:1, :1].double() - 1
    # 2^-24 a rounding: up to 16 in a lane's sum of weights and as many over
    # tiles, the inverse, the result, 2^-24 left out; singly rounded values
    # give an rms of 0.29 * 2^-23, a dozen of them 2^-23
    assert err.abs().max() <= 2.0 ** -19 and err.pow(2).mean().sqrt() <= 2.0 ** -23
    # of unknown sign, over 16384 outputs and more they cancel to below 2^-27
    # (weights cut instead of rounded: -2^-26.2 to -2^-25.6)
    assert err.mean().abs() <= 2.0 ** -27


@pytest.mark.parametrize("what", ["v", "q", "k"])
@pytest.mark.parametrize("e", [-108, -112, -118, -124])
@pytest.mark.parametrize("D", [64, 96, 128, 256])
def test_fp32_small_magnitudes(gpu, D, e, what):
    # below 2^-110 the third bf16 term of a float is under bf16's smallest
    # step; the products have to keep what float products keep
    wl, q, k, v, meta, mask, words = _case(gpu, D, "fp32", 8, [300, 0, 40], [8, 5, 20])
    print(f"case fp32-small D={D} 2^{e} {what}", flush=True)
    two = 2.0 ** e
    if what == "v":
        v *= two
    elif what == "q":
        q, k = q * two, k / two
    else:
        q, k = q / two, k * two
    out, lse = varlen_tree_attention(q, k, v, meta["cu_q"], meta["cu_kv"], meta["prefix_len"], meta["pack_len"], mask,
                                     return_lse=True, check=True)
    want, want_l = _exact(wl, q, k, v, words)
    got = out.double().cpu()
    # fp32 sums of up to 308 weights and products: 2^-24 * sqrt(308) * 4 < 5e-6,
    # and results below the smallest normal float on its grid of 2^-149
    assert (got - want).norm() <= 5e-6 * want.norm() + 2.0 ** -149 * want.numel() ** 0.5
    assert ((lse.double().cpu() - want_l).abs() <= 2e-5).all()


@pytest.mark.parametrize("nats", [40, 80, 84, 86])
def test_fp32_small_weights(gpu, nats):
    # a key of value zero holds all the weight but that of one far below it,
    # which alone makes the output: its weight has to be a float's
    wl, q, k, v, meta, mask, words = _case(gpu, 128, "fp32", 9, [300], [8])
    print(f"case fp32-small-weight {nats} nats", flush=True)
    q.zero_()[..., 0] = 1.0
    k.zero_()[..., 0] = -4000.0
    k[0, :, 0], k[1, :, 0] = 0.0, -nats * math.sqrt(128)
    v[0] = v[2:] = 0.0
    out = varlen_tree_attention(q, k, v, meta["cu_q"], meta["cu_kv"], meta["prefix_len"], meta["pack_len"], mask,
                                check=True)
    want, _ = _exact(wl, q, k, v, words)
    # the score in base 2, up to 124, is rounded to 2^-18: 2.6e-6 of the weight, twice
    assert ((out.double().cpu() - want).abs() <= 1e-5 * want.abs()).all()


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("D", [40, 96, 120, 192, 248])
@pytest.mark.parametrize("nats", [5.3, 10.1, 14.2, 16.7, 19.3])
def test_padded_small_weights(gpu, nats, D, dtype):
    # a key of value zero holds nearly all the weight; the others, alike and
    # far below it, make the output: their weights have to be held as floats
    wl, q, k, v, meta, mask, words = _case(gpu, D, dtype, 10, [400, 90], [16, 33])
    print(f"case padded-small-weights D={D} {dtype} {nats} nats", flush=True)
    q.zero_()[..., 0] = 1.0
    q[..., 1] = 1.0
    k.zero_()[..., 0] = -nats * math.sqrt(D)
    k[..., 1] = -nats * math.sqrt(D) - k[..., 0].float()       # what the format's rounding left
    for b in range(wl.B):
        first = int(wl.cu_kv[b])
        k[first] = 0.0
        v[first] = 0.0
    v.mul_(100.0)
    out = varlen_tree_attention(q, k, v, meta["cu_q"], meta["cu_kv"], meta["prefix_len"], meta["pack_len"], mask,
                                kv_split=-1, check=True)
    want, _ = _exact(wl, q, k, v, words)
    # the output's own rounding (half a step, 2^-25 at least in fp16), and of
    # the values' sum 2^-21 for the scores' and weights' roundings in fp32
    span = 100 * 4 * 433 * math.exp(-nats) * 2.0 ** -21
    assert ((out.double().cpu() - want).abs() <= 0.51 * EPS[dtype] * want.abs() + 2.0 ** -25 + span).all()
