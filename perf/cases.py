"""The calls whose speed this framework is about, as a program makes them.

A decode round drafts a token tree per request (draft), runs the target over
the packed trees with one tree-attention call per layer (attn, store), walks
the logits for the accepted path (accept) and appends the accepted K/V to the
store; "round" is a whole verify pass through the attention hook.

Lengths and pack sizes follow from the case alone ("mix" seeds them), all
values and tree shapes from prepare()'s seed.
"""
import heapq
import math

import numpy as np
import torch

from cast_amd import build_trees, greedy_accept, pack_trees, topk_marginals, tree_bitmask, varlen_tree_attention
from cast_amd import serving
from cast_amd.tree import TreeNode
from cast_amd.tree_attn import store_tree_attention

DEV = "cuda"
DRAFT_LEN = 15       # future positions the drafter scores
RANKS = 8            # candidates kept per position
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def _attn(name, kind, B, s_lo, s_hi, p_lo, p_hi, Hq, Hkv, D, dtype, lse=False, mix=0):
    c = dict(kind=kind, B=B, s_lo=s_lo, s_hi=s_hi, p_lo=p_lo, p_hi=p_hi, Hq=Hq, Hkv=Hkv, D=D, dtype=dtype, lse=lse,
             mix=mix)
    return dict(c, name=name) if name else c


def listed():
    return [
        # one request of a chat, a 16-token tree: the smallest call, two launches of a few microseconds each
        _attn("single-p16", "attn", 1, 2048, 2048, 16, 16, 32, 8, 128, "bf16"),
        # ordinary batch, ragged prefixes and packs of every size up to the largest
        _attn("ragged-b8", "attn", 8, 1024, 8192, 32, 128, 32, 8, 128, "bf16", lse=True, mix=3),
        # the benchmark's headline: full packs over long contexts
        _attn("long-b8-p128", "attn", 8, 8192, 8192, 128, 128, 32, 8, 128, "bf16"),
        # one request over a long document: few rows, many keys
        _attn("document-32k", "attn", 1, 32768, 32768, 128, 128, 32, 8, 128, "bf16"),
        # a server's batch at the widths a cost-aware policy picks: small odd packs, prefix read from the KV store
        _attn("serving-b32", "store", 32, 300, 4096, 2, 64, 32, 8, 128, "bf16", mix=5),
        # the largest: every request of a big batch at the full pack, from the KV store
        _attn("serving-b32-p128", "store", 32, 256, 4096, 128, 128, 32, 8, 128, "bf16", mix=7),
        # fp32 inputs, as an attention hook that up-casts its q, k and v hands them over (packs of one mask word)
        _attn("fp32-b8", "attn", 8, 1024, 4096, 2, 64, 32, 8, 128, "fp32", mix=11),
        # models with head dim 256
        _attn("d256-b8", "attn", 8, 4096, 8192, 64, 128, 16, 8, 256, "bf16", mix=13),
        # models whose head dim is no power of two
        _attn("d96-b4", "attn", 4, 500, 2000, 16, 64, 32, 8, 96, "fp16", mix=17),
        # accepted paths over a whole vocabulary's logits
        dict(name="accept-b8", kind="accept", B=8, p_lo=16, p_hi=128, V=151936, dtype="bf16", mix=19),
        # drafting for a batch: top-k of every future position, then the trees
        dict(name="draft-b8", kind="draft", B=8, L=DRAFT_LEN, V=151936, k=RANKS, N=127, dtype="bf16"),
        # a verify pass of a 36-layer model: packing, one hook call per layer, accept, KV append
        dict(name="round-b8", kind="round", B=8, s_lo=300, s_hi=2048, p_lo=8, p_hi=64, Hq=32, Hkv=8, D=128,
             dtype="bf16", layers=36, V=151936, mix=23),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _seconds(c):
    """A rough time of a case on the device, to bound drawn ones."""
    w = work(c)
    if "D" not in c:
        return w["bytes"] / 2e12
    rate = 6e14 if c["dtype"] != "fp32" else 8e13
    if c["D"] not in (64, 128, 256):
        rate = 2e12
    return w["bytes"] / 3e12 + w["flops"] / rate


def draw(rng):
    while True:
        kind = rng.choices(["attn", "store", "accept", "draft", "round"], [10, 5, 2, 2, 1])[0]
        mix = rng.randrange(1 << 20)
        if kind == "accept":
            P = _log_int(rng, 2, 128)
            return dict(kind=kind, B=_log_int(rng, 1, 8), p_lo=rng.randint(1, P), p_hi=P,
                        V=rng.choice([32000, 50257, 128256, 151936]),
                        dtype=rng.choice(["bf16", "bf16", "fp16", "fp32"]), mix=mix)
        if kind == "draft":
            return dict(kind=kind, B=_log_int(rng, 1, 32), L=rng.randint(4, 15),
                        V=rng.choice([32000, 50257, 128256, 151936]), k=rng.choice([4, 8, 8, 16]),
                        N=_log_int(rng, 8, 127), dtype=rng.choice(["bf16", "bf16", "fp16", "fp32"]))
        B = _log_int(rng, 1, 64) if kind != "round" else _log_int(rng, 1, 8)
        s_hi = _log_int(rng, 64, 32768) if kind != "round" else _log_int(rng, 64, 2048)
        p_hi = _log_int(rng, 2, 128) if kind != "round" else _log_int(rng, 2, 64)
        s_lo = rng.choice([s_hi, rng.randint(1, s_hi)])
        p_lo = rng.choice([p_hi, rng.randint(1, p_hi)])
        Hkv = rng.choice([8, 8, 8, 4, 2])
        Hq = Hkv * rng.choice([4, 4, 4, 8, 2, 1, 7])
        D = rng.choice([128] * 8 + [64] * 3 + [256] * 2 + [80, 96, 112, 192])
        dtype = rng.choice(["bf16"] * 5 + ["fp16"] * 2 + ["fp32"] * 2)
        if kind == "round":
            c = dict(kind=kind, B=B, s_lo=s_lo, s_hi=s_hi, p_lo=p_lo, p_hi=p_hi, Hq=Hq, Hkv=Hkv,
                     D=rng.choice([64, 128]), dtype="bf16", layers=rng.randint(16, 36),
                     V=rng.choice([32000, 128256, 151936]), mix=mix)
        else:
            c = _attn(None, kind, B, s_lo, s_hi, p_lo, p_hi, Hq, Hkv, D, dtype, rng.random() < 0.3, mix)
        if _seconds(c) < (1e-3 if kind == "round" else 3e-4 if D in (64, 128, 256) else 1.2e-3):
            return c


# ---- sizes

def _lengths(c):
    rng = np.random.default_rng(c["mix"])
    S = rng.integers(c["s_lo"], c["s_hi"] + 1, size=c["B"]) if "s_lo" in c else np.zeros(c["B"], np.int64)
    P = rng.integers(c["p_lo"], c["p_hi"] + 1, size=c["B"])
    return S.astype(np.int64), P.astype(np.int64)


def _esz(c):
    return 4 if c["dtype"] == "fp32" else 2


def work(c):
    if c["kind"] == "draft":
        n = c["B"] * c["L"] * c["V"]
        return {"bytes": n * _esz(c) + c["B"] * (c["L"] * c["k"] * 12 + c["N"] * 24), "flops": 2 * n}
    S, P = _lengths(c)
    if c["kind"] == "accept":
        n = int(P.sum()) * c["V"]
        return {"bytes": n * _esz(c) + int(P.sum()) * 16, "flops": n}
    kv = int((S + P).sum()) * c["Hkv"] * c["D"] * 2 * _esz(c)
    qo = int(P.sum()) * c["Hq"] * c["D"] * 2 * _esz(c)
    extra = int(P.sum()) * (16 + (4 * c["Hq"] if c.get("lse") else 0))
    w = {"bytes": kv + qo + extra, "flops": int((4 * P * (S + P)).sum()) * c["Hq"] * c["D"]}
    if c["kind"] == "round":
        n = int(P.sum()) * c["V"]
        w = {"bytes": w["bytes"] * c["layers"] + n * 2, "flops": w["flops"] * c["layers"] + n}
    return w


# ---- inputs

def _tree(rng, n, vocab):
    """A best-first tree of n nodes over drafter-like top-k log-probs."""
    gaps = rng.exponential(1.0, size=(DRAFT_LEN, RANKS))
    gaps[:, 0] *= 0.5
    lp = -np.cumsum(gaps, axis=1)
    tok = np.stack([rng.choice(vocab, RANKS, replace=False) if vocab < 4096 else rng.integers(0, vocab, RANKS)
                    for _ in range(DRAFT_LEN)])
    heap = [(-lp[0, r], 1, -1, r) for r in range(RANKS)]
    heapq.heapify(heap)
    nodes = []
    while heap and len(nodes) < n:
        neg, d, par, r = heapq.heappop(heap)
        nodes.append(TreeNode(int(tok[d - 1, r]), d, par, -neg))
        if d < DRAFT_LEN:
            for r2 in range(RANKS):
                heapq.heappush(heap, (neg - lp[d, r2], d + 1, len(nodes) - 1, r2))
    return nodes


def _packs(c, seed):
    S, P = _lengths(c)
    rng = np.random.default_rng([seed, c["mix"]])
    trees = [_tree(rng, int(p) - 1, c.get("V", 151936)) for p in P]
    roots = [int(x) for x in rng.integers(0, c.get("V", 151936), size=c["B"])]
    return S, P, trees, roots, pack_trees(trees, roots)


def _i32(a):
    return torch.as_tensor(np.ascontiguousarray(a, dtype=np.int32), device=DEV)


def _plant(logits, trees, cu_q, rng, accept_p=0.8):
    """Makes a root path of every tree the greedy choice of its rows."""
    rows, toks = [], []
    for b, nodes in enumerate(trees):
        cur = -1
        while True:
            kids = [i for i, nd in enumerate(nodes) if nd.parent == cur]
            if not kids or rng.random() > accept_p:
                break
            pick = kids[int(rng.integers(0, len(kids)))]
            rows.append(int(cu_q[b]) + cur + 1)
            toks.append(nodes[pick].token)
            cur = pick
    if rows:
        logits[torch.tensor(rows, device=DEV), torch.tensor(toks, device=DEV)] = 16.0


def prepare(c, seed):
    g = torch.Generator(DEV).manual_seed(seed)

    def randn(*shape, dtype=None):
        return torch.randn(*shape, generator=g, device=DEV, dtype=dtype or DTYPES[c["dtype"]])

    st = {"kind": c["kind"], "case": c}
    if c["kind"] == "draft":
        st.update(x=randn(c["B"] * c["L"], c["V"]).mul_(5.0), k=c["k"], shape=(c["B"], c["L"], c["k"]), N=c["N"])
        return st
    S, P, trees, roots, pk = _packs(c, seed)
    cu_q = _i32(pk.cu_q)
    parent = _i32(pk.parent)
    st.update(cu_q=cu_q, parent=parent, packed=pk, S=S, P=P)
    total_q = pk.total_q
    if c["kind"] in ("accept", "round"):
        logits = randn(total_q, c["V"])
        _plant(logits, trees, pk.cu_q, np.random.default_rng([seed, 1]))
        st.update(logits=logits, token=torch.from_numpy(pk.token).to(DEV))
        if c["kind"] == "accept":
            return st
    Hq, Hkv, D = c["Hq"], c["Hkv"], c["D"]
    if c["kind"] == "round":
        L, B = c["layers"], c["B"]
        cap = (int(S.max()) + 128 + 63) // 64 * 64
        store = randn(2, L, B, Hkv, cap, D)
        act = [[randn(1, total_q, h, D).transpose(1, 2) for h in (Hq, Hkv, Hkv)] for _ in range(L)]
        st.update(store=store, buf_k=[store[0, i] for i in range(L)], buf_v=[store[1, i] for i in range(L)], act=act,
                  trees=trees, roots=roots, store_len=[int(s) for s in S], scale=1 / math.sqrt(D))
        return st
    st.update(prefix=_i32(S), pack=_i32(P), words=tree_bitmask(parent, cu_q, 2), q=randn(total_q, Hq, D))
    if c["kind"] == "store":
        cap = (int(S.max()) + 128 + 63) // 64 * 64
        st.update(k=randn(c["B"], Hkv, cap, D), v=randn(c["B"], Hkv, cap, D),
                  kp=randn(total_q, Hkv, D).transpose(0, 1), vp=randn(total_q, Hkv, D).transpose(0, 1),
                  total_kv=int((S + P).sum()))
    else:
        cu_kv = np.concatenate([[0], np.cumsum(S + P)])
        st.update(k=randn(int(cu_kv[-1]), Hkv, D), v=randn(int(cu_kv[-1]), Hkv, D), cu_kv=_i32(cu_kv))
    return st


# ---- one pass

def run(st):
    c, kind = st["case"], st["kind"]
    if kind == "attn":
        return varlen_tree_attention(st["q"], st["k"], st["v"], st["cu_q"], st["cu_kv"], st["prefix"], st["pack"],
                                     st["words"], return_lse=c["lse"])
    if kind == "store":
        return store_tree_attention(st["q"], st["k"], st["v"], st["kp"], st["vp"], st["cu_q"], st["prefix"],
                                    st["pack"], st["words"], total_kv=st["total_kv"], return_lse=c["lse"])
    if kind == "accept":
        return greedy_accept(st["logits"], st["cu_q"], st["parent"], st["token"])
    if kind == "draft":
        idx, lp = topk_marginals(st["x"], st["k"], on_device=True)
        idx, lp, N = idx.view(st["shape"]), lp.view(st["shape"]), st["N"]
        token, depth, parent, score, n = build_trees(idx, lp, N)
        return idx, lp, token[:, :N], depth[:, :N], parent[:, :N], score[:, :N], n
    # a verify pass: the forward's attention calls, then accept and append
    ids, pos, _ = serving.begin_verify(st["buf_k"], st["buf_v"], st["store_len"], st["roots"], st["trees"],
                                       st["store_len"])
    plan = serving.PLAN
    outs = [serving._varlen_attention(None, q, k, v, None, scaling=st["scale"])[0] for q, k, v in st["act"]]
    path, plen, bonus, argmax = greedy_accept(st["logits"], plan.cu_q, plan.parent, ids[0])
    new_len = serving.append_accepted(st["buf_k"], st["buf_v"], plan.prefix_len, plan.cu_q, path, plen)
    plan.clear()
    return outs, path, plen, bonus, argmax, new_len, st["store"]


# ---- the same in 64 bits

def _visible(parent):
    n = len(parent)
    vis = np.zeros((n, n), dtype=bool)
    for i, p in enumerate(parent):
        if p >= 0:
            vis[i] = vis[p]
        vis[i, i] = True
    return torch.from_numpy(vis).to(DEV)


def _dense(q, k, v, vis):
    """q [P, Hq, D], k / v [Hkv, T, D] (prefix, then the pack) -> out, lse in float64."""
    P, Hq, D = q.shape
    Hkv, T, _ = k.shape
    G = Hq // Hkv
    qf = q.double().reshape(P, Hkv, G, D).permute(1, 0, 2, 3).reshape(Hkv, P * G, D)
    s = torch.matmul(qf, k.double().transpose(1, 2).contiguous()) / math.sqrt(D)
    s = s.view(Hkv, P, G, T)
    s[..., T - P:].masked_fill_(~vis[None, :, None, :], -math.inf)
    lse = torch.logsumexp(s, dim=-1)
    o = torch.matmul(torch.exp(s - lse[..., None]).view(Hkv, P * G, T), v.double().contiguous())
    return (o.view(Hkv, P, G, D).permute(1, 0, 2, 3).reshape(P, Hq, D),
            lse.permute(1, 0, 2).reshape(P, Hq))


def _first_max(x):
    m = x.max(dim=1, keepdim=True).values
    at = torch.arange(x.shape[1], device=x.device, dtype=torch.int32)
    return torch.where(x == m, at, x.shape[1]).min(dim=1).values


def _walk(st, argmax):
    pk, am = st["packed"], argmax.cpu().numpy()
    B = pk.batch
    path, plen, bonus = np.full((B, 128), -1, np.int32), np.zeros(B, np.int32), np.zeros(B, np.int64)
    for b in range(B):
        lo, n = int(pk.cu_q[b]), int(pk.pack_len[b])
        cur = 0
        while True:
            t = int(am[lo + cur])
            kid = next((j for j in range(1, n) if pk.parent[lo + j] == cur and pk.token[lo + j] == t), None)
            if kid is None:
                break
            path[b, plen[b]] = kid - 1
            plen[b] += 1
            cur = kid
        bonus[b] = t
    return tuple(torch.from_numpy(x).to(DEV) for x in (path, plen, bonus))


def exact(c, seed):
    st = prepare(c, seed)
    if c["kind"] == "draft":
        x = st["x"].double()
        val, idx = torch.sort(x, dim=1, descending=True, stable=True)
        lp = (val[:, :c["k"]] - torch.logsumexp(x, dim=1, keepdim=True)).view(st["shape"])
        return idx[:, :c["k"]].reshape(st["shape"]), lp, *_heap(idx[:, :c["k"]], lp, c)
    argmax = _first_max(st["logits"]) if "logits" in st else None
    if c["kind"] == "accept":
        return (*_walk(st, argmax), argmax)
    S, P, pk = st["S"], st["P"], st["packed"]
    cq = [int(x) for x in pk.cu_q]
    vis = [_visible(pk.parent[a:b]) for a, b in zip(cq, cq[1:])]

    def layer(q, keys):
        got = [_dense(q[cq[b]:cq[b + 1]], *keys(b), vis[b]) for b in range(c["B"])]
        return torch.cat([o for o, _ in got]), torch.cat([s for _, s in got])

    if c["kind"] == "attn":
        ck = np.concatenate([[0], np.cumsum(S + P)])
        o, lse = layer(st["q"], lambda b: [x[ck[b]:ck[b + 1]].transpose(0, 1) for x in (st["k"], st["v"])])
        return (o, lse) if c["lse"] else o

    def stored(buf_k, buf_v, kp, vp):
        return lambda b: [torch.cat([x[b, :, :S[b]], y[:, cq[b]:cq[b + 1]]], dim=1)
                          for x, y in ((buf_k, kp), (buf_v, vp))]

    if c["kind"] == "store":
        o, lse = layer(st["q"], stored(st["k"], st["v"], st["kp"], st["vp"]))
        return (o, lse) if c["lse"] else o
    outs = [layer(q[0].transpose(0, 1), stored(bk, bv, k[0], v[0]))[0][None]
            for (q, k, v), bk, bv in zip(st["act"], st["buf_k"], st["buf_v"])]
    path, plen, bonus = _walk(st, argmax)
    for b in range(c["B"]):
        keep = torch.cat([torch.zeros(1, device=DEV, dtype=torch.int64), path[b, :int(plen[b])].long() + 1]) + cq[b]
        for (_, k, v), bk, bv in zip(st["act"], st["buf_k"], st["buf_v"]):
            bk[b, :, S[b]:S[b] + len(keep)] = k[0][:, keep]
            bv[b, :, S[b]:S[b] + len(keep)] = v[0][:, keep]
    return outs, path, plen, bonus, argmax, torch.as_tensor(S, device=DEV) + plen + 1, st["store"]


def _heap(idx, lp, c):
    """Best-first trees over the log-probs as the drafter returns them (32 bits), scores in 64."""
    idx, lp = idx.view(c["B"], c["L"], c["k"]).cpu().numpy(), lp.float().double().cpu().numpy()
    B, N = c["B"], c["N"]
    token, depth, parent = (np.zeros((B, N), t) for t in (np.int64, np.int32, np.int32))
    score = np.zeros((B, N))
    for b in range(B):
        heap = [(-lp[b, 0, r], 1, -1, r) for r in range(c["k"])]
        heapq.heapify(heap)
        for n in range(N):
            neg, d, par, r = heapq.heappop(heap)
            token[b, n], depth[b, n], parent[b, n], score[b, n] = idx[b, d - 1, r], d, par, -neg
            if d < c["L"]:
                for r2 in range(c["k"]):
                    heapq.heappush(heap, (neg - lp[b, d, r2], d + 1, n, r2))
    return (*(torch.from_numpy(x).to(DEV) for x in (token, depth, parent, score)),
            torch.full((B,), N, device=DEV, dtype=torch.int32))


def tolerance(c):
    if c["kind"] == "accept":
        return "exact"
    if c["kind"] == "draft":
        # 32-bit log-probs; where two paths' sums differ by rounding alone, their order follows the rounding:
        # summing a row's exponentials in another order moved 2 to 15 % of the nodes
        return {"rel": 1e-5, "differ": 0.4}
    if c["dtype"] == "fp32":
        return {"rel": 1e-5}
    return {"rel": 1e-2 if c["dtype"] == "bf16" else 2e-3}
