"""Performance cases of the framework: calls of its public operators over the
sizes, data types and options they are used with.

``listed()`` gives the named cases, ``draw(rng)`` one more of the same ranges.
A case is a dict of plain values; ``kind`` names the entry points it goes
through:

* ``paged``   ``dvattn_paged_sdpa``: decode (S = 1), verification of a few
  speculated tokens (S = 2..8), chunks and prefill (S from 16 up, causal);
* ``varlen``  ``dvattn_varlen_paged_sdpa``: packed tokens, one decode token per
  sequence over several views, or decodes batched with prompt chunks;
* ``fused``   ``dvattn_fused`` on one contiguous cache per sequence;
* ``worker``  one layer's attention step of several workers that share all
  segments: ``dvattn_paged_kv_append``, ``dvattn_view_metadata`` and
  ``dvattn_fused``, in the order the model integration calls them;
* ``append``  ``dvattn_paged_kv_append``: new tokens written to their pages.

All heads are 128 wide with 16 query heads per KV head, the shape the operators
implement.
"""
from __future__ import annotations

import math

import numpy as np
import torch

E = 128
GQA = 16
SCALE = E ** -0.5
DTYPES = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}
ESIZE = {"fp32": 4, "fp16": 2, "bf16": 2}


# ---------------------------------------------------------------------------
# The cases.
def listed():
    return [
        # a single short sequence in fp32: the smallest call, where latency counts
        dict(name="fused_single_fp32", kind="fused", dtype="fp32", W=1, Hkv=1, lo=512, hi=512, layout=1, R=64),
        # interactive decode of one conversation
        dict(name="paged_single_bf16", kind="paged", dtype="bf16", W=1, Hkv=8, S=1, lo=3001, hi=3001, layout=2,
             R=128, bs=16),
        # batched decode, ragged lengths: the headline workload
        dict(name="paged_batch_bf16", kind="paged", dtype="bf16", W=32, Hkv=8, S=1, lo=1024, hi=8192, layout=3,
             R=128, bs=16),
        # long-context decode
        dict(name="paged_long_bf16", kind="paged", dtype="bf16", W=4, Hkv=8, S=1, lo=131072, hi=131072, layout=4,
             R=128, bs=64),
        # batched decode in fp32, a page size that is no power of two
        dict(name="paged_batch_fp32", kind="paged", dtype="fp32", W=24, Hkv=4, S=1, lo=512, hi=4096, layout=5,
             R=64, bs=24),
        # verification of four speculated tokens per sequence
        dict(name="paged_verify_bf16", kind="paged", dtype="bf16", W=32, Hkv=8, S=4, lo=1024, hi=8192, layout=6,
             R=128, bs=16),
        # chunk of 16 tokens on a long context
        dict(name="paged_chunk_bf16", kind="paged", dtype="bf16", W=16, Hkv=8, S=16, lo=8208, hi=8208, layout=7,
             R=32, bs=16),
        # prompt prefill in chunks of 2048 tokens, the largest amount of arithmetic
        dict(name="paged_prefill_bf16", kind="paged", dtype="bf16", W=2, Hkv=8, S=2048, lo=3800, hi=4400, layout=8,
             R=128, bs=16),
        # packed decode, every sequence's cache made of two to four views
        dict(name="varlen_views_fp16", kind="varlen", dtype="fp16", W=64, Hkv=4, lo=64, hi=32768, median=2048,
             views=4, chunks=0, chunk=0, layout=9, R=64, bs=16),
        # continuous batching: decodes and two prompt chunks in one call
        dict(name="varlen_mixed_bf16", kind="varlen", dtype="bf16", W=50, Hkv=4, lo=256, hi=8192, median=2048,
             views=1, chunks=2, chunk=250, layout=10, R=128, bs=16),
        # one layer's step of four workers over a shared prompt and each other's tokens
        dict(name="worker_step_bf16", kind="worker", dtype="bf16", W=4, Hkv=4, S=1, prompt=2500, lo=200, hi=700,
             layout=11, R=128, cap=4096),
        # keys and values of a prompt written to their pages
        dict(name="append_prompt_bf16", kind="append", dtype="bf16", W=4, Hkv=8, S=2047, lo=2047, hi=3000,
             layout=12, R=128, bs=16),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    limit = max(_cost(c) for c in listed())
    while True:
        family = rng.choice(["fused", "decode", "decode", "verify", "chunk", "prefill", "views", "mixed", "worker",
                             "append"])
        c = dict(dtype=rng.choice(["bf16", "bf16", "fp16", "fp32"]), Hkv=rng.choice([1, 2, 4, 8]),
                 layout=rng.randrange(1 << 30), R=rng.choice([32, 64, 128]))
        bs = rng.choice([16, 16, 24, 32, 64])
        if family == "fused":
            hi = _log_int(rng, 64, 8192)
            c.update(kind="fused", W=_log_int(rng, 1, 16), lo=max(1, hi // 2), hi=hi)
        elif family == "decode":
            hi = _log_int(rng, 128, 131072)
            c.update(kind="paged", W=_log_int(rng, 1, 64), S=1, lo=max(1, hi // 8), hi=hi, bs=bs)
        elif family == "verify":
            hi = _log_int(rng, 256, 16384)
            c.update(kind="paged", W=_log_int(rng, 1, 32), S=rng.randint(2, 8), lo=hi // 4, hi=hi, bs=bs)
        elif family == "chunk":
            hi = _log_int(rng, 256, 16384)
            c.update(kind="paged", W=_log_int(rng, 1, 16), S=rng.randint(9, 64), lo=hi // 2, hi=hi, bs=bs)
        elif family == "prefill":
            s = _log_int(rng, 65, 2048)
            hi = s + _log_int(rng, 1, 4096)
            c.update(kind="paged", W=_log_int(rng, 1, 4), S=s, lo=s, hi=hi, bs=bs)
        elif family == "views":
            median = _log_int(rng, 256, 4096)
            c.update(kind="varlen", W=_log_int(rng, 2, 64), lo=64, hi=8 * median, median=median,
                     views=rng.randint(2, 4), chunks=0, chunk=0, bs=bs)
        elif family == "mixed":
            median = _log_int(rng, 256, 4096)
            w = _log_int(rng, 2, 64)
            c.update(kind="varlen", W=w, lo=64, hi=4 * median, median=median, views=1,
                     chunks=rng.randint(1, min(w, 4)), chunk=_log_int(rng, 8, 512), bs=bs)
        elif family == "worker":
            own = _log_int(rng, 16, 2048)
            c.update(kind="worker", W=rng.randint(2, 8), S=rng.choice([1, 1, 1, 2, 5]),
                     prompt=_log_int(rng, 16, 8192), lo=max(8, own // 2), hi=own, cap=8192)
        else:
            s = _log_int(rng, 1, 4096)
            c.update(kind="append", W=_log_int(rng, 1, 64), S=s, lo=s, hi=s + _log_int(rng, 1, 2048), bs=bs)
        cost = _cost(c)
        if cost <= limit:
            return c


def _cost(case):
    w = work(case)
    rate = 1e14 if case["dtype"] == "fp32" else 1e15
    return w["bytes"] / 6e12 + w["flops"] / rate


# ---------------------------------------------------------------------------
# What a case's numbers fix: lengths, views and tokens (the same for every seed).
def _layout(case):
    rng = np.random.default_rng(case["layout"])
    kind, W = case["kind"], case["W"]
    if kind == "varlen":
        L = np.exp(rng.normal(math.log(case["median"]), 1.0, size=W))
        L = np.clip(np.round(L), case["lo"], case["hi"]).astype(np.int64)
    else:
        L = rng.integers(case["lo"], case["hi"], size=W, endpoint=True).astype(np.int64)
    if kind != "varlen":
        return dict(L=L)
    F = case["views"]
    tokens = np.ones(W, dtype=np.int64)
    if case["chunks"]:
        who = rng.choice(W, size=case["chunks"], replace=False)
        tokens[who] = np.maximum(1, np.minimum(L[who], case["chunk"] - rng.integers(0, 8, size=len(who))))
    lens = np.zeros((W, F), dtype=np.int64)
    nv = rng.integers(min(2, F), F, size=W, endpoint=True)
    for w in range(W):
        cuts = np.sort(rng.choice(np.arange(1, L[w]), size=nv[w] - 1, replace=False))
        lens[w, :nv[w]] = np.diff(np.concatenate([[0], cuts, [L[w]]]))
    return dict(L=L, tokens=tokens, lens=lens, nv=nv)


def work(case):
    """Bytes and operations of one pass: every visible K/V row of a sequence
    once, queries, outputs and tables once; 4 * E operations per query head and
    visible key."""
    kind, W, Hkv, es, R = case["kind"], case["W"], case["Hkv"], ESIZE[case["dtype"]], case["R"]
    lay = _layout(case)
    L = lay["L"]
    row = Hkv * 2 * E * es
    head = GQA * Hkv * E
    if kind == "append":
        n = W * case["S"]
        return dict(bytes=int(2 * n * row + 2 * n * R * es + 8 * n), flops=int(3 * n * Hkv * R))
    if kind == "paged":
        S = case["S"]
        seen = S * L - S * (S - 1) // 2  # query s of S sees L - S + s + 1 keys
        n = W * S
        tables = n * 4 + int(((L + case["bs"] - 1) // case["bs"]).sum()) * 4
        return dict(bytes=int(L.sum() * row + 2 * n * head * es + 2 * n * R * 4 + tables),
                    flops=int(seen.sum() * GQA * Hkv * 4 * E))
    if kind == "varlen":
        t = lay["tokens"]
        seen = t * L - t * (t - 1) // 2
        n, F = int(t.sum()), case["views"]
        tables = F * n * 4 + int(((L + case["bs"] - 1) // case["bs"]).sum()) * 4 + W * 4
        return dict(bytes=int(L.sum() * row + 2 * n * head * es + F * n * R * 4 + tables),
                    flops=int(seen.sum() * GQA * Hkv * 4 * E))
    if kind == "fused":
        return dict(bytes=int(L.max() * W * row + 3 * W * head * es + 2 * W * R * 4),
                    flops=int(L.sum() * GQA * Hkv * 4 * E))
    # worker: the segments are shared, so their rows are read once; the new
    # tokens' rows are read, written and attended to
    S, F = case["S"], W + 1
    n = W * S
    total = case["prompt"] + int(L.sum())
    return dict(bytes=int(total * row + 2 * n * row + (2 + F) * n * head * es + 2 * F * n * R * 4 * 2),
                flops=int(n * total * GQA * Hkv * 4 * E))


def tolerance(case):
    """About four times what the operators measured against 64-bit arithmetic:
    16-bit inputs and outputs, queries rounded after their rotation and
    probabilities rounded for the second product.  The largest single
    difference is looser: one rounding of a large element beside many small
    ones (a prompt's first tokens average few values)."""
    if case["dtype"] == "fp32":
        return {"rel": 5e-6, "max": 8e-5}
    if case["dtype"] == "fp16":
        return {"rel": 1.8e-3, "max": 2e-2}
    return {"rel": 1.8e-2, "max": 3e-1}


# ---------------------------------------------------------------------------
# Inputs.
def _rand(gen, shape, dtype, scale=1.0):
    t = torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32)
    if scale != 1.0:
        t.mul_(scale)
    return t.to(dtype)


def _inv_freq(R):
    return 1e4 ** (-np.arange(0, R, 2, dtype=np.float64) / R)


def _cos_sin(positions, R):
    """float32 ``[..., R]`` tables of integer positions, both halves alike."""
    ang = np.asarray(positions, dtype=np.float64)[..., None] * _inv_freq(R)
    ang = np.concatenate([ang, ang], axis=-1)
    return (torch.from_numpy(np.cos(ang).astype(np.float32)).cuda(),
            torch.from_numpy(np.sin(ang).astype(np.float32)).cuda())


def _i32(a):
    return torch.from_numpy(np.ascontiguousarray(a).astype(np.int32)).cuda()


def _pages(rng, counts, logical=None, width=None):
    """Block tables of sequences with ``counts[w]`` pages, scattered over the
    pool; ``logical[w]``: the logical pages that are backed (default: the first
    ``counts[w]``)."""
    W = len(counts)
    total = int(sum(counts))
    perm = rng.permutation(total).astype(np.int32)
    bt = np.zeros((W, width or max(1, int(max(counts)))), dtype=np.int32)
    o = 0
    for w in range(W):
        n = int(counts[w])
        bt[w, logical[w] if logical is not None else np.arange(n)] = perm[o:o + n]
        o += n
    return bt, total


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    rng = np.random.default_rng(seed)
    kind, W, Hkv, R = case["kind"], case["W"], case["Hkv"], case["R"]
    dt = DTYPES[case["dtype"]]
    Hq = GQA * Hkv
    lay = _layout(case)
    L = lay["L"]
    st = dict(kind=kind)
    if kind in ("paged", "append"):
        S, bs = case["S"], case["bs"]
        bt, P = _pages(rng, (L + bs - 1) // bs)
        pos = L[:, None] - S + np.arange(S)[None, :]
        st.update(block_tables=_i32(bt), k_cache=_rand(gen, (P, bs, Hkv, E), dt),
                  v_cache=_rand(gen, (P, bs, Hkv, E), dt))
        if kind == "paged":
            cos, sin = _cos_sin(pos[None], R)
            st.update(queries=_rand(gen, (W, Hq, S, E), dt, 2.0), locations=_i32(pos[None]), cos=cos, sin=sin,
                      lengths=_i32([L.max()]))
        else:
            # keys and values as the projections leave them, tokens before heads
            cos, sin = _cos_sin(pos, R)
            st.update(keys=_rand(gen, (W, S, Hkv, E), dt).transpose(1, 2),
                      values=_rand(gen, (W, S, Hkv, E), dt).transpose(1, 2), positions=_i32(pos), cos=cos.to(dt),
                      sin=sin.to(dt))
    elif kind == "varlen":
        bs, F, lens, tokens = case["bs"], case["views"], lay["lens"], lay["tokens"]
        fl = lens.max(axis=0)
        off = np.concatenate([[0], np.cumsum(fl)[:-1]])
        logical = []
        for w in range(W):
            backed = set()
            for f in range(F):
                if lens[w, f]:
                    backed.update(range(int(off[f]) // bs, int(off[f] + lens[w, f] - 1) // bs + 1))
            logical.append(sorted(backed))
        bt, P = _pages(rng, [len(x) for x in logical], logical, (int(fl.sum()) + bs - 1) // bs)
        seq = np.repeat(np.arange(W), tokens)
        T = len(seq)
        cu = np.concatenate([[0], np.cumsum(tokens)])
        back = tokens[seq] - 1 - (np.arange(T) - cu[seq])  # tokens of the sequence after this one
        # the last view holds the newest tokens: causal there, whole views before it
        loc = np.where(np.arange(F)[:, None] < lay["nv"][seq][None, :], lens[seq].T - 1, -1)
        last = lay["nv"][seq] - 1
        loc[last, np.arange(T)] -= back
        rel = rng.integers(0, 65536, size=(F, T)) if F > 1 else loc
        cos, sin = _cos_sin(rel, R)
        st.update(block_tables=_i32(bt), k_cache=_rand(gen, (P, bs, Hkv, E), dt),
                  v_cache=_rand(gen, (P, bs, Hkv, E), dt), queries=_rand(gen, (T, Hq, E), dt, 2.0),
                  locations=_i32(loc), cos=cos[..., :R // 2].contiguous(), sin=sin[..., :R // 2].contiguous(),
                  lengths=_i32(fl), cu_q=_i32(cu), cu_k=_i32(np.concatenate([[0], np.cumsum(L)])), seq=seq)
    elif kind == "fused":
        n = int(L.max())
        cos, sin = _cos_sin((L - 1)[None, :, None], R)
        st.update(keys=[_rand(gen, (W, Hkv, n, E), dt)], values=[_rand(gen, (W, Hkv, n, E), dt)],
                  queries=_rand(gen, (W, Hq, 1, E), dt, 2.0), locations=_i32((L - 1)[None, :, None]), cos=cos,
                  sin=sin, lengths=_i32([n]), rq=torch.empty((1, W, Hq, 1, E), dtype=dt, device="cuda"),
                  out=torch.empty((W, Hq, 1, E), dtype=dt, device="cuda"))
    else:
        S, cap, F = case["S"], case["cap"], W + 1
        lens = np.concatenate([[case["prompt"]], L])  # with the new tokens
        # every worker sees the prompt, the others' segments, then its own
        order = np.array([[0] + [1 + v for v in range(W) if v != w] + [1 + w] for w in range(W)])
        pos = L[:, None] - S + np.arange(S)[None, :]
        cos, sin = _cos_sin(pos, R)
        pk, pv = _rand(gen, (F, Hkv, cap, E), dt), _rand(gen, (F, Hkv, cap, E), dt)
        st.update(pool_k=pk, pool_v=pv, new_k=_rand(gen, (W, S, Hkv, E), dt).transpose(1, 2),
                  new_v=_rand(gen, (W, S, Hkv, E), dt).transpose(1, 2), positions=_i32(pos), new_cos=cos.to(dt),
                  new_sin=sin.to(dt), table=_i32(1 + np.arange(W)[:, None]), lengths=_i32(lens), order=_i32(order),
                  inv_freq=torch.from_numpy(_inv_freq(R).astype(np.float32)).cuda(), S=S,
                  round_to=None if dt == torch.float32 else dt, queries=_rand(gen, (W, Hq, S, E), dt, 2.0),
                  keys=[pk[f:f + 1] for f in range(F)], values=[pv[f:f + 1] for f in range(F)],
                  rq=torch.empty((F, W, Hq, S, E), dtype=dt, device="cuda"),
                  out=torch.empty((W, Hq, S, E), dtype=dt, device="cuda"))
    return st


def run(state):
    import dvattention_amd as dv

    s = state
    kind = s["kind"]
    if kind == "paged":
        return dv.dvattn_paged_sdpa(s["queries"], s["locations"], s["cos"], s["sin"], s["lengths"], s["k_cache"],
                                    s["v_cache"], s["block_tables"], SCALE)
    if kind == "varlen":
        return dv.dvattn_varlen_paged_sdpa(s["queries"], s["locations"], s["cos"], s["sin"], s["lengths"],
                                           s["k_cache"], s["v_cache"], s["block_tables"], s["cu_q"], s["cu_k"],
                                           SCALE)
    if kind == "fused":
        out = dv.dvattn_fused(s["queries"], s["locations"], s["keys"], s["values"], SCALE, s["lengths"], s["cos"],
                              s["sin"], rotated_queries=s["rq"], out=s["out"])
        return out, s["rq"]
    if kind == "append":
        return dv.dvattn_paged_kv_append(s["keys"], s["values"], s["positions"], s["cos"], s["sin"], s["k_cache"],
                                         s["v_cache"], s["block_tables"])
    dv.dvattn_paged_kv_append(s["new_k"], s["new_v"], s["positions"], s["new_cos"], s["new_sin"],
                              s["pool_k"].permute(0, 2, 1, 3), s["pool_v"].permute(0, 2, 1, 3), s["table"])
    loc, cos, sin = dv.dvattn_view_metadata(s["lengths"], s["order"], s["S"], s["inv_freq"], 1.0, s["round_to"])
    out = dv.dvattn_fused(s["queries"], loc, s["keys"], s["values"], SCALE, s["lengths"], cos, sin,
                          rotated_queries=s["rq"], out=s["out"])
    return out, s["rq"], loc, cos, sin, s["pool_k"], s["pool_v"]


# ---------------------------------------------------------------------------
# The same in 64 bits.
def _rotate(x, cos, sin):
    """Partial rotation of the last dim by ``[..., R/2]`` tables."""
    h = cos.shape[-1]
    a, b = x[..., :h], x[..., h:2 * h]
    ra = a * cos - b * sin
    rest = x[..., 2 * h:].expand(*ra.shape[:-1], x.shape[-1] - 2 * h)
    return torch.cat([ra, b * cos + a * sin, rest], dim=-1)


def _attend(q, k, v, visible):
    """One KV head: q per view ``[T, 16, E]``, k / v per view ``[n, E]``, visible
    keys per view ``[T]``; softmax over the keys of all views."""
    T = visible[0].shape[0]
    scores = []
    for qf, kf, nf in zip(q, k, visible):
        s = (qf.reshape(-1, E) @ kf.T).reshape(T, GQA, -1) * SCALE
        hidden = torch.arange(kf.shape[0], device=kf.device)[None, :] >= nf[:, None]
        scores.append(s.masked_fill_(hidden[:, None, :], -math.inf))
    s = torch.cat(scores, dim=-1) if len(scores) > 1 else scores[0]
    p = torch.nan_to_num(torch.softmax(s, dim=-1))
    return (p.reshape(T * GQA, -1) @ torch.cat(v)).reshape(T, GQA, E)


def exact(case, seed):
    st = prepare(case, seed)
    kind, W, Hkv, R = case["kind"], case["W"], case["Hkv"], case["R"]
    f64 = torch.float64
    h = R // 2
    lay = _layout(case)
    if kind in ("append", "worker"):
        cos = (st["cos"] if kind == "append" else st["new_cos"]).to(f64)[..., :h]
        sin = (st["sin"] if kind == "append" else st["new_sin"]).to(f64)[..., :h]
        k_new = st["keys"] if kind == "append" else st["new_k"]
        v_new = st["values"] if kind == "append" else st["new_v"]
        k_new = _rotate(k_new.to(f64), cos[:, None], sin[:, None])  # [W, Hkv, S, E]
        pos = st["positions"].long()
        if kind == "append":
            kc, vc = st["k_cache"].to(f64), st["v_cache"].to(f64)
            bs = case["bs"]
            page = torch.gather(st["block_tables"].long(), 1, pos // bs)
            kc[page, pos % bs] = k_new.transpose(1, 2)
            vc[page, pos % bs] = v_new.to(f64).transpose(1, 2)
            return kc, vc
        pk, pv = st["pool_k"].to(f64), st["pool_v"].to(f64)
        for w in range(W):
            pk[1 + w][:, pos[w]] = k_new[w]
            pv[1 + w][:, pos[w]] = v_new[w].to(f64)
        F, S = W + 1, case["S"]
        lens = st["lengths"].tolist()
        loc = torch.empty((F, W, S), dtype=torch.int64, device="cuda")
        for w, order in enumerate(st["order"].tolist()):
            total = 0
            for f in reversed(order):
                total += lens[f]
                loc[f, w] = total - S + torch.arange(S, device="cuda")
        # the operator's angles are products rounded to fp32
        ang = (loc.to(torch.float32)[..., None] * st["inv_freq"]).to(f64)
        cos, sin = torch.cos(ang), torch.sin(ang)  # [F, W, S, R/2]
        rq = _rotate(st["queries"].to(f64)[None], cos[:, :, None], sin[:, :, None])
        out = torch.empty((W, GQA * Hkv, S, E), dtype=f64, device="cuda")
        for w in range(W):
            for j in range(Hkv):
                o = _attend([rq[f, w, GQA * j:GQA * (j + 1)].transpose(0, 1) for f in range(F)],
                            [pk[f, j, :lens[f]] for f in range(F)], [pv[f, j, :lens[f]] for f in range(F)],
                            [torch.clamp(loc[f, w] + 1, max=lens[f]) for f in range(F)])
                out[w, GQA * j:GQA * (j + 1)] = o.transpose(0, 1)
        return (out, rq, loc.to(torch.int32), torch.cat([cos, cos], -1), torch.cat([sin, sin], -1), pk, pv)
    q = st["queries"].to(f64)
    cos, sin = st["cos"].to(f64)[..., :h], st["sin"].to(f64)[..., :h]
    if kind == "fused":
        rq = _rotate(q[None], cos[:, :, None], sin[:, :, None])
        out = torch.empty_like(q)
        for w in range(W):
            n = int(lay["L"][w])
            for j in range(Hkv):
                heads = slice(GQA * j, GQA * (j + 1))
                out[w, heads, 0] = _attend([rq[0, w, heads, 0][None]], [st["keys"][0][w, j, :n].to(f64)],
                                           [st["values"][0][w, j, :n].to(f64)],
                                           [torch.tensor([n], device="cuda")])[0]
        return out, rq
    bs = case["bs"]
    fl = st["lengths"].tolist()
    off = np.concatenate([[0], np.cumsum(fl)[:-1]]).astype(np.int64)
    bt = st["block_tables"].long()
    out = torch.empty_like(q)
    for w in range(W):
        if kind == "paged":
            qw, tok = q[w].transpose(0, 1), None  # [S, Hq, E]
            cw, sw, loc = cos[:, w], sin[:, w], st["locations"][:, w].long()
        else:
            tok = torch.from_numpy(np.flatnonzero(st["seq"] == w)).cuda()
            qw, cw, sw, loc = q[tok], cos[:, tok], sin[:, tok], st["locations"][:, tok].long()
        views = []
        for f in range(len(fl)):
            seen = torch.clamp(loc[f] + 1, min=0, max=fl[f])
            n = int(seen.max())
            if n == 0:
                continue
            p = int(off[f]) + torch.arange(n, device="cuda")
            page, row = bt[w, p // bs], p % bs
            views.append((_rotate(qw, cw[f][:, None], sw[f][:, None]), st["k_cache"][page, row],
                          st["v_cache"][page, row], seen))
        for j in range(Hkv):
            heads = slice(GQA * j, GQA * (j + 1))
            o = _attend([x[0][:, heads] for x in views], [x[1][:, j].to(f64) for x in views],
                        [x[2][:, j].to(f64) for x in views], [x[3] for x in views])
            if kind == "paged":
                out[w, heads] = o.transpose(0, 1)
            else:
                out[tok, heads] = o
    return out
