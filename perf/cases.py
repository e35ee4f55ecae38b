"""The work that programs give this framework, as cases that can be timed and compared.

A case is a dict of plain values:

    name    (listed cases)
    op      "train": forward and gradients of one attention layer
            "prefill": forward only, a whole prompt
            "decode": one or a few new queries per row against a KV cache (``flex_decode``)
            "fp8": forward from bf16 inputs quantised on the way (``flex_attention_fp8``)
    entry   "flex" (``flex_attention`` with a block mask) or "flash" (``flash_attention``, the
            reference's signature with a mask mod)
    dtype   "bf16" or "fp32"
    B, Hq, Hkv, Sq, Skv, D
    mask    "none", "causal", "window" (causal, ``window`` keys), "docs" (packed documents, causal),
            "prefix" (a Python callable: the first ``window`` keys, and the causal ones)
    score   "none", "alibi_softcap" (built-in descriptors), "callable" (a Python callable)
    cache   (decode) "plain": contiguous keys, all in use; "lens": contiguous, a length per row;
            "paged": pages of ``page`` keys in any order, a length per row
"""
import math
import os
import random
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "pallas-flexattn_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import pallas_flexattn as pf  # noqa: E402

DEV = "cuda"
SOFTCAP = 50.0
CALLABLE_CAP = 30.0


def _case(op, B, Hq, Hkv, Sq, Skv, D, mask="causal", window=0, score="none", dtype="bf16", entry="flex",
          cache="plain", page=0, **more):
    return dict(op=op, entry=entry, dtype=dtype, B=B, Hq=Hq, Hkv=Hkv, Sq=Sq, Skv=Skv, D=D, mask=mask, window=window,
                score=score, cache=cache, page=page, **more)


def listed():
    return [
        # a small model or a test: a ragged length, a few launches and the call's own cost
        _case("train", 2, 4, 4, 300, 300, 64, entry="flash", name="train_small_ragged_d64"),
        # the reference's own default precision, at a length that is no multiple of a tile
        _case("train", 4, 8, 8, 1000, 1000, 64, dtype="fp32", entry="flash", name="train_fp32_ragged_d64"),
        # the workload that the reference's benchmark quotes: causal B8 H16 S2048 D128
        _case("train", 8, 16, 16, 2048, 2048, 128, name="train_causal_2k"),
        # FlexAttention's reason to be: a Python mask (prefix-LM) and a Python score mod, traced and compiled
        _case("train", 4, 16, 16, 2048, 2048, 64, mask="prefix", window=500, score="callable",
              name="train_callables_2k_d64"),
        # the largest single-GPU training shape: causal B4 H32 S8192 D128
        _case("train", 4, 32, 32, 8192, 8192, 128, name="train_causal_8k"),
        # a sliding-window layer at the same size
        _case("train", 4, 32, 32, 8192, 8192, 128, mask="window", window=1024, name="train_window_8k"),
        # grouped heads, ALiBi and a soft-cap
        _case("train", 4, 32, 8, 4096, 4096, 128, score="alibi_softcap", name="train_gqa_alibi_softcap_4k"),
        # sequence packing: documents of 256 to 4096 tokens in rows of 16384
        _case("train", 2, 16, 16, 16384, 16384, 128, mask="docs", name="train_documents_16k"),
        # one prompt of ordinary length through a serving engine: few heads, a ragged length, no gradient
        _case("prefill", 1, 32, 8, 3000, 3000, 128, name="prefill_gqa_3k"),
        # continuous batching: 32 rows of mixed lengths in a paged cache
        _case("decode", 32, 32, 8, 1, 8192, 128, mask="none", cache="paged", page=128, name="decode_paged_mixed"),
        # long contexts, a contiguous cache: bound by the reads of K and V
        _case("decode", 8, 32, 8, 1, 32768, 128, mask="none", name="decode_long_32k"),
        # the fp8 forward with its quantisation, as a bf16 caller uses it
        _case("fp8", 4, 32, 32, 8192, 8192, 128, name="fp8_forward_8k"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    # the largest training shape's time in units of bf16 fwd + bwd operations; fp32 costs about 16 times as much
    top = 14.0 * 128 * (8192.0 * 8193 / 2) * 128
    while True:
        op = rng.choice(["train", "train", "train", "train", "train", "prefill", "decode", "decode", "fp8"])
        D = rng.choice([64, 128])
        if op == "train":
            dtype = "fp32" if rng.random() < 0.25 else "bf16"
            B, Hkv, g = _log(rng, 1, 8), rng.choice([2, 4, 8, 12, 16, 32]), rng.choice([1, 1, 1, 2, 4])
            S = _log(rng, 200, 3000 if dtype == "fp32" else 16384)
            mask = rng.choice(["none", "causal", "causal", "causal", "window", "docs"])
            c = _case(op, B, Hkv * g, Hkv, S, S, D, mask=mask, dtype=dtype,
                      window=_log(rng, 64, 2048) if mask == "window" else 0,
                      score=rng.choice(["none", "none", "none", "alibi_softcap"]),
                      entry="flex")
            if c["score"] == "none" and g == 1 and rng.random() < 0.4:
                c["entry"] = "flash"
        elif op == "prefill":
            Hkv, g = rng.choice([4, 8, 16]), rng.choice([1, 4, 8])
            S = _log(rng, 100, 16384)
            c = _case(op, rng.choice([1, 1, 2, 4]), Hkv * g, Hkv, S, S, D)
        elif op == "decode":
            Hkv, g = rng.choice([2, 4, 8, 16]), rng.choice([1, 4, 4, 8])
            cache = rng.choice(["plain", "lens", "paged"])
            Skv, page = _log(rng, 256, 32768), 0
            if cache == "paged":
                page = rng.choice([64, 128, 256, 512])
                Skv = -(-Skv // page) * page
            c = _case(op, _log(rng, 1, 64), Hkv * g, Hkv, rng.choice([1, 1, 1, 4]), Skv, D, mask="none", cache=cache,
                      page=page)
            if 4.0 * c["B"] * Hkv * Skv * D > 2e9:
                continue
        else:
            S, H = _log(rng, 500, 8192), rng.choice([8, 16, 32])
            c = _case(op, _log(rng, 1, 4), H, H, S, S, D, mask=rng.choice(["causal", "none"]))
        cost = work(c)["flops"] * (16 if c["dtype"] == "fp32" else 1)
        if cost <= top and c["B"] * c["Hq"] * c["Sq"] * D <= 4 * 32 * 8192 * 128:
            return c


# ---------------------------------------------------------------- what a case is made of ----
def _shape_rng(case, tag):
    return random.Random(f"{tag}/{case['B']}/{case['Sq']}/{case['Skv']}")


def _doc_lengths(case):
    """Document lengths of each batch row (256 to 4096 tokens in a row of 16384, in proportion below that)."""
    S, rows, r = case["Sq"], [], _shape_rng(case, "docs")
    lo, hi = max(1, min(256, S // 8)), max(2, min(4096, S // 2))
    for _ in range(case["B"]):
        lens, left = [], S
        while left > 0:
            lens.append(min(left, r.randint(lo, hi)))
            left -= lens[-1]
        rows.append(lens)
    return rows


def _kv_lens(case):
    """Keys in use of each batch row: the longest fills the cache, the others a tenth of it and more."""
    if case["cache"] == "plain":
        return [case["Skv"]] * case["B"]
    r = _shape_rng(case, "lens")
    return [case["Skv"]] + [max(case["Sq"], int(case["Skv"] * r.uniform(0.1, 1.0))) for _ in range(case["B"] - 1)]


def _pairs(case):
    """Unmasked (query, key) pairs of one head, summed over the batch."""
    S, B, w = case["Sq"], case["B"], case["window"]
    if case["op"] == "decode":
        return S * sum(_kv_lens(case))
    if case["mask"] == "none":
        return B * S * case["Skv"]
    if case["mask"] == "docs":
        return sum(n * (n + 1) // 2 for row in _doc_lengths(case) for n in row)
    if case["mask"] == "window":
        w = min(w, S)
        return B * (w * (w + 1) // 2 + (S - w) * w)
    causal = S * (S + 1) // 2
    if case["mask"] == "prefix":
        w = min(w, S)
        causal += w * (w - 1) // 2
    return B * causal


def work(case):
    B, Hq, Hkv, Sq, Skv, D = (case[x] for x in ("B", "Hq", "Hkv", "Sq", "Skv", "D"))
    es = 4 if case["dtype"] == "fp32" else 2
    q, pairs = B * Hq * Sq * D * es, _pairs(case)
    kv = 2 * B * Hkv * Skv * D * es
    if case["op"] == "decode":
        kv = 2 * sum(_kv_lens(case)) * Hkv * D * es
    if case["op"] == "train":  # q, k, v, dO in; O, dQ, dK, dV out
        return {"bytes": 4.0 * q + 2.0 * kv, "flops": 14.0 * D * pairs * Hq}
    return {"bytes": 2.0 * q + kv, "flops": 4.0 * D * pairs * Hq}


def tolerance(case):
    # measured against exact(): bf16 2.0e-3 (O) to 2.8e-3 (gradients), fp32 3e-7 to 6e-7, fp8 0.05 with the
    # inputs' own rounding in it.  "max" is wide because early causal rows are far larger than the mean row
    if case["op"] == "fp8":  # P is rounded to e4m3 against a running maximum: 2^-4 a value
        return {"rel": 0.03, "max": 0.5}
    if case["dtype"] == "fp32":
        return {"rel": 1e-5, "max": 2e-4}
    return {"rel": 0.01, "max": 0.2}


def _normals(case, seed, shapes):
    g = torch.Generator(device=DEV).manual_seed(int(seed) * 7919 + 11)
    dt = torch.float32 if case["dtype"] == "fp32" else torch.bfloat16
    return [torch.randn(*s, device=DEV, generator=g).to(dt) for s in shapes]


def _rows_of(case, seed):
    """The documents, or the cache lengths, of this seed: the case's own, in another order."""
    r = random.Random(int(seed))
    if case["mask"] == "docs":
        rows = _doc_lengths(case)
        for lens in rows:
            r.shuffle(lens)
        return rows
    lens = _kv_lens(case)
    r.shuffle(lens)
    return lens


def _callable_score(s, b, h, q, kv):
    return CALLABLE_CAP * torch.tanh(s / CALLABLE_CAP)


def _prefix_mask(n):
    def prefix_lm(q, kv):
        return (kv <= q) | (kv < n)
    return prefix_lm


def _mask_mod(case, seed):
    m = case["mask"]
    if m == "none":
        return None
    if m == "causal":
        return pf.causal_mask
    if m == "window":
        return pf.sliding_window_mask(case["window"] - 1, 0)
    if m == "docs":
        return pf.and_masks(pf.document_mask(_rows_of(case, seed)), pf.causal_mask)
    return _prefix_mask(case["window"])


def _score_mod(case):
    if case["score"] == "alibi_softcap":
        return pf.compose_score_mods(pf.alibi_score_mod(case["Hq"]), pf.softcap_score_mod(SOFTCAP))
    return _callable_score if case["score"] == "callable" else None


def prepare(case, seed):
    B, Hq, Hkv, Sq, Skv, D = (case[x] for x in ("B", "Hq", "Hkv", "Sq", "Skv", "D"))
    st = dict(op=case["op"], entry=case["entry"], gqa=Hq != Hkv)
    if case["op"] == "decode":
        q, k, v = _normals(case, seed, [(B, Hq, Sq, D), (B, Hkv, Skv, D), (B, Hkv, Skv, D)])
        st.update(q=q, k=k, v=v, lens=None, pages=None)
        if case["cache"] != "plain":
            st["lens"] = torch.tensor(_rows_of(case, seed), dtype=torch.int32, device=DEV)
        if case["cache"] == "paged":
            n = Skv // case["page"]
            g = torch.Generator().manual_seed(int(seed))
            perm = torch.randperm(B * n, generator=g)

            def paged(x):  # page perm[b n + i] of the cache holds keys i page .. of row b
                p = x.view(B, Hkv, n, case["page"], D).permute(0, 2, 1, 3, 4).reshape(B * n, Hkv, case["page"], D)
                out = torch.empty_like(p)
                out[perm.to(DEV)] = p
                return out
            st.update(k=paged(k), v=paged(v), pages=perm.view(B, n).to(torch.int32).to(DEV))
        return st
    mask = _mask_mod(case, seed)
    q, k, v = _normals(case, seed, [(B, Hq, Sq, D), (B, Hkv, Skv, D), (B, Hkv, Skv, D)])
    st.update(q=q, k=k, v=v, mask=mask, score=_score_mod(case), block_mask=None)
    if case["entry"] == "flex" and mask is not None:
        dev = DEV if case["mask"] != "prefix" else None
        st["block_mask"] = pf.create_block_mask(mask, B, Hq, Sq, Skv, 128, device=dev)
    if case["op"] == "train":
        for t in (q, k, v):
            t.requires_grad_(True)
        st["do"] = _normals(case, int(seed) + 1000003, [(B, Hq, Sq, D)])[0]
    return st


def run(st):
    q, k, v = st["q"], st["k"], st["v"]
    if st["op"] == "decode":
        return [pf.flex_decode(q, k, v, enable_gqa=st["gqa"], kv_lens=st["lens"], page_table=st["pages"])]
    if st["op"] == "fp8":
        return [pf.flex_attention_fp8(q, k, v, block_mask=st["block_mask"], enable_gqa=st["gqa"])]
    if st["entry"] == "flash":
        o = pf.flash_attention(q, k, v, mask_mod=st["mask"])
    else:
        o = pf.flex_attention(q, k, v, score_mod=st["score"], block_mask=st["block_mask"], enable_gqa=st["gqa"])
    if st["op"] == "prefill":
        return [o]
    dq, dk, dv = torch.autograd.grad(o, (q, k, v), st["do"])
    return [o.detach(), dq, dk, dv]


# ---------------------------------------------------------------- the same in 64 bits ----
def _dense_mask(case, rows, b):
    """Boolean (Sq, Skv) of batch row b, or None where everything is seen."""
    if case["mask"] == "none":
        return None
    qi = torch.arange(case["Sq"], device=DEV)[:, None]
    ki = torch.arange(case["Skv"], device=DEV)[None, :]
    m = ki <= qi
    if case["mask"] == "window":
        m = m & (qi - ki < case["window"])
    elif case["mask"] == "prefix":
        m = m | (ki < case["window"])
    elif case["mask"] == "docs":
        ids = torch.from_numpy(np.repeat(np.arange(len(rows[b])), rows[b])).to(DEV)
        m = m & (ids[:, None] == ids[None, :])
    return m


def exact(case, seed):
    B, Hq, Hkv, Sq, Skv, D = (case[x] for x in ("B", "Hq", "Hkv", "Sq", "Skv", "D"))
    g, f64 = Hq // Hkv, torch.float64
    q, k, v = _normals(case, seed, [(B, Hq, Sq, D), (B, Hkv, Skv, D), (B, Hkv, Skv, D)])
    train = case["op"] == "train"
    do = _normals(case, int(seed) + 1000003, [(B, Hq, Sq, D)])[0] if train else None
    rows = _rows_of(case, seed)
    out = torch.empty(q.shape, dtype=f64, device=DEV)
    grads = [torch.zeros(t.shape, dtype=f64, device=DEV) for t in (q, k, v)] if train else []
    scale = 1.0 / math.sqrt(D)
    slopes = (2.0 ** (-8.0 * torch.arange(Hq, dtype=f64) / Hq)).float().double().tolist()
    dist = None
    if case["score"] == "alibi_softcap":
        dist = (torch.arange(Skv, device=DEV)[None, :] - torch.arange(Sq, device=DEV)[:, None]).to(f64)
    cap = {"alibi_softcap": SOFTCAP, "callable": CALLABLE_CAP}.get(case["score"], 0.0)
    for b in range(B):
        n = rows[b] if case["op"] == "decode" else Skv
        mask = _dense_mask(case, rows, b)
        for h in range(Hq):
            kk, vv, qq = k[b, h // g, :n].to(f64), v[b, h // g, :n].to(f64), q[b, h].to(f64)
            s = (qq @ kk.t()) * scale
            if dist is not None:
                s += slopes[h] * dist
            if cap:
                th = torch.tanh(s / cap)
                s = cap * th
            if mask is not None:
                s.masked_fill_(~mask, -math.inf)
            p = torch.softmax(s, dim=-1)
            del s
            o = p @ vv
            out[b, h] = o
            if not train:
                continue
            dd = do[b, h].to(f64)
            grads[2][b, h // g] += p.t() @ dd
            ds = p * (dd @ vv.t() - (o * dd).sum(-1, keepdim=True))
            del p
            if cap:
                ds *= 1.0 - th * th
            grads[0][b, h] = (ds @ kk) * scale
            grads[1][b, h // g] += (ds.t() @ qq) * scale
            del ds
    return [out] + grads
