"""The work that the speed of this framework is judged by.

Every case goes through the public entry points of ``triton-kernels_amd``
(``kernels.attention``, ``kernels.decode``, ``kernels.speculative_decode``,
``kernels.paged_cache``) the way a serving program calls them: prefill of one
prompt and of batches (dense, ragged, paged chunks), cross attention, decode
steps, speculative decode steps and cache appends, in bf16, fp16 and fp32.

A case is a dict of plain values: ``kind`` names the family below, ``lens`` of
ragged and paged families follow from (``n``, ``lo``, ``hi``, ``lens_seed``).
"""

from __future__ import annotations

import math
import os
import random
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "triton-kernels_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from kernels.attention import flash_attention_v2  # noqa: E402
from kernels.decode import decode_attention  # noqa: E402
from kernels.paged_cache import paged_kv_append  # noqa: E402
from kernels.speculative_decode import speculative_decode_attention  # noqa: E402

PAGE = 16
_DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
_BYTES = {"bf16": 2, "f16": 2, "f32": 4}


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------

def listed():
    return [
        # One short prompt of a small model: the call's latency and the work of
        # very few thread blocks (the test suite's and benchmark's c1).
        dict(name="prefill_dense_small", kind="dense", dtype="f16", b=1, hq=8, hkv=8, lq=512,
             lk=512, d=64, causal=True),
        # Prefill of two equal prompts with grouped heads: the headline
        # configuration (c2).
        dict(name="prefill_dense_gqa", kind="dense", dtype="bf16", b=2, hq=32, hkv=8, lq=2048,
             lk=2048, d=128, causal=True),
        # A serving batch of prompts of unequal, odd lengths, packed token by
        # token (c3's shape).
        dict(name="prefill_ragged_gqa", kind="ragged", dtype="bf16", n=16, lo=128, hi=4096,
             lens_seed=0, q_lo=0, q_hi=0, hq=32, hkv=8, d=128, causal=True),
        # Chunked prefill against paged contexts: 128 new tokens per sequence,
        # diagonal at the context's end (c4's shape).
        dict(name="prefill_paged_chunk", kind="paged", dtype="bf16", n=32, lo=512, hi=8192,
             lens_seed=0, lq=128, hq=32, hkv=8, d=128, causal=True),
        # Long cross attention with one shared kv head (c5): the largest call.
        dict(name="cross_dense_mqa", kind="dense", dtype="bf16", b=4, hq=32, hkv=1, lq=1024,
             lk=16384, d=128, causal=False),
        # A batch of short queries over short memories of odd lengths, the
        # range of the reference benchmark's small points (B16, 8 query heads):
        # an encoder-decoder's or reranker's call.
        dict(name="cross_ragged_small", kind="ragged", dtype="f16", n=16, lo=65, hi=511,
             lens_seed=1, q_lo=17, q_hi=128, hq=8, hkv=2, d=128, causal=False),
        # Prefill of fp32 tensors (reference arithmetic: operands rounded to
        # fp16, fp32 accumulation and output), odd length.
        dict(name="prefill_dense_f32", kind="dense", dtype="f32", b=2, hq=16, hkv=4, lq=1500,
             lk=1500, d=128, causal=True),
        # A decode step of a full serving batch over a shuffled page pool
        # (the benchmark's d2).
        dict(name="decode_paged_gqa", kind="decode_paged", dtype="bf16", n=64, lo=512, hi=8192,
             lens_seed=2, m=0, hq=32, hkv=8, d=128),
        # A decode step of an interactive session: few sequences, short cache,
        # latency.
        dict(name="decode_dense_small", kind="decode_dense", dtype="f16", b=4, hq=32, hkv=8,
             lk=1023, d=128),
        # A speculative step, 8 drafts per sequence, many heads of 64 dims
        # without grouping (the benchmark's s1).
        dict(name="spec_paged_mha", kind="decode_paged", dtype="bf16", n=16, lo=8192, hi=8200,
             lens_seed=3, m=8, hq=8, hkv=8, d=64),
        # The same step on an fp32 cache with grouped heads (fp32 arithmetic).
        dict(name="spec_paged_f32", kind="decode_paged", dtype="f32", n=16, lo=512, hi=4096,
             lens_seed=4, m=8, hq=16, hkv=4, d=128),
        # Writing a prefill chunk's new keys and values into the page pools.
        dict(name="append_paged", kind="append", dtype="bf16", n=16, lo=64, hi=1024,
             lens_seed=5, hkv=8, d=128),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["dense", "cross", "ragged", "paged", "cross_ragged", "f32", "decode_paged",
                       "decode_dense", "spec", "spec_f32", "append"])
    half = rng.choice(["bf16", "f16"])
    heads = rng.choice([(8, 8), (8, 2), (16, 16), (16, 4), (32, 8), (32, 4)])
    d = rng.choice([64, 128, 128])
    seed = rng.randrange(1 << 20)
    if kind == "dense":
        n = _log_int(rng, 100, 4096)
        return dict(kind="dense", dtype=half, b=rng.randint(1, 4), hq=heads[0], hkv=heads[1],
                    lq=n, lk=n, d=d, causal=True)
    if kind == "cross":
        return dict(kind="dense", dtype=half, b=rng.randint(1, 4), hq=32, hkv=rng.choice([1, 4, 8]),
                    lq=_log_int(rng, 64, 1024), lk=_log_int(rng, 512, 16384), d=d, causal=False)
    if kind == "ragged":
        return dict(kind="ragged", dtype=half, n=rng.randint(2, 16), lo=rng.randint(1, 200),
                    hi=_log_int(rng, 300, 4096), lens_seed=seed, q_lo=0, q_hi=0, hq=heads[0],
                    hkv=heads[1], d=d, causal=True)
    if kind == "paged":
        return dict(kind="paged", dtype=half, n=rng.randint(2, 32), lo=rng.randint(128, 512),
                    hi=_log_int(rng, 600, 8192), lens_seed=seed, lq=rng.choice([32, 77, 128, 128]),
                    hq=heads[0], hkv=heads[1], d=d, causal=True)
    if kind == "cross_ragged":
        return dict(kind="ragged", dtype=half, n=rng.randint(2, 24), lo=rng.randint(1, 128),
                    hi=_log_int(rng, 200, 2048), lens_seed=seed, q_lo=rng.randint(1, 64),
                    q_hi=rng.randint(65, 512), hq=8, hkv=rng.choice([1, 2, 8]), d=d, causal=False)
    if kind == "f32":
        n = _log_int(rng, 100, 3000)
        return dict(kind="dense", dtype="f32", b=rng.randint(1, 3), hq=heads[0], hkv=heads[1],
                    lq=n, lk=n, d=d, causal=rng.random() < 0.7)
    if kind == "decode_paged":
        return dict(kind="decode_paged", dtype=half, n=_log_int(rng, 1, 64),
                    lo=rng.randint(16, 512), hi=_log_int(rng, 600, 8192), lens_seed=seed, m=0,
                    hq=heads[0], hkv=heads[1], d=d)
    if kind == "decode_dense":
        return dict(kind="decode_dense", dtype=half, b=_log_int(rng, 1, 16), hq=heads[0],
                    hkv=heads[1], lk=_log_int(rng, 64, 8192), d=d)
    if kind == "spec":
        return dict(kind="decode_paged", dtype=half, n=_log_int(rng, 1, 64),
                    lo=rng.randint(16, 512), hi=_log_int(rng, 600, 8192), lens_seed=seed,
                    m=rng.randint(2, 8), hq=heads[0], hkv=heads[1], d=d)
    if kind == "spec_f32":
        return dict(kind="decode_paged", dtype="f32", n=_log_int(rng, 1, 32),
                    lo=rng.randint(16, 512), hi=_log_int(rng, 600, 4096), lens_seed=seed,
                    m=rng.choice([0, 2, 4, 8]), hq=heads[0], hkv=heads[1], d=d)
    return dict(kind="append", dtype=half, n=_log_int(rng, 1, 64), lo=1,
                hi=_log_int(rng, 2, 2048), lens_seed=seed, hkv=heads[1], d=d)


# ---------------------------------------------------------------------------
# sizes
# ---------------------------------------------------------------------------

def _kv_lens(case):
    r = random.Random(case["lens_seed"])
    return [r.randint(case["lo"], case["hi"]) for _ in range(case["n"])]


def _q_lens(case):
    """Ragged: query rows per sequence (the kv lengths when self attention)."""
    if case["q_hi"] == 0:
        return _kv_lens(case)
    r = random.Random(case["lens_seed"] + 1)
    return [r.randint(case["q_lo"], case["q_hi"]) for _ in range(case["n"])]


def _pairs(lq, lk, causal, off):
    """Visible (query, key) pairs; row i sees keys j <= i + off."""
    if not causal:
        return lq * lk
    return sum(min(max(i + off + 1, 0), lk) for i in range(lq))


def _sequences(case):
    """(query rows, keys, causal, diagonal offset) of every sequence."""
    kind = case["kind"]
    if kind == "dense":
        return [(case["lq"], case["lk"], case["causal"], 0)] * case["b"]
    if kind == "ragged":
        return [(a, b, case["causal"], 0) for a, b in zip(_q_lens(case), _kv_lens(case))]
    if kind == "paged":  # the new rows are the context's last: contexts hold them
        return [(case["lq"], n, case["causal"], n - case["lq"]) for n in _kv_lens(case)]
    if kind == "decode_paged":
        m = case["m"]
        return [(max(m, 1), n, m > 0, n - max(m, 1)) for n in _kv_lens(case)]
    return [(1, case["lk"], False, 0)] * case["b"]  # decode_dense


def work(case):
    es, d = _BYTES[case["dtype"]], case["d"]
    if case["kind"] == "append":  # the new rows of K and V, read once and written once
        return {"bytes": 4 * sum(_kv_lens(case)) * case["hkv"] * d * es, "flops": 0}
    rows = keys = pairs = 0
    for lq, lk, causal, off in _sequences(case):
        rows += lq
        keys += lk
        pairs += _pairs(lq, lk, causal, off)
    return {"bytes": es * d * (2 * rows * case["hq"] + 2 * keys * case["hkv"]),
            "flops": 4 * d * case["hq"] * pairs}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _randn(g, shape, dtype):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32).to(dtype)


def _indptr(lens):
    return torch.tensor([0] + lens).cumsum(0).to(torch.int32).cuda()


def _tables(lens, seed, shuffled=True):
    """Block tables for K and V over a pool with some spare pages: two
    independent page orders, rows padded with -1."""
    pages = [-(-n // PAGE) for n in lens]
    pool = sum(pages) + 64
    g = torch.Generator().manual_seed(seed)
    out = []
    for _ in range(2):
        order = torch.randperm(pool, generator=g) if shuffled else torch.arange(pool)
        t = torch.full((len(lens), max(pages)), -1, dtype=torch.int32)
        at = 0
        for b, p in enumerate(pages):
            t[b, :p] = order[at:at + p].to(torch.int32)
            at += p
        out.append(t.cuda())
    return pool, out[0], out[1]


def prepare(case, seed):
    kind, dt, d = case["kind"], _DTYPES[case["dtype"]], case["d"]
    g = _gen(seed)
    hkv = case["hkv"]
    if kind == "dense":
        q = _randn(g, (case["b"], case["hq"], case["lq"], d), dt)
        k = _randn(g, (case["b"], hkv, case["lk"], d), dt)
        v = _randn(g, (case["b"], hkv, case["lk"], d), dt)
        return dict(case=case, fn=flash_attention_v2, args=(q, k, v),
                    kw=dict(is_causal=case["causal"]))
    if kind == "ragged":
        ql, kl = _q_lens(case), _kv_lens(case)
        q = _randn(g, (sum(ql), case["hq"], d), dt)
        k = _randn(g, (sum(kl), hkv, d), dt)
        v = _randn(g, (sum(kl), hkv, d), dt)
        return dict(case=case, fn=flash_attention_v2, args=(q, k, v),
                    kw=dict(is_causal=case["causal"], q_indptr=_indptr(ql), kv_indptr=_indptr(kl)))
    if kind == "decode_dense":
        q = _randn(g, (case["b"], case["hq"], d), dt)
        k = _randn(g, (case["b"], hkv, case["lk"], d), dt)
        v = _randn(g, (case["b"], hkv, case["lk"], d), dt)
        return dict(case=case, fn=decode_attention, args=(q, k, v), kw={})
    lens = _kv_lens(case)
    pool, kt, vt = _tables(lens, seed)
    if kind == "append":
        kc = _randn(g, (pool * PAGE, hkv, d), dt)
        vc = _randn(g, (pool * PAGE, hkv, d), dt)
        kn = _randn(g, (sum(lens), hkv, d), dt)
        vn = _randn(g, (sum(lens), hkv, d), dt)
        return dict(case=case, fn=paged_kv_append,
                    args=(kc, vc, kt, vt, kn, vn, _indptr(lens), PAGE),
                    kw=dict(start_pos=torch.zeros(len(lens), dtype=torch.int32, device="cuda")))
    k = _randn(g, (pool * PAGE, hkv, d), dt)
    v = _randn(g, (pool * PAGE, hkv, d), dt)
    kw = dict(kv_indptr=torch.tensor(lens, dtype=torch.int32, device="cuda"), k_block_table=kt,
              v_block_table=vt, kv_page_size=PAGE)
    if kind == "paged":
        q = _randn(g, (case["n"], case["hq"], case["lq"], d), dt)
        return dict(case=case, fn=flash_attention_v2, args=(q, k, v),
                    kw=dict(is_causal=case["causal"], causal_alignment="bottom_right", **kw))
    if case["m"] == 0:
        q = _randn(g, (case["n"], case["hq"], d), dt)
        return dict(case=case, fn=decode_attention, args=(q, k, v), kw=kw)
    q = _randn(g, (case["n"], case["hq"], case["m"], d), dt)
    return dict(case=case, fn=speculative_decode_attention, args=(q, k, v),
                kw=dict(causal=True, **kw))


def run(state):
    out = state["fn"](*state["args"], **state["kw"])
    if state["case"]["kind"] == "append":  # in place: the caches
        return state["args"][0], state["args"][1]
    return out


# ---------------------------------------------------------------------------
# what the results are held to
# ---------------------------------------------------------------------------

def tolerance(case):
    """Measured on MI355X against ``exact`` over the listed cases and drawn
    ones, times about four.  bf16: output and softmax weights rounded to 8
    bits; fp16: to 11 bits; fp32 prefill: operands and weights rounded to
    fp16; fp32 decode: fp32 throughout."""
    if case["kind"] == "append":
        return "exact"
    if case["dtype"] == "bf16":
        return {"rel": 1e-2}
    if case["dtype"] == "f16":
        return {"rel": 1.2e-3}
    return {"rel": 1.5e-3} if case["kind"] == "dense" else {"rel": 3e-6}


def _attend(q, k, v, causal, off, d):
    """Attention of [H, M, D] rows over [N, D] keys of one kv head in 64 bits,
    in blocks of rows (key j visible to row i iff j <= i + off)."""
    h, m, _ = q.shape
    n = k.shape[0]
    q, k, v = q.double(), k.double(), v.double()
    kt = k.t().contiguous()
    out = torch.empty((h, m, d), dtype=torch.float64, device=q.device)
    step = max(1, min(m, (1 << 26) // max(h * n, 1)))
    for r0 in range(0, m, step):
        r1 = min(r0 + step, m)
        s = (q[:, r0:r1].reshape(-1, d) @ kt) * d ** -0.5
        if causal:
            rows = torch.arange(r0, r1, device=q.device).repeat(h)
            hide = torch.arange(n, device=q.device)[None, :] > (rows + off)[:, None]
            s = s.masked_fill(hide, float("-inf"))
        out[:, r0:r1] = (torch.softmax(s, dim=-1) @ v).view(h, r1 - r0, d)
    return out


def exact(case, seed):
    if case["kind"] == "append":
        return None
    st = prepare(case, seed)
    q, k, v = st["args"]
    kind, d, hkv = case["kind"], case["d"], case["hkv"]
    grp = case["hq"] // hkv
    seqs = _sequences(case)
    if kind in ("decode_dense", "decode_paged") and q.dim() == 3:
        q = q.unsqueeze(2)
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    qa = ka = 0
    for b, (lq, lk, causal, off) in enumerate(seqs):
        if kind in ("dense", "decode_dense"):
            qb, kb, vb = q[b], k[b].transpose(0, 1), v[b].transpose(0, 1)
        elif kind == "ragged":
            qb = q[qa:qa + lq].transpose(0, 1)
            kb, vb = k[ka:ka + lk], v[ka:ka + lk]
        else:
            qb = q[b]
            at = torch.arange(lk, device=q.device)
            kb, vb = (c[t[b].long()[at // PAGE] * PAGE + at % PAGE]
                      for c, t in ((k, st["kw"]["k_block_table"]), (v, st["kw"]["v_block_table"])))
        for h in range(hkv):
            o = _attend(qb[h * grp:(h + 1) * grp], kb[:, h], vb[:, h], causal, off, d)
            if kind == "ragged":
                out[qa:qa + lq, h * grp:(h + 1) * grp] = o.transpose(0, 1)
            else:
                out[b, h * grp:(h + 1) * grp] = o
        qa += lq
        ka += lk
    if st["args"][0].dim() == 3 and kind != "ragged":
        out = out.squeeze(2)
    return out
