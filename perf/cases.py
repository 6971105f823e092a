"""The measured cases: what a serving program has this package do, through the package's own operators.

A decode step of one layer is three calls -- the fused prolog, the indexer, the attention -- and a prefill chunk is
the prolog and the attention.  The cases are those calls over the range of batches, query tokens per sequence, lengths,
head counts and cache formats in which they are used; the sizes of the model (7168 hidden channels, query rank 1536,
128 attention heads of 512 + 64, 64 indexer heads of 128, top-k 2048, pages of 128 positions) are the ones the
repository's tests and benchmark use.
"""
from __future__ import annotations

import math
import random

import torch

import pypto_amd

DEVICE = "cuda"
PAGE = 128
DN, DR = 512, 64                       # latent and rope widths of a cache row
HIDDEN, RANK, HEADS, IDX_HEADS, IDX_DIM = 7168, 1536, 128, 64, 128
TOPK = 2048
BF = torch.bfloat16


# ---------------------------------------------------------------- the cases

def listed():
    return [
        # one layer's decode step of a small interactive batch with multi-token prediction: prolog, indexer, attention
        dict(name="step_4x2", kind="step", b=4, s1=2, kv_lo=8192, kv_hi=65536),
        # a single user's decode step: latency of one query row
        dict(name="attn_decode_1", kind="attn", b=1, s1=1, heads=HEADS, topk=TOPK, kv_lo=3001, kv_hi=3001, cache="int8"),
        # the benchmark's decode batch
        dict(name="attn_decode_32", kind="attn", b=32, s1=1, heads=HEADS, topk=TOPK, kv_lo=8192, kv_hi=65536, cache="int8"),
        # two query tokens for each of 64 sequences
        dict(name="attn_mtp_64x2", kind="attn", b=64, s1=2, heads=HEADS, topk=TOPK, kv_lo=4096, kv_hi=32768, cache="int8"),
        # a prefill chunk of one sequence
        dict(name="attn_prefill_4096", kind="prefill", s1=4096, kv=4096),
        # the packed cache, young and ragged sequences (many rows have fewer keys than topk), three query tokens
        dict(name="attn_packed_11x3", kind="attn", b=11, s1=3, heads=HEADS, topk=TOPK, kv_lo=190, kv_hi=6000, cache="packed"),
        # a bf16 cache with the heads divided over two GPUs
        dict(name="attn_bf16_40_64h", kind="attn", b=40, s1=1, heads=64, topk=TOPK, kv_lo=1024, kv_hi=16384, cache="bf16"),
        # the indexer alone: few long sequences, the benchmark's batch, two query tokens per sequence with fp16 scales
        dict(name="indexer_4", kind="indexer", b=4, s1=1, kv_lo=32768, kv_hi=32768, dtype="fp32"),
        dict(name="indexer_32", kind="indexer", b=32, s1=1, kv_lo=8192, kv_hi=65536, dtype="fp32"),
        dict(name="indexer_mtp_64x2", kind="indexer", b=64, s1=2, kv_lo=4096, kv_hi=32768, dtype="fp16"),
        # both prologs: a decode batch and a ragged prefill chunk
        dict(name="prolog_decode_32", kind="prolog", b=32, s1=1),
        dict(name="prolog_prefill_1000", kind="prolog", b=1, s1=1000),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _span(rng, lo, hi):
    """A range of sequence lengths inside [lo, hi]."""
    a, b = _log(rng, lo, hi), _log(rng, lo, hi)
    return min(a, b), max(a, b)


def draw(rng):
    kind = rng.choice(("step", "attn", "attn", "attn", "prefill", "indexer", "indexer", "prolog", "prolog"))
    if kind == "step":
        s1 = rng.randint(1, 2)
        b = rng.randint(1, 8 // s1)
        lo, hi = _span(rng, 500, 65536)
        return dict(kind=kind, b=b, s1=s1, kv_lo=lo, kv_hi=hi)
    if kind == "attn":
        s1 = rng.choice((1, 1, 2, 3, 4))
        b = _log(rng, 1, 128)
        lo, hi = _span(rng, 100, min(65536, 2_400_000 // b))
        return dict(kind=kind, b=b, s1=s1, heads=rng.choice((128, 128, 128, 64, 32, 16)), topk=rng.choice((TOPK, TOPK, TOPK, 1024)),
                    kv_lo=lo, kv_hi=hi, cache=rng.choice(("int8", "int8", "packed", "bf16")))
    if kind == "prefill":
        s1 = _log(rng, 200, 3000)
        return dict(kind=kind, s1=s1, kv=s1 + rng.choice((0, _log(rng, 100, 9000))))
    if kind == "indexer":
        s1 = rng.choice((1, 1, 2, 3, 4))
        b = _log(rng, 1, 128)
        lo, hi = _span(rng, 500, min(131072, 2_400_000 // b))
        return dict(kind=kind, b=b, s1=s1, kv_lo=lo, kv_hi=hi, dtype=rng.choice(("fp16", "fp32")))
    if rng.random() < 0.5:
        return dict(kind="prolog", b=_log(rng, 1, 64), s1=rng.randint(1, 2))
    return dict(kind="prolog", b=1, s1=_log(rng, 130, 4096))


# ---------------------------------------------------------------- inputs

def _lengths(case):
    """Sequence lengths of a case: part of its shape, so the same for every seed."""
    if case["kind"] == "prefill":
        return [case["kv"]]
    r = random.Random(7 * case["b"] + case["kv_lo"])
    return [max(case["s1"], r.randint(case["kv_lo"], case["kv_hi"])) for _ in range(case["b"])]


def _keys(case):
    """Selected keys of every query row."""
    s1, topk = case["s1"], case.get("topk", TOPK)
    return [min(max(n - s1 + 1 + i, 0), topk) for n in _lengths(case) for i in range(s1)]


class _Maker:
    """Tensors from one seed, made on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEVICE).manual_seed(seed)

    def normal(self, shape, std=1.0, dtype=BF):
        out = torch.empty(shape, device=DEVICE, dtype=dtype)
        return out.normal_(0.0, std, generator=self.g)

    def uniform(self, shape, lo, hi, dtype=torch.float32):
        return torch.empty(shape, device=DEVICE, dtype=torch.float32).uniform_(lo, hi, generator=self.g).to(dtype)

    def int8(self, shape):
        return torch.randint(-127, 128, shape, device=DEVICE, dtype=torch.int8, generator=self.g)

    def pages(self, lengths):
        """(number of pages, block table with -1 in unused slots): the pages of the sequences lie in random order."""
        per = [-(-n // PAGE) for n in lengths]
        order = torch.randperm(sum(per), device=DEVICE, generator=self.g).to(torch.int32)
        table = torch.full((len(lengths), max(per)), -1, device=DEVICE, dtype=torch.int32)
        at = 0
        for i, n in enumerate(per):
            table[i, :n] = order[at:at + n]
            at += n
        return sum(per), table

    def selection(self, lengths, s1, topk):
        """Top-k rows as the indexer leaves them: a random choice of the positions a query token sees, in no order, or
        all of them where they are no more than topk; -1 after the last one."""
        rows = []
        pos = torch.arange(max(max(lengths), topk), device=DEVICE)
        for n in lengths:
            sees = torch.arange(n - s1 + 1, n + 1, device=DEVICE).clamp_(min=0)[:, None]
            key = torch.empty((s1, pos.numel()), device=DEVICE).uniform_(generator=self.g)
            key = torch.where(sees > topk, key, -pos.float()).masked_fill_(pos >= sees, -math.inf)
            got = key.topk(topk, dim=1).indices.to(torch.int32)
            rows.append(got.masked_fill_(torch.arange(topk, device=DEVICE) >= sees, -1))
        return torch.cat(rows)


def _slots(table, lengths, s1):
    """Cache rows of the newest s1 positions of every sequence."""
    pos = torch.tensor([[n - s1 + i for i in range(s1)] for n in lengths], device=DEVICE)
    page = table.to(torch.int64).gather(1, pos // PAGE)
    return (page * PAGE + pos % PAGE).reshape(-1)


def _cache(m, rows, fmt):
    """The latent cache as the attention takes it: (nope, rope, scales), or one packed array."""
    rope = m.normal([rows, DR])
    if fmt == "bf16":
        return m.normal([rows, DN]), rope, None
    nope, scales = m.int8([rows, DN]), m.uniform([rows, 4], 0.005, 0.02)
    if fmt == "int8":
        return nope, rope, scales
    packed = torch.cat([nope, rope.view(torch.int8), scales.view(torch.int8)], dim=1)
    return packed.contiguous(), None, None


def _hadamard():
    h = torch.ones([1, 1], device=DEVICE)
    while h.shape[0] < IDX_DIM:
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return (h * IDX_DIM ** -0.5).to(BF)


def _prolog(m, lengths, s1, pages, table):
    """Arguments of the fused prolog: hidden states, both halves' weights, the caches and the outputs."""
    t = len(lengths) * s1
    angle = m.uniform([t, DR], 0.0, 2 * math.pi)
    mla = [m.normal([t, HIDDEN]), m.normal([HIDDEN, RANK], HIDDEN ** -0.5), m.int8([RANK, HEADS * (128 + DR)]),
           m.uniform([HEADS * (128 + DR), 1], 0.5, 1.5).mul_(RANK ** -0.5 / 73), m.normal([HEADS, 128, DN], 128 ** -0.5),
           m.normal([HIDDEN, DN + DR], HIDDEN ** -0.5), m.uniform([RANK], 0.5, 1.5, BF), m.uniform([DN], 0.5, 1.5, BF),
           angle.cos().to(BF), angle.sin().to(BF), _slots(table, lengths, s1)]
    nope, rope, scales = _cache(m, pages * PAGE, "int8")
    kv = [nope.view(pages, PAGE, 1, DN), rope.view(pages, PAGE, 1, DR), scales.view(pages, PAGE, 1, 4)]
    idx = [m.int8([RANK, IDX_HEADS * IDX_DIM]), m.uniform([IDX_HEADS * IDX_DIM, 1], 0.5, 1.5).mul_(RANK ** -0.5 / 73),
           m.normal([HIDDEN, IDX_DIM], HIDDEN ** -0.5), m.normal([HIDDEN, IDX_HEADS], HIDDEN ** -0.5),
           m.uniform([IDX_DIM], 0.5, 1.5, BF), m.normal([IDX_DIM], 0.1), _hadamard(), _hadamard()]
    key = [m.int8([pages, PAGE, 1, IDX_DIM]), m.uniform([pages, PAGE, 1, 1], 0.005, 0.02, torch.float16)]
    new = lambda shape, dtype: torch.zeros(shape, device=DEVICE, dtype=dtype)  # noqa: E731
    query = [new([t, HEADS, DN], BF), new([t, HEADS, DR], BF)]
    iout = [new([t, IDX_HEADS, IDX_DIM], torch.int8), new([t, IDX_HEADS, 1], torch.float16)]
    weights = new([t, IDX_HEADS], torch.float16)
    args = mla + kv + idx + key + query + kv + iout + key + [weights, 1e-6, 1e-6, "PA_BSND", None,
                                                             pypto_amd.IndexerPrologQuantAttr(eps=1e-6),
                                                             pypto_amd.IndexerPrologQuantConfigs(), None]
    outs = dict(query_nope=query[0], query_rope=query[1], q_int8=iout[0], q_scale=iout[1], weights=weights, kv_cache=kv[0],
                kr_cache=kv[1], k_scale_cache=kv[2], k_cache=key[0], k_cache_scale=key[1])
    return args, outs


def prepare(case, seed):
    m, kind = _Maker(seed), case["kind"]
    if kind == "prolog":
        lengths = [case["s1"] + 24] * case["b"]
        args, outs = _prolog(m, lengths, case["s1"], *m.pages(lengths))
        return dict(kind=kind, args=args, outs=outs, decode=case["s1"] <= 4)
    lengths, s1 = _lengths(case), case["s1"]
    pages, table = m.pages(lengths)
    act = torch.tensor(lengths, device=DEVICE, dtype=torch.int32)
    t = len(lengths) * s1
    if kind == "indexer":
        dt, wt = (torch.float16, torch.float16) if case["dtype"] == "fp16" else (torch.float32, BF)
        res = torch.zeros([t, 1, TOPK], device=DEVICE, dtype=torch.int32)
        args = [m.int8([t, IDX_HEADS, IDX_DIM]), m.uniform([t, IDX_HEADS], 0.005, 0.02, dt), m.int8([pages, PAGE, 1, IDX_DIM]),
                m.uniform([pages, PAGE, 1], 0.005, 0.02, dt), m.normal([t, IDX_HEADS], 0.125, wt), act, table, res]
        return dict(kind=kind, args=args, res=res)
    scale = (DN + DR) ** -0.5
    if kind == "step":
        args, outs = _prolog(m, lengths, s1, pages, table)
        topk = torch.zeros([t, 1, TOPK], device=DEVICE, dtype=torch.int32)
        out = torch.zeros([case["b"], s1, HEADS, DN], device=DEVICE, dtype=BF)
        index = [outs["q_int8"], outs["q_scale"].view(t, IDX_HEADS), outs["k_cache"], outs["k_cache_scale"].view(pages, PAGE, 1),
                 outs["weights"], act, table, topk]
        attn = [outs["query_nope"].view(t * HEADS, DN), outs["query_rope"].view(t * HEADS, DR), outs["kv_cache"].view(-1, DN),
                outs["kr_cache"].view(-1, DR), outs["k_scale_cache"].view(-1, 4), topk.view(t, TOPK), table, act, out, HEADS, 1,
                scale, TOPK, PAGE, table.shape[1]]
        return dict(kind=kind, prolog=args, index=index, attn=attn, outs=dict(outs, topk=topk, out=out))
    heads, topk = case.get("heads", HEADS), case.get("topk", TOPK)
    nope, rope, scales = _cache(m, pages * PAGE, case.get("cache", "int8"))
    out = torch.zeros([len(lengths), s1, heads, DN], device=DEVICE, dtype=BF)
    query = [m.normal([t * heads, DN]), m.normal([t * heads, DR])]
    tail = [m.selection(lengths, s1, topk), table, act, out, heads, 1, scale, topk, PAGE, table.shape[1]]
    packed = case.get("cache") == "packed"
    return dict(kind=kind, packed=packed, args=query + ([nope] if packed else [nope, rope, scales]) + tail, out=out)


def run(state):
    kind = state["kind"]
    if kind == "attn":
        op = pypto_amd.sparse_attention_antiquant_d if state["packed"] else pypto_amd.sparse_flash_attention_quant_d
        op(*state["args"])
        return state["out"]
    if kind == "prefill":
        pypto_amd.sparse_flash_attention_quant_p(*state["args"])
        return state["out"]
    if kind == "indexer":
        pypto_amd.lightning_indexer_decode(*state["args"])
        return state["res"]
    if kind == "prolog":
        op = pypto_amd.mla_indexer_prolog_quant_d if state["decode"] else pypto_amd.mla_indexer_prolog_quant_p
        op(*state["args"])
        return state["outs"]
    pypto_amd.mla_indexer_prolog_quant_d(*state["prolog"])
    pypto_amd.lightning_indexer_decode(*state["index"])
    pypto_amd.sparse_flash_attention_quant_d(*state["attn"])
    return state["outs"]


# ---------------------------------------------------------------- what a pass cannot do without

def _attn_work(case):
    heads, s1 = case.get("heads", HEADS), case["s1"]
    keys, lengths = _keys(case), _lengths(case)
    row = 2 * (DN + DR) if case.get("cache") == "bf16" else DN + 2 * DR + 16
    # every selected cache row once per sequence
    rows = sum(min(n, sum(keys[i * s1:(i + 1) * s1])) for i, n in enumerate(lengths))
    t = len(keys)
    return dict(bytes=rows * row + 4 * sum(keys) + 2 * t * heads * (DN + DR + DN), flops=2 * heads * sum(keys) * (2 * DN + DR))


def _indexer_work(case):
    lengths, t = _lengths(case), case["b"] * case["s1"]
    size = 4 if case.get("dtype") == "fp32" else 2
    return dict(bytes=sum(lengths) * (IDX_DIM + size) + t * IDX_HEADS * (IDX_DIM + size + 2) + 4 * t * TOPK,
                flops=2 * IDX_HEADS * IDX_DIM * case["s1"] * sum(lengths))


def _prolog_work(t):
    q, iq = HEADS * (128 + DR), IDX_HEADS * IDX_DIM
    weights = (2 * HIDDEN * (RANK + DN + DR + IDX_DIM + IDX_HEADS) + RANK * (q + iq) + 4 * (q + iq) + 2 * HEADS * 128 * DN
               + 4 * IDX_DIM * IDX_DIM + 2 * (RANK + DN + 2 * IDX_DIM))
    token = (2 * HIDDEN + 4 * DR + 8 + 2 * HEADS * (DN + DR) + iq + 4 * IDX_HEADS + DN + 2 * DR + 16 + IDX_DIM + 2)
    flops = 2 * t * (HIDDEN * (RANK + DN + DR + IDX_DIM + IDX_HEADS) + RANK * (q + iq) + HEADS * 128 * DN
                     + (IDX_HEADS + 1) * IDX_DIM * IDX_DIM)
    return dict(bytes=weights + t * token, flops=flops)


def work(case):
    kind = case["kind"]
    if kind == "indexer":
        return _indexer_work(case)
    if kind == "prolog":
        return _prolog_work(case["b"] * case["s1"])
    if kind == "step":
        parts = _prolog_work(case["b"] * case["s1"]), _indexer_work(case), _attn_work(case)
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    return _attn_work(case)


def tolerance(case):
    kind = case["kind"]
    if kind == "indexer":
        return "exact"                                   # selected positions
    if kind in ("attn", "prefill"):
        return {"rel": 1e-2, "max": 5e-2}                # bf16 results, bf16 probabilities
    if case["b"] * case["s1"] <= 8:
        return {"rel": 1e-2, "max": 5e-2}                # whole numbers exact; the bf16 queries are sums in any order
    # from nine tokens on the sums over the hidden axis are in any order: an int8 value lies one step off now and then
    return {"rel": 1e-2, "max": 1e-1, "differ": 5e-3}
