"""Parity of the HIP lightning indexer (through the operator, pybind11 and the C ABI) against the CPU
oracle.  The bar is bit-exact indices."""
import numpy as np
import pytest
import torch

import pypto_amd
from pypto_amd.synthetic import gen_indexer_inputs

pytestmark = pytest.mark.gpu


def run_op(inp):
    dev = torch.device("cuda:0")
    d = inp.to(dev)
    d.topk_res.fill_(-7)
    ts = [pypto_amd.from_torch(t) for t in d.operator_tensors()]
    ret = pypto_amd.lightning_indexer_decode(*ts, [128, 64, 32, 16, 8, 4, 1], pypto_amd.LightningIndexerConfigs(),
                                             inp.selected_count)
    assert ret is None
    torch.cuda.synchronize()
    return d.topk_res.cpu()


def oracle(inp, c_oracle):
    return c_oracle.li_decode(inp.idx_query, inp.idx_query_scale, inp.idx_key_cache, inp.idx_key_scale,
                              inp.idx_weight, inp.act_seq_key, inp.block_table, inp.selected_count)


def assert_exact(got, ref, what):
    if not torch.equal(got, ref):
        bad = (got != ref).reshape(got.shape[0], -1)
        rows = torch.nonzero(bad.any(dim=1)).reshape(-1).tolist()
        r = rows[0]
        cols = torch.nonzero(bad[r]).reshape(-1)[:8].tolist()
        raise AssertionError(f"{what}: {int(bad.sum())} index mismatches in rows {rows[:8]}; row {r} cols {cols}: "
                             f"got {got[r, 0, cols].tolist()} want {ref[r, 0, cols].tolist()}")


@pytest.mark.parametrize("variant", ["fp16", "fp32"])
@pytest.mark.parametrize("b,s1,act,k", [
    (2, 1, [4096, 3000], 2048),        # above the select threshold, one ragged
    (3, 2, [300, 129, 5], 64),         # two query tokens per sequence, causal effective lengths
    (2, 1, [2048, 2049], 2048),        # exactly k and k+1 candidates
    (2, 1, [100, 1], 2048),            # fewer candidates than k: padded with -1
    (1, 4, [9000], 2048),              # s1 = 4
    (1, 1, [33], 16),                  # partial 32-key block
    # the two shapes of the reference's own system tests
    # (framework/tests/st/operator/src/test_deepseek_v3.2_exp/gen_lightning_indexer.py:374-376, 428-430)
    (4, 1, [768, 4097, 8192, 131071], 2048),
    (4, 2, [65536] * 4, 2048),
])
def test_indexer_bit_exact(c_oracle, variant, b, s1, act, k):
    inp = gen_indexer_inputs(b, s1, act, selected_count=k, seed=7 * b + s1 + k, variant=variant)
    assert_exact(run_op(inp), oracle(inp, c_oracle), f"{variant} b={b} s1={s1} act={act} k={k}")


def test_engineered_ties_and_zero_scores(c_oracle):
    """Many equal scores: zero weights make every score +-0, duplicated key rows make exact ties."""
    inp = gen_indexer_inputs(2, 1, [5000, 6000], selected_count=2048, seed=31, variant="fp16")
    inp.idx_weight[0] = 0                                # token 0: all scores are zero -> positions 0..2047
    kc = inp.idx_key_cache.reshape(-1, 128)
    ks = inp.idx_key_scale.reshape(-1)
    # token 1: every logical position p >= 3000 repeats the row of position p - 3000
    pos = torch.arange(6000)
    phys = inp.block_table[1].long()[pos // 128] * 128 + pos % 128
    kc[phys[3000:]] = kc[phys[:3000]]
    ks[phys[3000:]] = ks[phys[:3000]]
    got = run_op(inp)
    ref = oracle(inp, c_oracle)
    assert ref[0, 0].tolist() == list(range(2048))
    assert_exact(got, ref, "ties")


def test_negative_weights_and_mixed_signs(c_oracle):
    inp = gen_indexer_inputs(1, 1, [7000], selected_count=2048, seed=41, variant="fp32")
    inp.idx_weight[:] = -inp.idx_weight.abs()            # all scores <= 0: the best are the zeros
    assert_exact(run_op(inp), oracle(inp, c_oracle), "negative")


def test_config1_full_size(c_oracle):
    """B=4, KV 32768 each, shuffled block table, top-2048."""
    for variant in ("fp16", "fp32"):
        inp = gen_indexer_inputs(4, 1, [32768] * 4, selected_count=2048, seed=1, variant=variant)
        assert_exact(run_op(inp), oracle(inp, c_oracle), f"cfg1 {variant}")


def test_bf16_key_scales(c_oracle):
    """Key scales in bf16 (two per staged dword, either half), fp16 query scales, bf16 weights."""
    inp = gen_indexer_inputs(2, 2, [4500, 2600], selected_count=2048, seed=51, variant="fp32")
    inp.idx_key_scale = inp.idx_key_scale.to(torch.bfloat16)
    inp.idx_query_scale = inp.idx_query_scale.to(torch.float16)
    assert_exact(run_op(inp), oracle(inp, c_oracle), "bf16 key scales")


def test_long_runs_wide_block_table(c_oracle):
    """64 query tokens over a block table 1024 pages wide: the launch then gives every wave the longest
    run of keys it supports, the lengths end inside runs, pairs and 32-key blocks, and the longest
    sequence is the maximum the operator accepts (131072)."""
    from pypto_amd.synthetic import gen_block_table
    g = torch.Generator().manual_seed(61)
    act = [131072, 65536 + 17, 40000, 2049, 2048, 2047, 4096 + 33, 1] + \
          [int(x) for x in torch.randint(1, 3000, [56], generator=g)]
    block_num, table = gen_block_table(act, 128, g, shuffle=True, max_kv=131072)
    inp = gen_indexer_inputs(len(act), 1, act, selected_count=2048, seed=62, variant="fp32", block_table=table,
                             block_num=block_num)
    assert_exact(run_op(inp), oracle(inp, c_oracle), "wide block table")


def score_launch(b, s1, width):
    """(query tokens per unit, whether the runs are spread over all sequences) of the score kernel's launch over a block table of
    `width` positions: the rule of pto_li_decode_launch."""
    from pypto_amd import _C
    waves = torch.cuda.get_device_properties(0).multi_processor_count * _C.LI_SCORE_WAVES
    pairs = s1 % 2 == 0 and b * (s1 // 2) * ((width + 63) // 64) >= _C.LI_PAIR_MIN * waves
    units = b * s1 // (2 if pairs else 1)
    return 2 if pairs else 1, b <= _C.LI_MAX_BALANCED_SEQS and units <= _C.LI_MAX_BALANCED_UNITS


def wide_inputs(b, s1, act, width, variant, k=2048, seed=0):
    """Inputs whose block table has `width` positions, however short the sequences are."""
    from pypto_amd.synthetic import gen_block_table
    num, table = gen_block_table(act, 128, torch.Generator().manual_seed(seed), max_kv=width)
    return gen_indexer_inputs(b, s1, act, selected_count=k, seed=seed + 1, variant=variant, block_table=table, block_num=num)


@pytest.mark.parametrize("b,s1,balanced", [
    (100, 1, True),     # runs spread over all sequences, rows 1.. of the table of sequences (64 and up)
    (40, 4, True),      # the same with four query tokens per sequence
    (130, 4, True),     # 520 query tokens
    (515, 1, False),    # more sequences than the table holds: runs of a fixed length
    (515, 3, False),
])
def test_many_query_tokens_short_sequences(c_oracle, b, s1, balanced):
    """More sequences than one row of the score kernel's table holds, and more than the whole table; short ragged sequences so
    the oracle stays cheap."""
    g = torch.Generator().manual_seed(1000 + b)
    act = [int(x) for x in torch.randint(s1, 700, [b], generator=g)]
    act[0], act[-1] = 699, s1                      # a long first and the shortest possible last sequence
    inp = gen_indexer_inputs(b, s1, act, selected_count=128, seed=b + s1, variant="fp16")
    assert score_launch(b, s1, inp.block_table.shape[1] * 128) == (1, balanced)
    assert_exact(run_op(inp), oracle(inp, c_oracle), f"b={b} s1={s1}")


@pytest.mark.parametrize("variant,b,s1,width,tokens", [
    ("fp32", 28, 3, 0, 1), ("fp16", 28, 4, 0, 1),                      # an odd number of tokens, and too few keys: units of one token
    ("fp32", 28, 4, 28160, 2), ("fp16", 28, 4, 28160, 2), ("fp16", 30, 2, 56320, 2)])
def test_token_pairs_share_a_key_pass(c_oracle, variant, b, s1, width, tokens):
    """Two query tokens of a sequence per key pass (the reference scores all s1 tokens against a page at once,
    lightning_indexer_quant_impl.py:163-169) where the block table has room for enough keys: s1 = 4 makes two units per
    sequence; ragged lengths end inside runs and pairs."""
    g = torch.Generator().manual_seed(300 + b)
    act = [int(x) for x in torch.randint(2100, 20480, [b], generator=g)]
    act[0], act[1] = 20480, 2049
    inp = wide_inputs(b, s1, act, max(width, 20480), variant, seed=b * s1)
    assert score_launch(b, s1, inp.block_table.shape[1] * 128) == (tokens, True)
    assert_exact(run_op(inp), oracle(inp, c_oracle), f"{variant} b={b} s1={s1}")


@pytest.mark.parametrize("variant,b,s1,width", [("fp16", 28, 3, 0), ("fp16", 2, 1, 0), ("fp32", 2, 1, 0), ("fp16", 28, 4, 28160), ("fp32", 28, 4, 28160)])
def test_largest_dot_products(c_oracle, variant, b, s1, width):
    """Queries and keys of -128 and 127 only, with runs of one value: dot products up to +-2^21, both ends of the range in which
    the accumulators' bits are read as floats; with fp16 scales and weights the fused head sum; units of one token and of two."""
    g = torch.Generator().manual_seed(b)
    act = [int(x) for x in torch.randint(2100, 20480, [b], generator=g)]
    act[0] = 20480
    inp = wide_inputs(b, s1, act, max(width, 20480), variant, seed=5 + b)
    assert score_launch(b, s1, inp.block_table.shape[1] * 128)[0] == (2 if width else 1)
    inp.idx_query = torch.where(inp.idx_query < 0, -128, 127).to(torch.int8)
    inp.idx_key_cache = torch.where(inp.idx_key_cache < 0, -128, 127).to(torch.int8)
    inp.idx_query[:, ::3] = -128
    inp.idx_query[:, 1::3] = 127
    inp.idx_key_cache[:, ::7] = -128
    inp.idx_key_cache[:, 1::7] = 127
    assert_exact(run_op(inp), oracle(inp, c_oracle), f"{variant} b={b} s1={s1} extremes")


@pytest.mark.parametrize("variant,b,s1,width,tokens,balanced", [
    ("fp16", 260, 4, 2304, 1, True), ("fp32", 260, 3, 2304, 1, True), ("fp16", 260, 4, 3072, 2, True),
    ("fp16", 516, 4, 2304, 2, False), ("fp32", 516, 2, 3328, 2, False), ("fp16", 515, 2, 3328, 2, False)])
def test_token_pairs_beyond_the_balanced_mapping(c_oracle, variant, b, s1, width, tokens, balanced):
    """Token pairs per key pass among hundreds of sequences, with runs spread over all of them and, beyond 512, of a fixed length --
    past the far end of the operator's documented decode range (b up to 128 with s1 up to 4 and long KV,
    examples/models/deepseek_v32_exp/README.md:6-24)."""
    g = torch.Generator().manual_seed(500 + s1)
    act = [int(x) for x in torch.randint(s1, 2300, [b], generator=g)]
    act[0], act[1], act[-1] = 2300, 2049, s1
    inp = wide_inputs(b, s1, act, width, variant, seed=b + s1)
    assert score_launch(b, s1, inp.block_table.shape[1] * 128) == (tokens, balanced)
    assert_exact(run_op(inp), oracle(inp, c_oracle), f"{variant} b={b} s1={s1}")


def test_small_pages_and_small_k(c_oracle):
    """32-key pages (every block of a pair on its own page) and small selection counts."""
    for k, act in ((1, [5000, 70]), (17, [2500, 31]), (512, [700, 513])):
        inp = gen_indexer_inputs(2, 1, act, selected_count=k, seed=70 + k, variant="fp16", block_size=32)
        assert_exact(run_op(inp), oracle(inp, c_oracle), f"bs=32 k={k}")


def test_select_falls_back_on_degenerate_rows(c_oracle):
    """Rows the sampled pivot cannot split: a constant row with one spike (every sampled score equal),
    and two-valued scores where far more than the list holds tie above the pivot."""
    inp = gen_indexer_inputs(2, 1, [40000, 30000], selected_count=2048, seed=81, variant="fp32")
    kc = inp.idx_key_cache.reshape(-1, 128)
    ks = inp.idx_key_scale.reshape(-1)
    pos0 = torch.arange(40000)
    phys0 = inp.block_table[0].long()[pos0 // 128] * 128 + pos0 % 128
    kc[phys0] = kc[phys0[0]].clone()              # token 0: every key equal ...
    ks[phys0] = ks[phys0[0]].clone()
    ks[phys0[12345]] = ks[phys0[0]].clone() * 4   # ... except one, four times the score
    pos1 = torch.arange(30000)
    phys1 = inp.block_table[1].long()[pos1 // 128] * 128 + pos1 % 128
    kc[phys1] = kc[phys1[0]].clone()              # token 1: two score values, 3/4 of the keys on the larger
    ks[phys1] = ks[phys1[0]].clone()
    ks[phys1[pos1 % 4 == 1]] = ks[phys1[0]].clone() * 0.5
    assert_exact(run_op(inp), oracle(inp, c_oracle), "degenerate rows")


def run_variant(inp):
    dev = torch.device("cuda:0")
    d = inp.to(dev)
    d.topk_res.fill_(-7)
    ret = pypto_amd.lightning_indexer_decode(*d.operator_tensors(), None, None, inp.selected_count,
                                             arith_variant="fp16_dequant")
    assert ret is None
    torch.cuda.synchronize()
    return d.topk_res.cpu()


@pytest.mark.parametrize("b,s1,act,k", [
    (2, 1, [4096, 3000], 2048),
    (3, 2, [300, 129, 5], 64),
    (1, 1, [33], 16),
    (2, 2, [9000, 2049], 2048),
])
def test_fp16_dequant_variant_bit_exact(b, s1, act, k):
    """The arithmetic of the reference's chained C++ operator (fp16 scales applied before the ReLU), against
    its own oracle."""
    from oracle import li_oracle as lo
    inp = gen_indexer_inputs(b, s1, act, selected_count=k, seed=11 * b + s1 + k, variant="fp16")
    want = lo.lightning_indexer_fp16_dequant_ref(inp.idx_query, inp.idx_query_scale, inp.idx_key_cache, inp.idx_key_scale,
                                                 inp.idx_weight, inp.act_seq_key, inp.block_table, k)
    assert_exact(run_variant(inp), want, f"fp16_dequant b={b} s1={s1} act={act} k={k}")


def test_fp16_dequant_variant_refuses_other_dtypes():
    inp = gen_indexer_inputs(1, 1, [300], selected_count=64, seed=1, variant="fp32").to(torch.device("cuda:0"))
    with pytest.raises(TypeError):
        pypto_amd.lightning_indexer_decode(*inp.operator_tensors(), None, None, 64, arith_variant="fp16_dequant")
    with pytest.raises(ValueError):
        pypto_amd.lightning_indexer_decode(*inp.operator_tensors(), None, None, 64, arith_variant="other")


@pytest.mark.parametrize("k,act", [
    (1, [1023, 1024, 1040, 2047]),               # 63 full groups of the sample (the general way), 64, 65, 127
    (64, [65, 1025, 16383, 16385]),
    (2047, [2048, 2049, 2064, 8193]),
    (2048, [2049, 32767, 32769, 65537]),         # chunks of the row scan: one short of full, one key into the next
])
def test_row_lengths_of_the_select(c_oracle, k, act):
    """Lengths at the edges of the sample, of the scan's chunks and of the selection itself; scores of both signs, many equal."""
    inp = gen_indexer_inputs(len(act), 1, act, selected_count=k, seed=k, variant="fp16")
    inp.idx_weight[1] = inp.idx_weight[1].sign() * 0.25
    inp.idx_query[1] = inp.idx_query[1].sign()
    inp.idx_key_cache[::3] = inp.idx_key_cache[0]
    assert_exact(run_op(inp), oracle(inp, c_oracle), f"k={k} act={act}")


@pytest.mark.parametrize("b,s1,lo,hi,cap", [
    (40, 1, 1, 3000, 131072),          # pages for far more keys than there are: a launch of more waves than one round
    (18, 3, 20000, 131072, 131072),    # the same with runs of every length, and a unit of one token
    (64, 1, 66000, 70000, 70016),      # more keys than a round of the longest runs holds
    (300, 3, 1, 3000, 3072),           # more units than sequences in a row of the table, one token each
    (520, 4, 1, 3000, 3072),           # more sequences than the table holds: runs of a fixed length, two tokens to a unit
    (521, 3, 1, 5000, 5120),           # the same, one token to a unit: the last workgroup is not full
])
def test_indexer_launches_of_more_than_one_round(b, s1, lo, hi, cap):
    """The rows of a batch whose runs are spread over all its sequences against the same rows scored one sequence at a time.  All
    sequences read the same 2048 pages in orders of their own."""
    g = torch.Generator().manual_seed(b)
    dev, pages, k = torch.device("cuda:0"), 2048, 2048
    act = torch.randint(lo, hi + 1, (b,), generator=g, dtype=torch.int32)
    act[-1] = hi
    table = torch.randint(0, pages, (b, cap // 128), generator=g, dtype=torch.int32).to(dev)
    q = torch.randint(-127, 128, (b * s1, 64, 128), generator=g, dtype=torch.int8).to(dev)
    qs = (torch.rand((b * s1, 64), generator=g) * 0.015 + 0.005).to(dev)
    w = (torch.randn((b * s1, 64), generator=g) * 0.125).to(torch.bfloat16).to(dev)
    keys = torch.randint(-127, 128, (pages, 128, 1, 128), generator=g, dtype=torch.int8).to(dev)
    ks = (torch.rand((pages, 128, 1), generator=g) * 0.015 + 0.005).to(dev)
    act = act.to(dev)
    got = torch.full((b * s1, 1, k), -7, dtype=torch.int32, device=dev)
    pypto_amd.lightning_indexer_decode(q, qs, keys, ks, w, act, table, got)
    one = torch.full((s1, 1, k), -7, dtype=torch.int32, device=dev)
    for i in range(b):
        r = slice(i * s1, (i + 1) * s1)
        pypto_amd.lightning_indexer_decode(q[r], qs[r], keys, ks, w[r], act[i:i + 1], table[i:i + 1].contiguous(), one)
        assert torch.equal(got[r], one), i


@pytest.mark.parametrize("variant", ["fp16", "fp32"])
@pytest.mark.parametrize("act,k,equal,far", [([513, 512, 1000, 1023, 1024, 1025, 2047, 2048], 2048, 900, 1500), ([600, 599, 513, 601, 20], 600, 600, 600),
                                             ([1, 2, 3, 63, 64, 65, 100, 129, 450], 2048, 900, 1500), ([1, 2, 1], 1, 1, 1),
                                             ([2049, 3000, 4096, 4097, 8191, 8192, 8193], 2048, 5000, 7000), ([1025, 7169, 9000], 1000, 8192, 1001)])
def test_short_rows_are_ordered_by_buckets_or_another_way(c_oracle, variant, act, k, equal, far):
    """All keys of a short row go to the buckets.  The last two rows have equal scores (all of them) and a score far from the
    rest, so that nearly all keys fall into one bucket."""
    act = act + [equal, far]
    inp = gen_indexer_inputs(len(act), 1, act, selected_count=k, seed=k, variant=variant)
    inp.idx_weight[-2] = 0
    pos = min(17, act[-1] - 1)
    page = inp.block_table[-1].long()[pos // 128]
    inp.idx_key_scale.reshape(-1)[page * 128 + pos % 128] = 60000.0
    assert_exact(run_op(inp), oracle(inp, c_oracle), f"{variant} k={k}")


def set_key_scale(inp, seq, positions, value):
    for pos in positions:
        inp.idx_key_scale.reshape(-1)[int(inp.block_table[seq, pos // 128]) * 128 + pos % 128] = value


@pytest.mark.parametrize("k,act", [(2048, [40, 1500, 2048]), (2048, [2049, 3000, 8192, 8193, 20000]), (100, [129, 1025, 5000])])
def test_select_with_infinite_scores(c_oracle, k, act):
    """Some scores infinite, of either sign: no range spreads the others over buckets.  Equal ones in the order of their positions."""
    inp = gen_indexer_inputs(len(act), 1, act, selected_count=k, seed=k + len(act), variant="fp32")
    for i, n in enumerate(act):
        set_key_scale(inp, i, range(3, n, 37), float("inf"))
    assert_exact(run_op(inp), oracle(inp, c_oracle), f"k={k} act={act}")


def test_select_of_every_key_with_scores_that_are_no_numbers(c_oracle):
    """Rows of at most k keys: those whose score is not a number come first, in the order of their positions, then the others."""
    act, bad = [65, 500, 1500, 2048], 41
    inp = gen_indexer_inputs(len(act), 1, act, selected_count=2048, seed=9, variant="fp32")
    want = oracle(inp, c_oracle)
    for i, n in enumerate(act):
        odd = list(range(5, n, bad))
        set_key_scale(inp, i, odd, float("nan"))
        rest = [x for x in want[i, 0, :n].tolist() if x not in odd]
        want[i, 0, :n] = torch.tensor(odd + rest, dtype=torch.int32)
    assert_exact(run_op(inp), want, "not a number")


@pytest.mark.parametrize("b,lengths,common", [(2, (3000, 5000), 16), (20, (300, 3000), 2), (40, (1, 2600), 20)])
def test_sequences_with_common_pages(c_oracle, b, lengths, common):
    """Sequences that begin with the same pages, all of them or every other one: their keys are kept in the caches, other ones not."""
    from pypto_amd.synthetic import gen_block_table
    g = torch.Generator().manual_seed(b)
    act = [int(x) for x in torch.randint(lengths[0], lengths[1] + 1, [b], generator=g)]
    num, table = gen_block_table(act, 128, g, shuffle=True, max_kv=lengths[1])
    first = table[max(range(b), key=lambda i: act[i])].clone()
    for i in range(0, b, 1 if b < 30 else 2):
        n = min(common, (act[i] + 127) // 128)
        table[i, :n] = first[:n]
    inp = gen_indexer_inputs(b, 1, act, selected_count=500, seed=b, variant="fp32", block_table=table, block_num=num)
    assert_exact(run_op(inp), oracle(inp, c_oracle), f"b={b} common={common}")
