"""The operators' native call path (csrc/torch_calls.cpp): what it takes it treats as the Python path does."""
import pytest
import torch

import pypto_amd
from pypto_amd.synthetic import gen_indexer_inputs, gen_indexer_prolog_inputs, gen_mla_prolog_inputs, gen_sfa_inputs

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")


def attention_call():
    """(operator, arguments, positions of the written tensors): 4 rows of 16 heads, top-k 64."""
    inp = gen_sfa_inputs(4, 1, 16, [200, 90, 64, 33], topk=64, seed=1)
    d = inp.to(DEV)
    out = torch.zeros([4, 1, 16, 512], dtype=torch.bfloat16, device=DEV)
    args = [*d.operator_tensors(), out, 16, 1, inp.softmax_scale, 64, inp.block_size, inp.max_blocknum_perbatch, None]
    return pypto_amd.sparse_flash_attention_quant_d, args, [8]


def packed_attention_call():
    from pypto_amd.synthetic import pack_nope_cache
    inp = gen_sfa_inputs(4, 1, 16, [200, 90, 64, 33], topk=64, seed=1)
    d = inp.to(DEV)
    packed = pack_nope_cache(inp.key_nope_2d, inp.key_rope_2d, inp.k_nope_scales).to(DEV)
    out = torch.zeros([4, 1, 16, 512], dtype=torch.bfloat16, device=DEV)
    args = [d.query_nope, d.query_rope, packed, d.topk_indices, d.block_table, d.kv_act_seqs, out, 16, 1, inp.softmax_scale, 64,
            inp.block_size, inp.max_blocknum_perbatch, None]
    return pypto_amd.sparse_attention_antiquant_d, args, [6]


def indexer_call():
    inp = gen_indexer_inputs(4, 1, [200, 90, 64, 300], selected_count=64, seed=2)
    d = inp.to(DEV)
    return pypto_amd.lightning_indexer_decode, [*d.operator_tensors(), None, None, 64], [7]


def prolog_tensors():
    kw = dict(h=128, q_lora_rank=512)
    mla = gen_mla_prolog_inputs(4, 1, [130] * 4, seed=3, n_heads=2, **kw).to(DEV)
    lip = gen_indexer_prolog_inputs(4, 1, [130] * 4, seed=4, n_heads=4, **kw).to(DEV)
    new = lambda shape, dtype: torch.zeros(shape, dtype=dtype, device=DEV)          # noqa: E731
    q = dict(nope=new([4, 2, 512], torch.bfloat16), rope=new([4, 2, 64], torch.bfloat16), norm=new([4, 512], torch.int8),
             norm_scale=new([4, 1], torch.float32), int8=new([4, 4, 128], torch.int8), scale=new([4, 4, 1], torch.float16),
             weights=new([4, 4], torch.float16))
    return mla, lip, q


def mla_prolog_call():
    mla, _, q = prolog_tensors()
    args = [*mla.input_tensors(), q["norm"], q["norm_scale"], q["nope"], q["rope"], mla.kv_cache, mla.kr_cache, mla.k_scale_cache,
            1e-5, 1e-5, "PA_BSND", None, None]
    return pypto_amd.mla_prolog_quant_d, args, [14, 15, 16, 17, 18, 19, 20]


def indexer_prolog_call():
    _, lip, q = prolog_tensors()
    return pypto_amd.lightning_indexer_prolog_quant, [*lip.input_tensors(), q["int8"], q["scale"], lip.k_cache, lip.k_cache_scale,
                                                      q["weights"]], [16, 17, 18, 19, 20]


def fused_prolog_call():
    m, l, q = prolog_tensors()
    args = [*m.input_tensors(), l.w_qb, l.w_qb_scale, l.wk, l.w_proj, l.ln_gamma_k, l.ln_beta_k, l.hadamard_q, l.hadamard_k, l.k_cache,
            l.k_cache_scale, q["nope"], q["rope"], m.kv_cache, m.kr_cache, m.k_scale_cache, q["int8"], q["scale"], l.k_cache,
            l.k_cache_scale, q["weights"], 1e-5, 1e-5, "PA_BSND", None, None, None, None]
    return pypto_amd.mla_indexer_prolog_quant_d, args, list(range(24, 34))


CALLS = {f.__name__: f for f in (attention_call, packed_attention_call, indexer_call, mla_prolog_call, indexer_prolog_call,
                                 fused_prolog_call)}


@pytest.mark.parametrize("which", CALLS)
def test_outputs_that_share_memory_copy_on_write_are_written_apart(which):
    """An output (cache-out included) that is a lazy clone of another tensor gets memory of its own: the other tensor keeps its
    values, and the clone holds what an ordinary output holds."""
    op, args, written = CALLS[which]()
    op(*args)
    torch.cuda.synchronize()
    want = [args[i].clone() for i in written]
    op, args, written = CALLS[which]()
    base = [args[i] for i in written]
    before = [t.clone() for t in base]
    lazy = {id(t): torch._lazy_clone(t) for t in base}
    args = [lazy.get(id(a), a) for a in args]                      # a cache is passed in and out as one tensor
    op(*args)
    torch.cuda.synchronize()
    for t, b, i, w in zip(base, before, written, want):
        assert torch.equal(t.view(torch.uint8), b.view(torch.uint8)), i
        assert torch.equal(args[i].clone().view(torch.uint8), w.view(torch.uint8)), i


@pytest.mark.parametrize("which", ["mla_prolog_call", "indexer_prolog_call", "fused_prolog_call"])
def test_cache_out_that_is_a_lazy_clone_of_cache_in_is_another_cache(which):
    """Cache-in and cache-out share memory copy-on-write until one is written: cache-in stays as it was."""
    op, args, written = CALLS[which]()
    op(*args)
    torch.cuda.synchronize()
    want = [args[i].clone() for i in written]
    op, args, written = CALLS[which]()
    caches = [i for i in written if any(args[i] is a for a in args[:written[0]])]
    base, before = [args[i] for i in caches], [args[i].clone() for i in caches]
    for i in caches:
        args[i] = torch._lazy_clone(args[i])
    op(*args)
    torch.cuda.synchronize()
    for t, b in zip(base, before):
        assert torch.equal(t.view(torch.uint8), b.view(torch.uint8))
    for i, w in zip(written, want):
        assert torch.equal(args[i].clone().view(torch.uint8), w.view(torch.uint8)), i


def outcome(op, args):
    try:
        op(*args)
    except Exception as e:                                           # noqa: BLE001 (whatever it raises is what is compared)
        return type(e), str(e)
    torch.cuda.synchronize()
    return None


NATIVE = ("sfa_call", "sa_antiquant_call", "li_decode_call", "mla_prolog_call", "li_prolog_call", "fused_prolog_call")


@pytest.fixture
def python_path():
    """A call with the native path switched off."""
    from pypto_amd import _native
    C = _native.load()

    def run(op, args):
        with pytest.MonkeyPatch.context() as m:
            for name in NATIVE:
                m.setattr(C, name, lambda *a: False)
            return outcome(op, args)
    return run


def other_type(t):
    return t.to(torch.int64 if t.dtype != torch.int64 and not t.dtype.is_floating_point else torch.float64)


def strided(t):
    wide = torch.zeros([*t.shape, 2], dtype=t.dtype, device=t.device)
    return wide[..., 0]


MALFORMED = {"type": other_type, "host": lambda t: t.cpu(), "strided": strided, "short": lambda t: t[:-1].clone(),
             "dimension": lambda t: t.unsqueeze(0), "none": lambda t: None, "list": lambda t: [1, 2]}


@pytest.mark.parametrize("how", MALFORMED)
@pytest.mark.parametrize("which", CALLS)
def test_malformed_tensors_end_the_same_way_on_both_paths(which, how, python_path):
    """Every tensor argument in turn, of the wrong type, device, stride or shape: refused with the same error by either path,
    or (where only the number of elements counts) taken by both."""
    op, args, _ = CALLS[which]()
    refused = 0
    for i, a in enumerate(args):
        if not torch.is_tensor(a) or (how == "short" and which == "packed_attention_call" and i == 2):
            continue                                                 # (a packed cache of one row fewer is another valid cache)
        bad = list(args)
        bad[i] = MALFORMED[how](a)
        want = python_path(op, bad)
        assert outcome(op, bad) == want, i
        refused += want is not None
    assert refused > 0


BIG = 1 << 62
MALFORMED_NUMBERS = {
    "attention_call": [(9, v) for v in (0, -1, 7, BIG, 1 << 64, "x", None)] + [(10, v) for v in (0, 2, BIG)] +
                      [(12, v) for v in (0, -1, 63, BIG, BIG + 16)] + [(13, v) for v in (0, -1, 1 << 40, BIG)] +
                      [(14, v) for v in (1 << 20, BIG)] + [(11, v) for v in (float("nan"), float("inf"), 1e300, "x", None)],
    "packed_attention_call": [(7, v) for v in (0, -1, 7, BIG, 1 << 64)] + [(8, v) for v in (0, 2, BIG)] +
                             [(10, v) for v in (0, 63, BIG)] + [(11, v) for v in (0, 1 << 40)] + [(12, BIG), (9, float("nan"))],
    "indexer_call": [(10, v) for v in (0, -1, 63, 4096, BIG, BIG + 64, "x", None)],
    "mla_prolog_call": [(21, v) for v in (float("nan"), -1.0, "x", None)] + [(22, float("inf")), (23, "BSND")],
    "fused_prolog_call": [(34, v) for v in (float("nan"), -1.0, "x", None)] + [(35, float("inf")), (36, "BSND")],
}


@pytest.mark.parametrize("which", MALFORMED_NUMBERS)
def test_malformed_numbers_end_the_same_way_on_both_paths(which, python_path):
    """Counts that are zero, negative, no divisor, or large enough that products of them would wrap; scalars that are not finite
    or no numbers."""
    op, args, _ = CALLS[which]()
    for i, v in MALFORMED_NUMBERS[which]:
        bad = list(args)
        bad[i] = v
        want = python_path(op, bad)
        assert want is not None, (i, v)
        assert outcome(op, bad) == want, (i, v)
