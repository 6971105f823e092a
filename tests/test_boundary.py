"""The C-ABI library loads and exports every symbol the header declares; host-side argument
checking of the C ABI and of the Python operators (no GPU needed: nothing is launched)."""
import ctypes
import os
import re

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "pypto_amd", "libpypto_amd_sfa.so")
HEADER = os.path.join(ROOT, "include", "pypto_amd_sfa.h")


@pytest.fixture(scope="module")
def lib():
    if not os.path.exists(LIB):
        from pypto_amd.build import build_all
        build_all()
    return ctypes.CDLL(LIB)


def _declared():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(pto_\w+)\s*\(", text)))


def test_header_symbols_are_exported(lib):
    names = _declared()
    assert {"pto_sfa_quant_launch", "pto_sfa_quant_workspace_bytes", "pto_li_decode_launch",
            "pto_li_decode_workspace_bytes", "pto_li_prolog_quant_launch", "pto_li_prolog_quant_workspace_bytes",
            "pto_mla_prolog_quant_launch", "pto_mla_prolog_quant_workspace_bytes",
            "pto_last_error", "pto_version"} <= set(names)
    for n in names:
        assert hasattr(lib, n), n


def test_version_and_error_string(lib):
    lib.pto_version.restype = ctypes.c_char_p
    lib.pto_last_error.restype = ctypes.c_char_p
    assert re.fullmatch(rb"\d+\.\d+\.\d+", lib.pto_version())
    # the revision of the argument structs the library was built with is the one the header states
    declared = int(re.search(r"#define\s+PTO_ABI_REVISION\s+(\d+)", open(HEADER).read()).group(1))
    assert lib.pto_abi_revision() == declared
    n = ctypes.c_size_t(0)
    assert lib.pto_sfa_quant_workspace_bytes(None, ctypes.byref(n)) == -1
    assert b"NULL" in lib.pto_last_error()


def test_pybind_workspace_and_argument_errors():
    from pypto_amd import _native
    C = _native.load()
    # 32 rows x 8 splits x 128 heads x (512 fp16 + 2 fp32)
    assert C.sfa_quant_workspace_bytes(32, 1, 128, 1, 2048, 128, 512, 1 << 20, 0.04, 8) == 32 * 8 * 128 * (512 * 2 + 8)
    # more rows than compute units, a cache much larger than the selections: neither split nor de-quantised copy
    assert C.sfa_quant_workspace_bytes(4096, 1, 128, 1, 2048, 128, 32, 1 << 21, 0.04, 0) == 0
    # the automatic split (a host without a device plans for 256 compute units in 8 XCDs): 32 rows in 8 pieces each;
    # 200 rows whole; 300 rows as 256 whole rows and the other 44 in 5 pieces each; 260 rows as 256 whole rows and
    # the other 4 in 16 pieces (a piece keeps at least four tiles of 32 keys)
    assert C.sfa_quant_workspace_bytes(32, 1, 128, 1, 2048, 128, 512, 1 << 21, 0.04, 0) == 32 * 8 * 128 * (512 * 2 + 8)
    assert C.sfa_quant_workspace_bytes(200, 1, 128, 1, 2048, 128, 32, 1 << 21, 0.04, 0) == 0
    assert C.sfa_quant_workspace_bytes(300, 1, 128, 1, 2048, 128, 32, 1 << 21, 0.04, 0) == 44 * 5 * 128 * (512 * 2 + 8)
    assert C.sfa_quant_workspace_bytes(260, 1, 128, 1, 2048, 128, 32, 1 << 21, 0.04, 0) == 4 * 16 * 128 * (512 * 2 + 8)
    # prefill-shaped (every cache row selected by many query rows): one bf16 copy of the 4096 cache rows
    assert C.sfa_quant_workspace_bytes(4096, 1, 128, 1, 2048, 128, 32, 4096, 0.04, 0) == 4096 * 512 * 2
    assert C.li_decode_workspace_bytes(4, 4, 64, 128, 1024, 128, 256, 2048, 0, 0, 0) == 4 * (32768 + 2048) * 4
    # prolog: 4 int32 partial projections [t, 8192] + 112 block sums [t, 192] fp32
    assert C.li_prolog_quant_workspace_bytes(8, 7168, 1536, 64, 1 << 20) == 4 * 8 * 8192 * 4 + 112 * 8 * 192 * 4
    with pytest.raises(ValueError):
        C.li_prolog_quant_workspace_bytes(8, 7168, 1280, 64, 1 << 20)                # q_lora_rank not supported
    with pytest.raises(ValueError):
        C.li_prolog_quant_workspace_bytes(8, 7100, 1536, 64, 1 << 20)                # h not a multiple of 64
    with pytest.raises(ValueError):
        C.li_prolog_quant_workspace_bytes(8, 7168, 1536, 65, 1 << 20)                # more than 64 heads
    # MLA prolog: 14 group sums [t, 1536 + 576] fp32 + 4 int32 partial projections [t, 128 * 192]
    assert C.mla_prolog_quant_workspace_bytes(8, 7168, 1536, 128, 1 << 16) == 14 * 8 * 2112 * 4 + 4 * 8 * 24576 * 4
    # from 9 tokens on the partial sums over the hidden axis may be the matrix-core form's ranges (up to fourteen, one
    # per block of 64 hidden rows at most): a 192-wide hidden axis is one group but three ranges
    assert C.mla_prolog_quant_workspace_bytes(150, 192, 512, 2, 1 << 16) == 3 * 150 * 1088 * 4 + 4 * 150 * 384 * 4
    assert C.mla_prolog_quant_workspace_bytes(32, 192, 512, 2, 1 << 16) == 3 * 32 * 1088 * 4 + 4 * 32 * 384 * 4
    assert C.mla_prolog_quant_workspace_bytes(15, 192, 512, 2, 1 << 16) == 3 * 15 * 1088 * 4 + 4 * 15 * 384 * 4
    assert C.mla_prolog_quant_workspace_bytes(8, 192, 512, 2, 1 << 16) == 1 * 8 * 1088 * 4 + 4 * 8 * 384 * 4
    with pytest.raises(ValueError, match="sum_mode"):                                # indexer prolog: sum_mode is 0, 1 or 2
        C.li_prolog_quant_launch(*([0] * 19), 0, 0, 8, 7168, 1536, 64, 1 << 20, 1e-6, 3, 0)
    with pytest.raises(ValueError):
        C.mla_prolog_quant_workspace_bytes(8, 7168, 1536, 127, 1 << 16)              # odd head count
    with pytest.raises(ValueError):
        C.mla_prolog_quant_workspace_bytes(8, 32768, 1536, 128, 1 << 16)             # hidden size beyond the limit
    with pytest.raises(ValueError):
        C.sfa_quant_workspace_bytes(1, 1, 128, 2, 2048, 128, 32, 4096, 0.04, 0)      # n_kv != 1
    with pytest.raises(ValueError):
        C.li_decode_workspace_bytes(4, 4, 32, 128, 1024, 128, 256, 2048, 0, 0, 0)    # 32 heads
    with pytest.raises(ValueError):
        C.li_decode_workspace_bytes(4, 4, 64, 128, 1024, 128, 256, 4096, 0, 0, 0)    # selected_count > 2048
    with pytest.raises(ValueError):
        C.li_decode_workspace_bytes(4, 4, 64, 128, 4096, 128, 2048, 2048, 0, 0, 0)   # longer than 128K
    with pytest.raises(ValueError):                                                  # NULL tensors
        C.sfa_quant_launch(0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 1, 1, 16, 1, 256, 128, 32, 4096, 0.04, 0, 0)


def test_from_torch_contract():
    import pypto_amd
    t = torch.zeros(4, 6)
    h = pypto_amd.from_torch(t, name="x", dynamic_axis=[0])
    assert h.shape == [4, 6] and h.dtype == torch.float32 and h.data_ptr == t.data_ptr() and h.name == "x"
    with pytest.raises(TypeError):
        pypto_amd.from_torch([1, 2, 3])
    with pytest.raises(RuntimeError):
        pypto_amd.from_torch(t.t())


def test_operators_refuse_cpu_tensors_loudly():
    """There is no CPU fallback behind the operator names."""
    import pypto_amd
    from pypto_amd.synthetic import gen_sfa_inputs, gen_indexer_inputs
    inp = gen_sfa_inputs(1, 1, 16, [256], topk=64, seed=0)
    out = torch.zeros(1, 1, 16, 512, dtype=torch.bfloat16)
    with pytest.raises(RuntimeError):
        pypto_amd.sparse_flash_attention_quant_d(*inp.operator_tensors(), out, 16, 1, inp.softmax_scale, 64, 128,
                                                 inp.max_blocknum_perbatch, None)
    li = gen_indexer_inputs(1, 1, [256], selected_count=64, seed=0)
    with pytest.raises(RuntimeError):
        pypto_amd.lightning_indexer_decode(*li.operator_tensors(), None, None, 64)


def test_prolog_operators_refuse_cpu_tensors_and_unbuilt_variants():
    import pypto_amd
    from pypto_amd.synthetic import gen_indexer_prolog_inputs, gen_mla_prolog_inputs
    kw = dict(h=128, q_lora_rank=512, n_heads=2)
    lip = gen_indexer_prolog_inputs(1, 1, [130], seed=0, **kw)
    outs = (torch.zeros(1, 2, 128, dtype=torch.int8), torch.zeros(1, 2, 1, dtype=torch.float16), lip.k_cache,
            lip.k_cache_scale, torch.zeros(1, 2, dtype=torch.float16))
    with pytest.raises(RuntimeError):
        pypto_amd.lightning_indexer_prolog_quant(*lip.input_tensors(), *outs)
    with pytest.raises(ValueError):
        pypto_amd.lightning_indexer_prolog_quant(*lip.input_tensors(), *outs,
                                                 pypto_amd.IndexerPrologQuantAttr(layerout_key="BSND"))
    mla = gen_mla_prolog_inputs(1, 1, [130], seed=0, **kw)
    mouts = (torch.zeros(1, 512, dtype=torch.int8), torch.zeros(1, 1), torch.zeros(1, 2, 512, dtype=torch.bfloat16),
             torch.zeros(1, 2, 64, dtype=torch.bfloat16), mla.kv_cache, mla.kr_cache, mla.k_scale_cache)
    with pytest.raises(RuntimeError):
        pypto_amd.mla_prolog_quant_d(*mla.input_tensors(), *mouts, 1e-5, 1e-5, "PA_BSND", None, None)
    with pytest.raises(RuntimeError):                    # an accepted cache mode (the reference asserts "PA_BSND" or "PA_NZ"
        pypto_amd.mla_prolog_quant_d(*mla.input_tensors(), *mouts, 1e-5, 1e-5, "PA_NZ", None, None)   # and treats them alike)
    with pytest.raises(ValueError):
        pypto_amd.mla_prolog_quant_d(*mla.input_tensors(), *mouts, 1e-5, 1e-5, "BSND", None, None)
    args = list(mla.input_tensors())
    args[3] = None                                       # no dequant scale: the non-quantized up-projection
    with pytest.raises(ValueError):
        pypto_amd.mla_prolog_quant_d(*args, *mouts, 1e-5, 1e-5, "PA_BSND", None, None)


def test_cache_out_overlapping_cache_in_is_refused():
    """The prolog operators copy cache-in to cache-out unless they are the same tensor; two views that share
    memory without being the same range must not be copied onto each other."""
    import torch
    from pypto_amd.converter import copy_unless_same
    base = torch.arange(64, dtype=torch.int8)
    copy_unless_same(base[:32], base[:32], "k_int8")                 # same range: nothing happens
    other = torch.zeros(32, dtype=torch.int8)
    copy_unless_same(other, base[:32], "k_int8")                     # disjoint: copied
    assert torch.equal(other, base[:32])
    with pytest.raises(ValueError, match="overlap"):
        copy_unless_same(base[8:40], base[:32], "k_int8")


@pytest.mark.parametrize("nq,topk,rows", [
    (128, 128, range(1, 20)), (128, 192, range(1, 20)), (128, 224, range(1, 20)), (64, 224, range(1, 40)), (16, 96, range(1, 80)),
    (16, 128, range(1, 80)), (16, 224, range(1, 80)), (32, 256, range(25, 75)), (16, 256, range(281, 328)), (32, 320, range(75, 113)),
    (64, 256, range(25, 40)), (128, 256, range(281, 284)), (16, 1024, range(129, 171)), (32, 768, range(129, 157)),
    (16, 2048, range(169, 193)), (32, 1536, range(169, 193)), (64, 2048, range(169, 171)), (128, 2048, range(169, 171)),
    (256, 2048, range(81, 86))])
def test_attention_launches_without_half_precision_partials(nq, topk, rows):
    """These launches (short selections at small batches, batches that just miss the next round of the chip) keep their rows
    whole or leave the partial results of split rows in fp32, never in fp16."""
    from pypto_amd import _C
    for r in rows:
        need = _C.sfa_quant_workspace_bytes(r, 1, nq, 1, topk, 128, 512, 1 << 30, 0.04, 0)
        assert need in [0] + [r * s * nq * (512 * 4 + 8) for s in range(2, 9)], r


@pytest.mark.parametrize("nq,topk,rows,splits", [(128, 2048, 1, 32), (128, 2048, 32, 8), (16, 256, 24, 4), (128, 256, 4, 8), (16, 2048, 168, 3)])
def test_attention_launches_with_half_precision_partials(nq, topk, rows, splits):
    from pypto_amd import _C
    assert _C.sfa_quant_workspace_bytes(rows, 1, nq, 1, topk, 128, 512, 1 << 30, 0.04, 0) == rows * splits * nq * (512 * 2 + 8)


def attention_plan(rows, nq, topk, splits=0):
    from pypto_amd import _C
    args = (rows, 1, nq, 1, topk, 128, 512, 1 << 30, 0.04, splits)
    return _C.sfa_quant_plan(*args), _C.sfa_quant_workspace_bytes(*args)


@pytest.mark.parametrize("nq", [1, 16, 33, 64, 100, 128, 192])
@pytest.mark.parametrize("topk", [1, 32, 200, 256, 768, 2048, 2049, 4096])
def test_attention_plan_stays_within_the_bytes_a_caller_is_asked_for(nq, topk):
    """A launch checks the workspace against the bytes asked for; what its plan lays out there is never more."""
    for rows in [*range(1, 80), 127, 128, 129, 168, 200, 255, 256, 257, 283, 300, 513, 4096]:
        plan, need = attention_plan(rows, nq, topk)
        assert plan["heads_per_workgroup"] in (32, 64, 128) and 1 <= plan["key_splits"] <= (topk + 31) // 32
        assert plan["key_splits"] * 2048 >= topk, rows                     # a split's keys fit a workgroup
        split_rows = rows - plan["whole_rows"] if plan["key_splits"] > 1 else 0
        assert plan["partial_bytes"] == split_rows * plan["key_splits"] * nq * (512 * plan["partial_element_bytes"] + 8) <= need, rows
        assert plan["partial_element_bytes"] != 4 or plan["key_splits"] <= 8, rows


@pytest.mark.parametrize("nq,topk,rows,keys,block", [
    (64, 2048, [167, 168], range(1664, 2048, 128), 128), (40, 2048, [167], [1984], 64), (64, 256, [10], range(160, 256, 16), 16),
    (128, 256, [5], range(192, 256, 16), 16), (33, 2048, [168], [1920], 64), (128, 2048, [1, 2, 5, 33, 258, 300], range(128, 2048, 128), 128),
    (16, 1024, [3, 24, 128, 170, 258], range(128, 1024, 128), 128), (32, 2048, [4, 100, 147, 170], range(128, 2048, 128), 128)])
def test_short_block_tables_leave_no_row_fewer_bits(nq, topk, rows, keys, block):
    """A call whose pages hold fewer keys than topk may be divided another way than by topk: here in no more splits, whole rows still
    whole, no partial result in fewer bits, and for the same workspace."""
    from pypto_amd import _C
    for r in rows:
        for n in keys:
            args = lambda pages: (r, 1, nq, 1, topk, block, pages, 1 << 30, 0.04, 0)  # noqa: E731
            wide, short = _C.sfa_quant_plan(*args(topk // block)), _C.sfa_quant_plan(*args(n // block))
            assert short["key_splits"] <= wide["key_splits"], (r, n)
            assert short["key_splits"] == 1 or short["whole_rows"] == wide["whole_rows"], (r, n)
            assert short["key_splits"] == 1 or short["partial_element_bytes"] == wide["partial_element_bytes"], (r, n)
            assert short["partial_bytes"] <= _C.sfa_quant_workspace_bytes(*args(n // block)) == _C.sfa_quant_workspace_bytes(*args(topk // block)), (r, n)


@pytest.mark.parametrize("b,s1,nq,topk,keys,last", [
    (1, 8, 128, 2048, 2048, False), (1, 9, 128, 2048, 2048, True), (32, 1, 128, 2048, 65536, False),        # decoding rows; a chunk
    (1, 4096, 128, 2048, 4096, True), (1, 1000, 64, 1024, 1024, True), (1, 300, 64, 512, 384, True),        # most rows still growing
    (1, 2000, 128, 512, 2048, False), (1, 1219, 64, 256, 1280, False), (1, 1219, 64, 1024, 1664, False),    # most rows of full length
    (1, 1219, 32, 256, 1280, True), (64, 16, 32, 512, 384, True),                                           # short rows of one group of heads
    (8, 128, 64, 2048, 128, False), (2, 300, 64, 2048, 384, True), (5, 2000, 128, 2048, 2048, True)])       # several sequences
def test_rows_that_a_launch_of_whole_rows_starts_with(b, s1, nq, topk, keys, last):
    """Longest first where the launch then ends with short rows, and not where rows of full length would start together."""
    from pypto_amd import _C
    assert _C.sfa_last_first(b, s1, nq, topk, keys, 256) == last


@pytest.mark.parametrize("rows,nq,topk,pages,splits", [(5, 64, 1024, 6, 12), (6, 48, 2048, 14, 14), (3, 128, 2048, 14, 14), (6, 128, 2048, 15, 10), (12, 64, 2048, 11, 8)])
def test_short_block_tables_in_more_splits(rows, nq, topk, pages, splits):
    """More splits than by topk, where their price says so by enough, within the workspace that is asked for whatever the table."""
    from pypto_amd import _C
    args = lambda pages: (rows, 1, nq, 1, topk, 128, pages, 1 << 30, 0.04, 0)  # noqa: E731
    wide, short = _C.sfa_quant_plan(*args(topk // 128)), _C.sfa_quant_plan(*args(pages))
    assert short["key_splits"] == splits >= wide["key_splits"] and short["partial_element_bytes"] == wide["partial_element_bytes"]
    assert short["partial_bytes"] <= _C.sfa_quant_workspace_bytes(*args(pages)) == _C.sfa_quant_workspace_bytes(*args(topk // 128))


@pytest.mark.parametrize("s1,nq,topk,pages,whole", [
    (300, 128, 2048, 3, True), (530, 64, 2048, 5, True), (800, 128, 2048, 7, True), (600, 64, 512, 5, True), (300, 16, 2048, 3, True), (2338, 128, 2048, 20, True),
    (518, 128, 512, 5, False), (518, 64, 2048, 6, False), (780, 128, 512, 7, False), (1030, 64, 512, 9, False), (2060, 64, 1024, 18, False)])
def test_chunks_whose_rows_stay_whole(s1, nq, topk, pages, whole):
    """Rows of all lengths stay whole, unless what is left for a last round is little beside the rounds before it."""
    from pypto_amd import _C
    plan = _C.sfa_quant_plan(1, s1, nq, 1, topk, 128, pages, 1 << 14, 0.04, 0)
    assert (plan["key_splits"] == 1) == whole, plan


@pytest.mark.parametrize("heads,splits,element,names", [
    (64, 4, 2, "sfa_slice_kernel<true> + sfa_combine_kernel<4, false>"), (128, 1, 0, "sfa_decode_kernel<4, true>"),
    (128, 7, 2, "sfa_decode_kernel<4, true> + sfa_combine_kernel<8, false>"), (32, 2, 4, "sfa_decode_kernel<1, true> + sfa_combine_kernel<2, true>"),
    (64, 9, 2, "sfa_slice_kernel<true> + sfa_combine_wide_kernel<4>"), (32, 22, 2, "sfa_decode_kernel<1, true> + sfa_combine_wide_kernel<8>")])
def test_benchmark_follows_the_plan_of_the_library(heads, splits, element, names):
    """Split count and kernels in the benchmark's line are those of the plan, whatever it is: counter figures taken with another
    one are then recognised as stale."""
    from types import SimpleNamespace
    import bench
    plan = dict(heads_per_workgroup=heads, key_splits=splits, whole_rows=0, partial_element_bytes=element, partial_bytes=0)
    assert bench.attention_plan(SimpleNamespace(sfa_quant_plan=lambda *a: plan), 32, 1) == (splits, names)
    from pypto_amd import _C
    assert bench.attention_plan(_C, 32, 1, 128, 1, 2048, 128, 512, 1 << 21, 0.04)[0] == _C.sfa_quant_plan(32, 1, 128, 1, 2048, 128, 512, 1 << 21, 0.04, 0)["key_splits"]


@pytest.mark.parametrize("pages", [1024, 8615, 40000])
def test_benchmark_times_the_indexer_over_keys_that_are_in_no_cache(pages):
    """Between two passes over one copy of the keys the benchmark reads more than the memory-side cache holds."""
    import bench
    sets = bench.key_sets(torch.empty([pages, 128, 1, 128], dtype=torch.int8, device="meta"), torch.empty([pages, 128, 1], device="meta"))
    one = pages * 128 * (128 + 4)
    assert all(k.shape == sets[0][0].shape and s.shape == sets[0][1].shape for k, s in sets)
    assert bench.MEMORY_SIDE_CACHE == 256 << 20 and 2 * bench.MEMORY_SIDE_CACHE <= (len(sets) - 1) * one <= 2 * bench.MEMORY_SIDE_CACHE + one
