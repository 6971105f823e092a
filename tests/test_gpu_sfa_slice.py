"""Attention with 64 heads per workgroup (33 heads and more, few rows) against the CPU oracle where it can go wrong: edges of
tiles and of the two key halves of a tile, partial head shares, splits without keys, maxima that move at every tile, whole and
split rows in one launch, all cache formats."""
import pytest
import torch

import pypto_amd
from pypto_amd import sparse_flash_attention_quant_impl as impl
from pypto_amd.synthetic import gen_sfa_inputs, pack_nope_cache

from test_gpu_sfa import check, oracle, run_op

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_q", [33, 64, 100])
@pytest.mark.parametrize("keys", [1, 15, 16, 17, 31, 33, 64, 65, 97, 129, 700])
def test_edges_of_tiles(n_q, keys):
    inp = gen_sfa_inputs(2, 1, n_q, [keys, 700], topk=768, seed=n_q + keys)
    check(run_op(inp), oracle(inp), f"nq={n_q} keys={keys}")
    check(run_op(inp, num_splits=2), oracle(inp), f"nq={n_q} keys={keys}, 2 splits")


@pytest.mark.parametrize("scale", [0.0416666679084301, -0.0416666679084301, 0.0, 2.0])
@pytest.mark.parametrize("order", [1, -1])
def test_moving_maxima(scale, order):
    """Scores that grow (or fall) with the position, by far more than the running maximum may lag behind within a tile."""
    inp = gen_sfa_inputs(1, 2, 64, [640], topk=640, seed=11, shuffle_table=False)
    inp.softmax_scale = scale
    pos = torch.arange(640, dtype=torch.int32)
    inp.topk_indices[:] = pos if order > 0 else pos.flip(0)
    inp.topk_indices[0, :] = torch.where(inp.topk_indices[0] >= 639, 0, inp.topk_indices[0])
    inp.query_nope[:] = (inp.query_nope.float() * 0.2 + 1.0).to(torch.bfloat16)
    inp.k_nope_scales[:640] = torch.linspace(1e-3, 2e-2, 640)[:, None]
    inp.key_nope_2d[:640] = inp.key_nope_2d[:640].abs()
    check(run_op(inp), oracle(inp), f"scale={scale} order={order}")
    check(run_op(inp, num_splits=3), oracle(inp), f"scale={scale} order={order}, 3 splits")


@pytest.mark.parametrize("n_q,b,s1,topk", [(64, 40, 2, 2048), (64, 71, 4, 512), (128, 8, 2, 2048), (128, 31, 1, 1024)])
def test_formats_agree(n_q, b, s1, topk):
    """int8, packed and bf16 caches: the same bits; and the split launch against one workgroup per row and head share."""
    from oracle import sfa_oracle as so
    inp = gen_sfa_inputs(b, s1, n_q, [100 + 61 * i for i in range(b)], topk=topk, seed=b)
    d = inp.to(torch.device("cuda:0"))
    out = run_op(inp)
    other = torch.full_like(out, float("nan"), device="cuda:0")
    tail = (d.topk_indices, d.block_table, d.kv_act_seqs, other, n_q, 1, inp.softmax_scale, topk, inp.block_size, inp.max_blocknum_perbatch)
    pypto_amd.sparse_flash_attention_quant_d(d.query_nope, d.query_rope, so.dequant_kn(inp.key_nope_2d, inp.k_nope_scales).cuda(),
                                             d.key_rope_2d, None, *tail)
    assert torch.equal(other.cpu().view(torch.int16), out.view(torch.int16))
    other.fill_(float("nan"))
    pypto_amd.sparse_attention_antiquant_d(d.query_nope, d.query_rope, pack_nope_cache(d.key_nope_2d, d.key_rope_2d, d.k_nope_scales), *tail)
    assert torch.equal(other.cpu().view(torch.int16), out.view(torch.int16))
    whole = run_op(inp, num_splits=1).float()
    # a partial's rounding to fp16 (2^-11), the result's and P's to bf16 (2^-9 each), on a weighted mean of values
    assert (out.float() - whole).abs().max() <= 3 * 2.0 ** -8 * whole.abs().max()
