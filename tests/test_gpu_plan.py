"""The plan that la_mla_decode_plan reports, kernel by kernel (host only: no
pointer is read). Tests of one kernel assert through it that their sizes reach
that kernel."""

from __future__ import annotations

import ctypes

import pytest

from mla_cases import cfg_with_heads

from latent_attn import capi

pytestmark = pytest.mark.gpu

CODE = {"bf16": capi.LA_DTYPE_BF16, "f16": capi.LA_DTYPE_F16, "f32": capi.LA_DTYPE_F32, "fp8": capi.LA_DTYPE_FP8_E4M3}


def plan_args(dtype, heads, num_seqs, seq_len, qps=1, wdtype=None, **kw):
    a = capi.DecodeArgs()
    fake = 0x10000
    a.kv_cache = a.q_nope = a.W_UK = a.q_rope = a.W_UV = a.rope_cos = a.rope_sin = a.output = fake
    a.kv_dtype = CODE[dtype]
    a.w_uk_dtype = a.w_uv_dtype = CODE[wdtype or {"fp8": "bf16"}.get(dtype, dtype)]
    a.num_seqs, a.seq_len, a.queries_per_seq, a.total_rows = num_seqs, seq_len, qps, num_seqs * seq_len
    a.cfg = capi.config(cfg_with_heads(heads))
    for k, v in kw.items():
        setattr(a, k, v)
    return a


def plan(*args, **kw):
    a, info = plan_args(*args, **kw), capi.PlanInfo()
    assert capi.load().la_mla_decode_plan(ctypes.byref(a), ctypes.byref(info)) == capi.LA_SUCCESS
    return info


# (dtype, heads, sequences, rows, queries, other fields): attention, head_groups, heads_per_workgroup, filled_rows, merge
MFMA, F32, VALU = capi.LA_PLAN_ATTENTION_MFMA, capi.LA_PLAN_ATTENTION_MFMA_F32, capi.LA_PLAN_ATTENTION_VALU
LENS = {"seq_lens": 0x10000}


@pytest.mark.parametrize("args,kw,want", [
    (("bf16", 128, 1, 512), {}, (MFMA, 1, 16, 0, capi.LA_PLAN_MERGE_MFMA_HALVES)),
    (("bf16", 128, 32, 8192), {}, (MFMA, 1, 128, 0, capi.LA_PLAN_MERGE_MFMA)),
    (("f16", 48, 1, 16384, 3), {}, (MFMA, 2, 128, 0, capi.LA_PLAN_MERGE_MFMA_HALVES)),
    (("fp8", 16, 32, 4099), {}, (MFMA, 1, 16, 0, capi.LA_PLAN_MERGE_MFMA_HALVES)),
    (("fp8", 128, 16, 6016), LENS, (MFMA, 1, 128, 1, capi.LA_PLAN_MERGE_MFMA_HALVES)),
    (("bf16", 128, 16, 6016), {**LENS, "chunk_rows": 512}, (MFMA, 1, 128, 0, capi.LA_PLAN_MERGE_MFMA_HALVES)),
    (("f32", 128, 4, 1000), {}, (F32, 8, 16, 0, capi.LA_PLAN_MERGE_MFMA_F32_HALVES)),
    (("f32", 20, 64, 1000), {}, (F32, 2, 16, 0, capi.LA_PLAN_MERGE_MFMA_F32_HALVES)),
    (("f32", 128, 32, 100), {}, (F32, 8, 16, 0, capi.LA_PLAN_MERGE_MFMA_F32)),
    (("f32", 128, 4, 1000), {"kernel_variant": 1}, (VALU, 128, 1, 0, capi.LA_PLAN_MERGE_MFMA_F32)),
])
def test_plan_names_the_kernels(cuda, args, kw, want):
    import torch

    if torch.cuda.get_device_properties(cuda).multi_processor_count != 256:
        pytest.skip("the sizes are of 256 CUs")
    i = plan(*args, **kw)
    assert (i.attention, i.head_groups, i.heads_per_workgroup, i.filled_rows, i.merge) == want
    assert i.absorb == (capi.LA_PLAN_ABSORB_MFMA_F32 if args[0] == "f32" else capi.LA_PLAN_ABSORB_MFMA_QPREP)


@pytest.mark.parametrize("heads,num_seqs,seq_len,filled", [
    (128, 200, 5368704, 0),  # 1,024 chunks of 2^20 rows: 824 pieces would hold 1.24 times that each
    (128, 16, 67108832, 0),  # 1,008 pieces, still more than 2^20 rows each
    (128, 32, 1048576, 1),   # 256 chunks of 131,072 rows, pieces of at most 149,824
])
def test_filled_pieces_stay_within_the_kernels_chunk_length(cuda, heads, num_seqs, seq_len, filled):
    """Every sequence full, the pieces of filled rows are up to num_chunks / (num_chunks - num_seqs)
    times the plan's chunks: a plan whose pieces could pass 2^20 rows keeps its chunks of the regions."""
    i = plan("fp8", heads, num_seqs, seq_len, rope_rows=8192, **LENS)
    assert i.attention == MFMA and i.filled_rows == filled and i.num_chunks >= 4 * num_seqs
    if filled:
        n = i.num_chunks - num_seqs
        assert (num_seqs * seq_len + n - 1) // n <= 1 << 20


@pytest.mark.parametrize("heads,seq_len", [(1, 100000), (3, 50000), (16, 100000), (128, 1000)])
def test_float32_workspace_serves_any_alignment(cuda, heads, seq_len):
    """Alignment decides which float32 kernel runs; a workspace sized with one set of pointers holds
    the step over any other."""
    size = lambda **kw: capi.load().la_mla_decode_workspace_size(ctypes.byref(plan_args("f32", heads, 1, seq_len, **kw)))
    valu, mfma = size(kernel_variant=1), size()
    assert plan("f32", heads, 1, seq_len).attention == F32
    assert valu <= mfma
    for name in ("kv_cache", "q_rope", "rope_cos", "rope_sin", "workspace"):
        kw = {name: 0x10004}
        assert plan("f32", heads, 1, seq_len, **kw).attention == VALU
        assert size(**kw) == mfma == plan("f32", heads, 1, seq_len, **kw).workspace_bytes


@pytest.mark.parametrize("dtype", ["bf16", "fp8"])
@pytest.mark.parametrize("num_seqs,seq_len,heads,want", [
    (1, 8192, 16, 128), (1, 32768, 16, 256), (1, 131072, 16, 256), (2, 32768, 16, 256), (3, 32768, 16, 384),
    (4, 32768, 16, 512), (32, 4099, 16, 483), (1, 32768, 32, 256),
])
def test_few_heads_keep_the_slots_of_a_sequence_few(cuda, dtype, num_seqs, seq_len, heads, want):
    """Two chunks per CU at 16 heads, but no more than 128 per sequence while one per CU remains: the
    merge of a query row reads a slot per chunk in a few workgroups."""
    import torch

    if torch.cuda.get_device_properties(cuda).multi_processor_count != 256:
        pytest.skip("the counts are of 256 CUs")
    i = plan(dtype, heads, num_seqs, seq_len)
    assert (i.num_chunks, i.heads_per_workgroup) == (want, 16)


@pytest.mark.parametrize("dtype,heads,num_seqs,seq_len,want", [
    ("bf16", 16, 64, 8192, 16), ("bf16", 32, 32, 4099, 16), ("f16", 32, 30, 8000, 16), ("f16", 32, 30, 8001, 128),
    ("bf16", 32, 1, 200000, 16), ("bf16", 32, 1, 200001, 128), ("fp8", 32, 64, 8192, 16),
    ("bf16", 48, 1, 8192, 16), ("bf16", 48, 32, 4099, 128),
])
def test_few_heads_over_large_caches(cuda, dtype, heads, num_seqs, seq_len, want):
    """32 heads leave the 16-head kernel where their 16-bit cache outgrows the infinity cache."""
    i = plan(dtype, heads, num_seqs, seq_len)
    assert i.attention == MFMA and i.heads_per_workgroup == want
    if heads == 32:  # with lengths only the device knows how many rows stream
        assert plan(dtype, heads, num_seqs, seq_len, **LENS).heads_per_workgroup == 16
        assert plan(dtype, heads, num_seqs, seq_len, chunk_rows=512, **LENS).heads_per_workgroup == want


@pytest.mark.parametrize("heads,num_seqs,seq_len,kw,filled", [
    (128, 32, 512, {}, 0),                          # chunks of 128 rows end with the regions: the pieces are the same
    (128, 32, 512, {"seq_offsets": 0x10000}, 1),    # regions of any length
    (128, 32, 520, {}, 1),                          # chunks across regions
    (128, 16, 8192, {}, 1),                         # 512-row chunks, pieces down to 128
    (16, 32, 1024, {}, 0), (16, 32, 2048, {}, 1),   # 64-row and 128-row chunks of the 16-head kernel
])
def test_filled_rows_are_cut_where_that_makes_other_pieces(cuda, heads, num_seqs, seq_len, kw, filled):
    import torch

    if torch.cuda.get_device_properties(cuda).multi_processor_count != 256:
        pytest.skip("the sizes are of 256 CUs")
    i = plan("bf16", heads, num_seqs, seq_len, **LENS, **kw)
    assert i.num_chunks >= 4 * num_seqs and i.filled_rows == filled
