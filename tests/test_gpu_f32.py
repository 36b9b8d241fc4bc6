"""The fp32 MFMA kernels (csrc/la_f32.hip, merge_project_f32_kernel) at their
edges: tiles of 32 positions, 8 rows per wave, 16 heads per workgroup, 16
query rows per merge, against the float64 oracle at the fp32 tolerance."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from conftest import assert_close
from mla_cases import TORCH_DTYPE, cfg_with_heads, make_queries, make_weights, rope, staircase_case, to_np
from oracle import mla_oracle as mo
from test_gpu_plan import F32, VALU, plan

from latent_attn import capi

pytestmark = pytest.mark.gpu


def _dims(cfg):
    return mo.Dims(cfg.d_model, 512, cfg.qk_nope_head_dim, 64, cfg.num_heads, 128)


@pytest.mark.parametrize("layout", ["ragged", "paged"])
@pytest.mark.parametrize("heads,chunk", [(1, 0), (16, 64), (20, 33), (32, 0)])
def test_edges(cuda, layout, heads, chunk):
    from latent_attn import functional as F

    cfg = cfg_with_heads(heads)
    lens = [1, 7, 8, 9, 31, 32, 33, 0, 63, 64, 65, 100, 5, 15, 16, 17, 40]  # 17 query rows: two merge blocks
    B, bs, per = len(lens), 32, 4
    where = {"ragged": dict(seq_offsets=0x10000, total_rows=sum(lens)),
             "paged": dict(seq_lens=0x10000, block_table=0x10000, block_size=bs, blocks_per_seq=per, total_rows=B * per * bs)}
    i = plan("f32", heads, B, 0, chunk_rows=chunk, **where[layout])
    assert (i.attention, i.heads_per_workgroup) == (F32, 16)
    assert i.merge in (capi.LA_PLAN_MERGE_MFMA_F32, capi.LA_PLAN_MERGE_MFMA_F32_HALVES)
    W_UK, W_UV = make_weights(cfg, "f32", 3, cuda)
    q_nope, q_rope = make_queries((B,), cfg, 4, cuda)
    cos, sin = rope(max(lens), cfg, cuda)
    g = torch.Generator().manual_seed(5)
    seqs = [torch.randn(n, 576, generator=g) for n in lens]
    if layout == "ragged":
        off = torch.tensor(np.concatenate([[0], np.cumsum(lens)]), dtype=torch.int32, device=cuda)
        out = F.mla_decode(torch.cat(seqs).to(cuda), q_nope, q_rope, W_UK, W_UV, cos, sin, cfg, seq_offsets=off,
                           chunk_rows=chunk)
    else:
        table = torch.randperm(B * per, generator=g).to(torch.int32).view(B, per)
        pool = torch.full((B * per, bs, 576), 96.0)  # unfilled rows would show
        for b, s in enumerate(seqs):
            for p in range(0, len(s), bs):
                pool[table[b, p // bs], :min(bs, len(s) - p)] = s[p:p + bs]
        out = F.mla_decode(pool.view(-1, 576).to(cuda), q_nope, q_rope, W_UK, W_UV, cos, sin, cfg, chunk_rows=chunk,
                           seq_lens=torch.tensor(lens, dtype=torch.int32, device=cuda), block_table=table.to(cuda),
                           block_size=bs)
    d = _dims(cfg)
    off_np = np.concatenate([[0], np.cumsum(lens)]).tolist()
    ref = mo.decode_sequences(to_np(torch.cat(seqs)), off_np, mo.absorb_q(to_np(q_nope), to_np(W_UK), d), to_np(q_rope),
                              to_np(W_UV), to_np(cos), to_np(sin), d)
    assert_close(out.cpu().numpy(), ref, "f32", f"f32 {layout} H={heads} chunk {chunk}")


def test_rising_maximum_and_shared_cache(cuda):
    """O rescaled as the maximum rises; absorbed queries; fp32 weights on both kinds of partial rows."""
    from latent_attn import functional as F

    cfg = cfg_with_heads(128)
    kv, qa, qr = staircase_case(1, 300, "f32", 6, cuda)
    _, W_UV = make_weights(cfg, "f32", 7, cuda)
    cos, sin = rope(300, cfg, cuda)
    d = _dims(cfg)
    args = (to_np(qa), to_np(qr), to_np(W_UV), to_np(cos), to_np(sin), d)
    out = F.fused_mla(kv[0], qa[0], qr[0], W_UV, cos, sin, cfg)
    ref = mo.decode_sequences(to_np(kv[0]), [0, 300], *args)
    assert_close(out.cpu().numpy()[None], ref, "f32", "f32 rising maximum")
    kv16 = kv[0].to(torch.bfloat16)
    out = F.fused_mla(kv16, qa[0], qr[0], W_UV, cos, sin, cfg)
    ref = mo.decode_sequences(to_np(kv16), [0, 300], *args)
    assert_close(out.cpu().numpy()[None], ref, "bf16", "bf16 cache, fp32 weights")


@pytest.mark.parametrize("tokens,dn", [(1, 128), (16, 128), (17, 128), (3, 16), (5, 144)])
def test_absorb(cuda, tokens, dn):
    from latent_attn import functional as F

    cfg = cfg_with_heads(3)
    cfg.qk_nope_head_dim = dn
    g = torch.Generator().manual_seed(8)
    q = torch.randn(tokens, 3, dn, generator=g)
    W = torch.randn(3 * dn, 512, generator=g)
    got = F.absorb_q(q.to(cuda), W.to(cuda), cfg)
    ref = np.einsum("thi,hic->thc", to_np(q), to_np(W).reshape(3, dn, 512))
    assert_close(got.cpu().numpy(), ref, "f32", f"absorb f32 tokens {tokens} dn {dn}")


@pytest.mark.parametrize("seq,heads", [(2048, 128), (4099, 16)])
def test_shared_cache_workspace(cuda, seq, heads):
    """The shared-cache entry points size their workspace for the fp32 kernel's chunks (more than the VALU kernel's)."""
    from latent_attn import functional as F

    cfg = cfg_with_heads(heads)
    _, W_UV = make_weights(cfg, "f32", 9, cuda)
    cos, sin = rope(seq, cfg, cuda)
    g = torch.Generator().manual_seed(10)
    kv = torch.randn(seq, 576, generator=g).to(cuda)
    qa = torch.randn(2, heads, 512, generator=g).to(cuda)
    qr = torch.randn(2, heads, 64, generator=g).to(cuda)
    out = F.batched_fused_mla(kv, qa, qr, W_UV, cos, sin, cfg).cpu().numpy()
    one = F.fused_mla(kv, qa[1], qr[1], W_UV, cos, sin, cfg).cpu().numpy()
    args = [to_np(x) for x in (W_UV, cos, sin)]
    for b in range(2):
        ref = mo.decode_sequences(to_np(kv), [0, seq], to_np(qa[b])[None], to_np(qr[b])[None], *args, _dims(cfg))
        assert_close(out[b][None], ref, "f32", f"f32 shared cache S={seq} H={heads} query {b}")
    assert_close(one[None], ref, "f32", f"f32 fused S={seq} H={heads}")


@pytest.mark.parametrize("shift", [0, 1])
def test_absorb_into_an_output_that_is_only_float_aligned(cuda, shift):
    """The MFMA absorption stores 16-byte vectors: an output without that alignment takes the VALU
    kernel, as a q_nope without it does (the same bits)."""
    lib, cfg = capi.load(), cfg_with_heads(3)
    g = torch.Generator().manual_seed(11)
    q = torch.randn(5 * 3 * 128, generator=g).to(cuda)
    W = torch.randn(3 * 128, 512, generator=g).to(cuda)
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)

    def absorb(q_shift, out_shift):
        buf = torch.empty(q.numel() + 4, device=cuda)
        buf[q_shift:q_shift + q.numel()] = q
        out = torch.full((5 * 3 * 512 + 4,), 7.0, device=cuda)
        c = capi.config(cfg)
        assert lib.la_absorb_q(buf.data_ptr() + 4 * q_shift, W.data_ptr(), capi.LA_DTYPE_F32,
                               out.data_ptr() + 4 * out_shift, 5, ctypes.byref(c), stream) == capi.LA_SUCCESS
        torch.cuda.synchronize()
        rest = torch.cat([out[:out_shift], out[out_shift + 5 * 3 * 512:]])
        assert torch.all(rest == 7.0)
        return out[out_shift:out_shift + 5 * 3 * 512]

    got, valu = absorb(0, shift), absorb(1, 0)
    assert torch.equal(got, valu) == bool(shift)  # the MFMA kernel sums in another order
    ref = np.einsum("thi,hic->thc", to_np(q).reshape(5, 3, 128), to_np(W).reshape(3, 128, 512))
    assert_close(got.cpu().numpy().reshape(5, 3, 512), ref, "f32", f"absorb f32, output shift {shift}")


@pytest.mark.parametrize("heads", [1, 16])
@pytest.mark.parametrize("shift", [0, 4])
def test_workspace_that_is_only_float_aligned(cuda, heads, shift):
    """A float32 step over a workspace without 16-byte alignment runs on the VALU kernels."""
    lib, cfg = capi.load(), cfg_with_heads(heads)
    B, S = 2, 300
    W_UK, W_UV = make_weights(cfg, "f32", 3, cuda)
    q_nope, q_rope = make_queries((B,), cfg, 4, cuda)
    cos, sin = rope(S, cfg, cuda)
    kv = torch.randn(B * S, 576, generator=torch.Generator().manual_seed(5)).to(cuda)
    out = torch.empty(B, heads, 128, device=cuda)
    a, info = capi.DecodeArgs(), capi.PlanInfo()
    a.kv_cache, a.kv_dtype, a.total_rows, a.num_seqs, a.seq_len = kv.data_ptr(), capi.LA_DTYPE_F32, B * S, B, S
    a.queries_per_seq, a.q_nope, a.W_UK, a.q_rope, a.W_UV = 1, q_nope.data_ptr(), W_UK.data_ptr(), q_rope.data_ptr(), W_UV.data_ptr()
    a.w_uk_dtype = a.w_uv_dtype = capi.LA_DTYPE_F32
    a.rope_cos, a.rope_sin, a.rope_rows, a.output = cos.data_ptr(), sin.data_ptr(), S, out.data_ptr()
    a.cfg = capi.config(cfg)
    a.workspace = 0x10000 + shift
    assert lib.la_mla_decode_plan(ctypes.byref(a), ctypes.byref(info)) == capi.LA_SUCCESS
    assert info.attention == (VALU if shift else F32)
    assert info.absorb == (capi.LA_PLAN_ABSORB_VALU if shift else capi.LA_PLAN_ABSORB_MFMA_F32)
    assert info.merge == (capi.LA_PLAN_MERGE_VALU if shift else capi.LA_PLAN_MERGE_MFMA_F32_HALVES)
    ws = torch.empty(info.workspace_bytes + 16, dtype=torch.uint8, device=cuda)
    a.workspace, a.workspace_bytes = ws.data_ptr() + shift, info.workspace_bytes
    assert lib.la_mla_decode(ctypes.byref(a), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
    torch.cuda.synchronize()
    d = _dims(cfg)
    ref = mo.decode_sequences(to_np(kv), [0, S, 2 * S], mo.absorb_q(to_np(q_nope), to_np(W_UK), d), to_np(q_rope),
                              to_np(W_UV), to_np(cos), to_np(sin), d)
    assert_close(out.cpu().numpy(), ref, "f32", f"f32 H={heads}, workspace + {shift} B")


@pytest.mark.parametrize("cache", ["f32", "bf16"])
@pytest.mark.parametrize("B,S", [(17, 70), (33, 40), (20, 300)])
def test_full_merge(cuda, cache, B, S):
    """float32 weights and enough query rows for the merge of both latent halves in one workgroup
    (two blocks of 16 rows or three, the last with one), over fp32 and fp16 partial rows."""
    from latent_attn import functional as F

    cfg = cfg_with_heads(128)
    if torch.cuda.get_device_properties(cuda).multi_processor_count == 256:
        assert plan(cache, 128, B, S, wdtype="f32", chunk_rows=64).merge == capi.LA_PLAN_MERGE_MFMA_F32
    W_UK, W_UV = make_weights(cfg, "f32", 21, cuda)
    q_nope, q_rope = make_queries((B,), cfg, 22, cuda)
    cos, sin = rope(S, cfg, cuda)
    kv = torch.randn(B, S, 576, generator=torch.Generator().manual_seed(23)).to(TORCH_DTYPE[cache]).to(cuda)
    out = F.mla_decode(kv, q_nope, q_rope, W_UK, W_UV, cos, sin, cfg, chunk_rows=64).cpu().numpy()
    d = _dims(cfg)
    ref = mo.decode_sequences(to_np(kv).reshape(B * S, 576), [b * S for b in range(B + 1)],
                              mo.absorb_q(to_np(q_nope), to_np(W_UK), d), to_np(q_rope), to_np(W_UV), to_np(cos),
                              to_np(sin), d)
    assert_close(out, ref, cache, f"full fp32 merge, {cache} cache, {B} rows")
