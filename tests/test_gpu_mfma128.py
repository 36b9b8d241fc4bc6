"""The 128-head MFMA attention kernel (decode_mfma_kernel, csrc/la_mfma.hip) at
its edges, at sizes whose plan takes it: more than two 16-head workgroups per
CU (with fewer the step runs decode_mfma16_kernel). Split points that cut
tiles and sequences, empty and short sequences, chunks under a tile, paged
blocks of 1 to 8 tiles, partial head groups and the lazily raised maximum,
against the float64 oracle."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from conftest import assert_close
from mla_cases import TORCH_DTYPE, cfg_with_heads, make_queries, make_weights, rope, staircase_case, to_np
from oracle import mla_oracle as mo
from test_gpu_plan import plan

from latent_attn import capi
from latent_attn import functional as F

pytestmark = pytest.mark.gpu

ROW = 576


def _dims(heads):
    return mo.Dims(5120, 512, 128, 64, heads, 128)


def _reaches(*args, **kw):
    i = plan(*args, **kw)
    assert (i.attention, i.heads_per_workgroup) == (capi.LA_PLAN_ATTENTION_MFMA, 128), (args, kw)


def _cache(rows, dtype, seed, cuda):
    g = torch.Generator(device=cuda).manual_seed(seed)
    dt = torch.float8_e4m3fn if dtype == "fp8" else TORCH_DTYPE[dtype]
    return torch.randn(rows, ROW, generator=g, device=cuda).to(dt)


def _check(out, kv, offs, q_nope, q_rope, W_UK, W_UV, cos, sin, heads, dtype, what, picks=None):
    """Sequences `picks` (all by default) of rows offs[s] .. offs[s + 1] of kv."""
    d = _dims(heads)
    qa = mo.absorb_q(to_np(q_nope), to_np(W_UK), d)
    for s in range(len(offs) - 1) if picks is None else picks:
        rows = to_np(kv[int(offs[s]):int(offs[s + 1])].float())
        ref = mo.decode_sequences(rows, [0, len(rows)], qa[s:s + 1], to_np(q_rope[s:s + 1]), to_np(W_UV), to_np(cos),
                                  to_np(sin), d)
        if len(rows) == 0:
            assert torch.count_nonzero(out[s]).item() == 0
        else:
            assert_close(out[s:s + 1].cpu().numpy(), ref, "bf16" if dtype == "fp8" else dtype, f"{what} seq {s}")


@pytest.mark.parametrize("B,S,chunk,picks", [(2, 1100, 32, None), (4, 1600, 96, None), (4, 1700, 100, None),
                                             (4, 12700, 777, (0, 3)), (66, 3001, 3000, (0, 31, 65))])
def test_split_invariance(cuda, B, S, chunk, picks):
    _reaches("bf16", 128, B, S, chunk_rows=chunk)
    cfg = cfg_with_heads(128)
    kv = _cache(B * S, "bf16", 21, cuda)
    W_UK, W_UV = make_weights(cfg, "bf16", 22, cuda)
    q_nope, q_rope = make_queries((B,), cfg, 23, cuda)
    cos, sin = rope(S, cfg, cuda)
    out = F.mla_decode(kv.view(B, S, ROW), q_nope, q_rope, W_UK, W_UV, cos, sin, cfg, chunk_rows=chunk)
    _check(out, kv, [b * S for b in range(B + 1)], q_nope, q_rope, W_UK, W_UV, cos, sin, 128, "bf16", f"chunk {chunk}",
           picks)


@pytest.mark.parametrize("dtype", ["bf16", "f16", "fp8"])
@pytest.mark.parametrize("lens,chunk", [([5, 0, 1, 33, 700, 31, 64, 2049], 32), ([5, 0, 1, 33, 700, 31, 64, 2049] * 6, 256),
                                        ([400, 137], 7), ([70], 1)])
def test_ragged_and_short_chunks(cuda, dtype, lens, chunk):
    B, T = len(lens), sum(lens)
    _reaches(dtype, 128, B, 0, seq_offsets=0x10000, total_rows=T, chunk_rows=chunk)
    cfg = cfg_with_heads(128)
    kv = _cache(T, dtype, 31, cuda)
    W_UK, W_UV = make_weights(cfg, "f16" if dtype == "f16" else "bf16", 32, cuda)
    q_nope, q_rope = make_queries((B,), cfg, 33, cuda)
    cos, sin = rope(max(lens), cfg, cuda)
    offs = np.concatenate([[0], np.cumsum(lens)])
    out = F.mla_decode(kv, q_nope, q_rope, W_UK, W_UV, cos, sin, cfg, chunk_rows=chunk,
                       seq_offsets=torch.tensor(offs, dtype=torch.int32, device=cuda))
    _check(out, kv, offs, q_nope, q_rope, W_UK, W_UV, cos, sin, 128, dtype, f"ragged {dtype} chunk {chunk}")


# blocks of 1, 2, 3, 5 and 8 tiles: the divide by tiles per block. Chunks of 128 rows, and (0) pieces of filled rows
@pytest.mark.parametrize("dtype", ["bf16", "f16", "fp8"])
@pytest.mark.parametrize("bs", [32, 64, 96, 160, 256])
@pytest.mark.parametrize("chunk", [128, 0])
def test_paged_equals_contiguous(cuda, bs, dtype, chunk):
    cap = -(-2400 // bs) * bs
    lens0 = [cap, 1, 1700, 0, 33, cap]
    B = len(lens0)
    kw = {"seq_lens": 0x10000, "chunk_rows": chunk}
    _reaches(dtype, 128, B, cap, **kw)
    _reaches(dtype, 128, B, 0, total_rows=B * cap, block_table=0x10000, block_size=bs, blocks_per_seq=cap // bs, **kw)
    assert plan(dtype, 128, B, cap, **kw).filled_rows == (chunk == 0 and cap % 128 != 0)
    cfg = cfg_with_heads(128)
    cache = _cache(B * cap, dtype, 51, cuda)
    table = torch.randperm(B * cap // bs, generator=torch.Generator().manual_seed(52))
    pool = torch.empty_like(cache)
    pool.view(torch.uint8).view(-1, bs, pool.view(torch.uint8).size(1))[table.to(cuda)] = \
        cache.view(torch.uint8).view(-1, bs, pool.view(torch.uint8).size(1))
    lens = torch.tensor(lens0, dtype=torch.int32, device=cuda)
    W_UK, W_UV = make_weights(cfg, "f16" if dtype == "f16" else "bf16", 53, cuda)
    q_nope, q_rope = make_queries((B,), cfg, 54, cuda)
    cos, sin = rope(cap, cfg, cuda)
    args = (q_nope, q_rope, W_UK, W_UV, cos, sin, cfg)
    out_c = F.mla_decode(cache.view(B, cap, ROW), *args, seq_lens=lens, chunk_rows=chunk)
    out_p = F.mla_decode(pool, *args, seq_lens=lens, chunk_rows=chunk, block_table=table.to(torch.int32).view(B, -1).to(cuda),
                         block_size=bs)
    assert torch.equal(out_p, out_c), float((out_p - out_c).abs().max())
    filled = torch.cat([cache[b * cap:b * cap + n] for b, n in enumerate(lens0) if n], 0) if dtype != "fp8" else \
        torch.cat([cache.view(torch.uint8)[b * cap:b * cap + n] for b, n in enumerate(lens0)], 0).view(torch.float8_e4m3fn)
    _check(out_p, filled, np.concatenate([[0], np.cumsum(lens0)]), q_nope, q_rope, W_UK, W_UV, cos, sin, 128, dtype,
           f"paged {dtype} bs {bs}", picks=(1, 2, 3, 4, 5))


@pytest.mark.parametrize("paged", [False, True])
def test_fp8_equals_its_bf16_copy(cuda, paged):
    """The rows expand to bf16 exactly, and the rest of the path is the same."""
    B, cap, bs, chunk = 3, 3072, 96, 128
    for dt in ("fp8", "bf16"):
        _reaches(dt, 128, B, cap, wdtype="bf16", seq_lens=0x10000, chunk_rows=chunk)
    cfg = cfg_with_heads(128)
    kv = _cache(B * cap, "fp8", 111, cuda)
    lens = torch.tensor([cap, 77, 2300], dtype=torch.int32, device=cuda)
    W_UK, W_UV = make_weights(cfg, "bf16", 112, cuda)
    q_nope, q_rope = make_queries((B,), cfg, 113, cuda)
    cos, sin = rope(cap, cfg, cuda)
    kw = dict(seq_lens=lens, chunk_rows=chunk)
    args = (q_nope, q_rope, W_UK, W_UV, cos, sin, cfg)
    want = F.mla_decode(kv.to(torch.bfloat16).view(B, cap, ROW), *args, **kw)
    if paged:
        perm = torch.randperm(B * cap // bs, generator=torch.Generator().manual_seed(114)).to(cuda)
        pool = torch.empty_like(kv)
        pool.view(torch.uint8).view(-1, bs, ROW)[perm] = kv.view(torch.uint8).view(-1, bs, ROW)
        got = F.mla_decode(pool, *args, block_table=perm.to(torch.int32).view(B, -1), block_size=bs, **kw)
    else:
        got = F.mla_decode(kv.view(B, cap, ROW), *args, **kw)
    assert torch.equal(got, want), float((got - want).abs().max())


# 48, 64, 112 and 144 (48 x 3) query heads leave partial groups of 128, 256 two whole ones
@pytest.mark.parametrize("heads,qps,lens,chunk", [
    (48, 1, [2570, 3000, 64], 32), (48, 3, [257, 4000, 64], 64), (64, 1, [1000, 3200, 33], 32), (112, 1, [2401], 32),
    (128, 2, [2000, 300, 70], 64)])
def test_partial_head_groups(cuda, heads, qps, lens, chunk):
    B, T = len(lens), sum(lens)
    _reaches("bf16", heads, B, 0, qps, seq_offsets=0x10000, total_rows=T, chunk_rows=chunk)
    lib, cfg, d = capi.load(), cfg_with_heads(heads), _dims(heads)
    kv = _cache(T, "bf16", 71, cuda)
    W_UK, W_UV = make_weights(cfg, "bf16", 72, cuda)
    q_nope, q_rope = make_queries((B * qps,), cfg, 73, cuda)
    cos, sin = rope(max(lens), cfg, cuda)
    offs = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    off_t = torch.tensor(offs, device=cuda)
    out = torch.full((B * qps, heads, 128), float("nan"), device=cuda)
    a = capi.DecodeArgs()
    a.kv_cache, a.kv_dtype, a.total_rows, a.num_seqs = kv.data_ptr(), capi.LA_DTYPE_BF16, T, B
    a.seq_offsets, a.queries_per_seq, a.chunk_rows = off_t.data_ptr(), qps, chunk
    a.q_nope, a.W_UK, a.w_uk_dtype = q_nope.data_ptr(), W_UK.data_ptr(), capi.LA_DTYPE_BF16
    a.q_rope, a.W_UV, a.w_uv_dtype = q_rope.data_ptr(), W_UV.data_ptr(), capi.LA_DTYPE_BF16
    a.rope_cos, a.rope_sin, a.rope_rows = cos.data_ptr(), sin.data_ptr(), cos.shape[0]
    a.output, a.cfg = out.data_ptr(), capi.config(cfg)
    ws = torch.empty(lib.la_mla_decode_workspace_size(ctypes.byref(a)), dtype=torch.uint8, device=cuda)
    a.workspace, a.workspace_bytes = ws.data_ptr(), ws.numel()
    st = lib.la_mla_decode(ctypes.byref(a), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert st == capi.LA_SUCCESS, lib.la_status_string(st).decode()
    torch.cuda.synchronize()
    qa = mo.absorb_q(to_np(q_nope), to_np(W_UK), d)
    ref = np.zeros((B * qps, heads, 128))
    for t in range(B * qps):
        s = t // qps
        ref[t:t + 1] = mo.decode_sequences(to_np(kv[offs[s]:offs[s + 1]]), [0, lens[s]], qa[t:t + 1],
                                           to_np(q_rope[t:t + 1]), to_np(W_UV), to_np(cos), to_np(sin), d)
    assert_close(out.cpu().numpy(), ref, "bf16", f"{heads} heads x {qps} queries")


# The lazily raised maximum in chunks of 32 and 10 tiles (tests/test_rescale_inputs.py walks the same segments)
@pytest.mark.parametrize("dtype", ["bf16", "f16", "fp8"])
@pytest.mark.parametrize("paged", [False, True])
@pytest.mark.parametrize("B,chunk", [(24, 1024), (7, 320)])
def test_rescale(cuda, dtype, paged, B, chunk):
    S, cap, bs, picks = 3000, 3072, 96, (0, B // 2, B - 1)
    _reaches(dtype, 128, B, cap if paged else S, chunk_rows=chunk, **({"seq_lens": 0x10000} if paged else {}))
    cfg = cfg_with_heads(128)
    kv, qa, qr = staircase_case(B, S, "f16" if dtype == "f16" else "bf16", 5, cuda)
    if dtype == "fp8":  # the staircase halved (exact in E4M3) and the query weights on it doubled
        kv, qa = (kv.float() * 0.5).to(torch.float8_e4m3fn), qa.clone()
        qa[:, :, 0:2] *= 2.0
    _, W_UV = make_weights(cfg, "f16" if dtype == "f16" else "bf16", 6, cuda)
    cos, sin = rope(cap, cfg, cuda)
    args = (qa, qr, W_UV, cos, sin, cfg)
    if paged:
        u8 = kv.view(torch.uint8)
        full = torch.zeros(B, cap, u8.size(-1), dtype=torch.uint8, device=cuda)
        full[:, :S] = u8
        perm = torch.randperm(B * cap // bs, generator=torch.Generator().manual_seed(9)).to(cuda)
        pool = torch.empty_like(full).view(-1, bs, u8.size(-1))
        pool[perm] = full.view(-1, bs, u8.size(-1))
        out = F.mla_decode_absorbed(pool.view(-1, u8.size(-1)).view(kv.dtype), *args, chunk_rows=chunk,
                                    seq_lens=torch.full((B,), S, dtype=torch.int32, device=cuda),
                                    block_table=perm.to(torch.int32).view(B, -1), block_size=bs)
    else:
        out = F.mla_decode_absorbed(kv, *args, chunk_rows=chunk)
    for b in picks:
        ref = mo.decode_sequences(to_np(kv[b].float()), [0, S], to_np(qa[b:b + 1]), to_np(qr[b:b + 1]), to_np(W_UV),
                                  to_np(cos)[:S], to_np(sin)[:S], _dims(128))
        assert_close(out[b:b + 1].cpu().numpy(), ref, "f16" if dtype == "f16" else "bf16",
                     f"rescale {dtype} chunk {chunk} paged {paged} seq {b}")
