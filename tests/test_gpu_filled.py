"""Decode with per-sequence lengths: the MFMA kernels' chunks share the filled
rows, found on the device (seq_in_plan / ChunkWalk, csrc/la_internal.hpp).
More sequences than a wave has lanes, empty ones, lengths around the padding
of 32, one long sequence among short ones, pieces longer than the shortest,
over capacity, packed and paged caches, against the float64 oracle over the
filled rows; unfilled rows hold values that would dominate any softmax. The
plan says that the pieces are of filled rows."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import assert_close
from mla_cases import TORCH_DTYPE, cfg_with_heads, make_queries, make_weights, rope, to_np
from oracle import mla_oracle as mo
from test_gpu_plan import plan

pytestmark = pytest.mark.gpu


SHORT = [0, 31, 32, 33, 0, 200, 64]  # a leading and a middle empty sequence
MANY = [0, 31, 32, 33, 1, 0, 200] + [5, 64] * 33  # 73: more than a wave has lanes (at 128 heads never: 256 chunks)
ALL = [("bf16", 128), ("fp8", 128), ("f16", 16), ("f32", 16)]
CASES = [(lens, cap, dt, heads) for lens, cap, kinds in [
    (SHORT, 544, ALL), (MANY, 544, ALL[2:]), ([0] * 3, 544, ALL), ([3000, 1, 40], 3040, ALL), ([2001], 3040, ALL),
    ([10016, 9000, 10016, 9999], 10016, ALL[:3]),  # nearly full: pieces longer than the plan's shortest
] for dt, heads in kinds]


@pytest.mark.parametrize("layout", ["capacity", "packed", "paged"])
@pytest.mark.parametrize("lens,cap,dtype,heads", CASES)
def test_filled_rows(cuda, layout, dtype, heads, lens, cap):
    from latent_attn import functional as F

    cfg = cfg_with_heads(heads)
    B, bs = len(lens), 32
    if torch.cuda.get_device_properties(cuda).multi_processor_count == 256:  # the sizes are of 256 CUs
        i = plan(dtype, heads, B, 0 if layout == "paged" else cap, total_rows=B * cap, seq_lens=0x10000, **{
            "capacity": {}, "packed": {"seq_offsets": 0x10000},
            "paged": {"block_table": 0x10000, "block_size": bs, "blocks_per_seq": cap // bs}}[layout])
        assert i.filled_rows == 1 and i.num_chunks >= 4 * B
    wt = {"fp8": "bf16"}.get(dtype, dtype)
    dt = torch.float8_e4m3fn if dtype == "fp8" else TORCH_DTYPE[dtype]
    W_UK, W_UV = make_weights(cfg, wt, 3, cuda)
    q_nope, q_rope = make_queries((B,), cfg, 4, cuda)
    cos, sin = rope(cap, cfg, cuda)
    g = torch.Generator().manual_seed(5)
    seqs = [torch.randn(n, 576, generator=g).to(dt) for n in lens]
    rows = torch.full((B * cap, 576), 96.0).to(dt).view(torch.uint8)
    for b, s in enumerate(seqs):
        rows[b * cap:b * cap + len(s)] = s.view(torch.uint8)
    len_t = torch.tensor(lens, dtype=torch.int32, device=cuda)
    args = (q_nope, q_rope, W_UK, W_UV, cos, sin, cfg)
    if layout == "capacity":
        out = F.mla_decode(rows.view(dt).to(cuda).view(B, cap, 576), *args, seq_lens=len_t)
    elif layout == "packed":
        off = torch.arange(B + 1, dtype=torch.int32, device=cuda) * cap
        out = F.mla_decode(rows.view(dt).to(cuda), *args, seq_offsets=off, seq_lens=len_t)
    else:
        table = torch.randperm(B * cap // bs, generator=g)
        pool = torch.empty_like(rows).view(-1, bs, rows.size(1))
        pool[table] = rows.view(-1, bs, rows.size(1))
        out = F.mla_decode(pool.view(-1, rows.size(1)).view(dt).to(cuda), *args, seq_lens=len_t,
                           block_table=table.to(torch.int32).view(B, -1).to(cuda), block_size=bs)
    d = mo.Dims(cfg.d_model, 512, 128, 64, heads, 128)
    qa = mo.absorb_q(to_np(q_nope), to_np(W_UK), d)
    off_np = np.concatenate([[0], np.cumsum(lens)]).tolist()
    packed = np.concatenate([to_np(s).reshape(-1, 576) for s in seqs])
    ref = mo.decode_sequences(packed, off_np, qa, to_np(q_rope), to_np(W_UV), to_np(cos), to_np(sin), d)
    if not any(lens):
        assert torch.count_nonzero(out).item() == 0
        return
    assert_close(out.cpu().numpy(), ref, wt, f"filled {layout} {dtype} H={heads} B={B}")


@pytest.mark.parametrize("heads,dtype", [(128, "bf16"), (16, "bf16"), (128, "f32")])
def test_workspace_serves_a_batch_with_and_without_lengths(cuda, heads, dtype):
    """A workspace sized for whole regions holds the same batch with lengths, contiguous and paged (host only)."""
    import ctypes

    from latent_attn import capi

    lib = capi.load()
    a = capi.DecodeArgs()
    fake = 0x10000
    code = {"bf16": capi.LA_DTYPE_BF16, "f32": capi.LA_DTYPE_F32}[dtype]
    a.kv_cache = a.q_nope = a.W_UK = a.q_rope = a.W_UV = a.rope_cos = a.rope_sin = a.output = fake
    a.kv_dtype = a.w_uk_dtype = a.w_uv_dtype = code
    a.num_seqs, a.seq_len, a.queries_per_seq, a.total_rows = 32, 8192, 1, 32 * 8192
    a.cfg = capi.config(cfg_with_heads(heads))
    whole = lib.la_mla_decode_workspace_size(ctypes.byref(a))
    a.seq_lens = fake
    assert 0 < lib.la_mla_decode_workspace_size(ctypes.byref(a)) <= whole
    a.seq_len, a.block_table, a.block_size, a.blocks_per_seq = 0, fake, 64, 128
    assert 0 < lib.la_mla_decode_workspace_size(ctypes.byref(a)) <= whole
