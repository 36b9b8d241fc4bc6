"""The 16-head MFMA attention kernel (csrc/la_mfma16.hip) at the edges of its
tiles (16 rows per wave, 64 or 128 positions), over every cache layout and
type it serves, against the float64 oracle. Up to 32 query heads take it (32
over 16-bit caches within the infinity cache); more do while its workgroups
fill the chip at most twice."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import assert_close
from mla_cases import TORCH_DTYPE, cfg_with_heads, make_queries, make_weights, rope, staircase_case, to_np
from oracle import mla_oracle as mo
from test_gpu_plan import MFMA, plan

pytestmark = pytest.mark.gpu


def _ref(cfg, seqs, q_abs, q_rope, W_UV, cos, sin):
    d = mo.Dims(cfg.d_model, 512, 128, 64, cfg.num_heads, 128)
    off = np.concatenate([[0], np.cumsum([len(s) for s in seqs])]).tolist()
    return mo.decode_sequences(np.concatenate([to_np(s) for s in seqs]), off, q_abs, to_np(q_rope), to_np(W_UV),
                               to_np(cos), to_np(sin), d)


# lengths: one row, around a wave's 16 rows, around one and two tiles; chunks
# of 64 rows (several slots and tiles cut short), and one chunk
@pytest.mark.parametrize("layout", ["ragged", "paged"])
@pytest.mark.parametrize("dtype", ["bf16", "f16", "fp8"])
@pytest.mark.parametrize("heads,chunk", [(16, 0), (32, 64), (48, 128), (128, 0), (16, 512)])
def test_edges(cuda, layout, dtype, heads, chunk):
    from latent_attn import functional as F

    cfg = cfg_with_heads(heads)
    lens = [1, 15, 16, 17, 63, 64, 65, 0, 127, 128, 129, 200]
    B, bs, per = len(lens), 32, 8
    where = {"ragged": dict(seq_offsets=0x10000, total_rows=sum(lens)),
             "paged": dict(seq_lens=0x10000, block_table=0x10000, block_size=bs, blocks_per_seq=per, total_rows=B * per * bs)}
    i = plan(dtype, heads, B, 0, chunk_rows=chunk, kernel_variant=2, **where[layout])
    assert (i.attention, i.heads_per_workgroup) == (MFMA, 16)
    wt = "f16" if dtype == "f16" else "bf16"
    W_UK, W_UV = make_weights(cfg, wt, 3, cuda)
    q_nope, q_rope = make_queries((B,), cfg, 4, cuda)
    cos, sin = rope(max(lens), cfg, cuda)
    g = torch.Generator().manual_seed(5)
    dt = torch.float8_e4m3fn if dtype == "fp8" else TORCH_DTYPE[dtype]
    seqs = [torch.randn(n, 576, generator=g).to(dt) for n in lens]
    if layout == "ragged":
        off = torch.tensor(np.concatenate([[0], np.cumsum(lens)]), dtype=torch.int32, device=cuda)
        out = F.mla_decode(torch.cat([s.view(torch.uint8) for s in seqs]).view(dt).to(cuda), q_nope, q_rope, W_UK, W_UV,
                           cos, sin, cfg, seq_offsets=off, chunk_rows=chunk, kernel_variant=2)
    else:
        table = torch.randperm(B * per, generator=g).to(torch.int32).view(B, per)
        pool = torch.full((B * per, bs, 576), 96.0).to(dt)  # unfilled rows would show
        for b, s in enumerate(seqs):
            for p in range(0, len(s), bs):
                n = min(bs, len(s) - p)
                pool.view(torch.uint8)[table[b, p // bs], :n] = s[p:p + n].view(torch.uint8)
        out = F.mla_decode(pool.view(-1, 576).to(cuda), q_nope, q_rope, W_UK, W_UV, cos, sin, cfg, chunk_rows=chunk,
                           kernel_variant=2, seq_lens=torch.tensor(lens, dtype=torch.int32, device=cuda),
                           block_table=table.to(cuda), block_size=bs)
    d = mo.Dims(cfg.d_model, 512, 128, 64, heads, 128)
    ref = _ref(cfg, seqs, mo.absorb_q(to_np(q_nope), to_np(W_UK), d), q_rope, W_UV, cos, sin)
    assert_close(out.cpu().numpy(), ref, wt, f"mfma16 {layout} {dtype} H={heads} chunk {chunk}")


@pytest.mark.parametrize("chunk", [0, 256])
def test_rising_maximum(cuda, chunk):
    """Running maxima that rise from tile to tile, at other tiles for other heads (O is rescaled)."""
    from latent_attn import functional as F

    cfg = cfg_with_heads(128)
    assert plan("bf16", 128, 1, 700, chunk_rows=chunk, kernel_variant=2).heads_per_workgroup == 16
    kv, qa, qr = staircase_case(1, 700, "bf16", 6, cuda)
    _, W_UV = make_weights(cfg, "bf16", 7, cuda)
    cos, sin = rope(700, cfg, cuda)
    out = F.mla_decode_absorbed(kv, qa, qr, W_UV, cos, sin, cfg, chunk_rows=chunk, kernel_variant=2)
    ref = _ref(cfg, [kv[0].cpu()], to_np(qa), qr, W_UV, cos, sin)
    assert_close(out.cpu().numpy(), ref, "bf16", f"mfma16 rising maximum, chunk {chunk}")
