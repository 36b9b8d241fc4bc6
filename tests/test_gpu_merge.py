"""The half-row merge (merge_project_half_kernel, csrc/la_proj.hip) at the edges
of its rules: query rows around 8 and 16 per workgroup, slots around 8, 16 and
32 per task, against the float64 oracle."""

from __future__ import annotations

import pytest
import torch

from conftest import assert_close
from mla_cases import cfg_with_heads, make_cache, make_queries, make_weights, rope, to_np
from oracle import mla_oracle as mo
from test_gpu_plan import plan

from latent_attn import capi
from latent_attn import functional as F

pytestmark = pytest.mark.gpu


# heads, sequences (one query row each), rows per sequence, rows per chunk
@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("heads,B,S,chunk", [
    (128, 8, 256, 32), (128, 9, 256, 32), (128, 12, 70, 32), (128, 15, 250, 64), (128, 16, 256, 32),  # 16 rows, <= 8 slots
    (48, 17, 96, 32), (48, 64, 160, 64), (16, 130, 96, 32),  # with a last block of 1, 16 and 2 rows
    (128, 9, 288, 32), (128, 16, 512, 32), (128, 16, 544, 32), (128, 3, 1000, 16),  # more slots: 8 rows, or waves per row
    (128, 8, 544, 32), (128, 16, 1056, 32),  # one and two workgroups per CU: batches of 32 and of 16
    (128, 9, 1056, 32), (128, 12, 288, 32), (128, 13, 544, 32), (48, 24, 850, 50),  # room for seven, four, three rows
])
def test_rows_and_slots(cuda, dtype, heads, B, S, chunk):
    if torch.cuda.get_device_properties(cuda).multi_processor_count == 256:
        assert plan(dtype, heads, B, S, chunk_rows=chunk).merge == capi.LA_PLAN_MERGE_MFMA_HALVES
    cfg = cfg_with_heads(heads)
    kv = make_cache((B, S), cfg, dtype, 61, cuda)
    W_UK, W_UV = make_weights(cfg, dtype, 62, cuda)
    q_nope, q_rope = make_queries((B,), cfg, 63, cuda)
    cos, sin = rope(S, cfg, cuda)
    out = F.mla_decode(kv, q_nope, q_rope, W_UK, W_UV, cos, sin, cfg, chunk_rows=chunk).cpu().numpy()
    d = mo.Dims(cfg.d_model, 512, 128, 64, heads, 128)
    ref = mo.decode_sequences(to_np(kv).reshape(B * S, 576), [b * S for b in range(B + 1)],
                              mo.absorb_q(to_np(q_nope), to_np(W_UK), d), to_np(q_rope), to_np(W_UV), to_np(cos),
                              to_np(sin), d)
    assert_close(out, ref, dtype, f"half merge H={heads} rows {B} chunks of {chunk} in {S}")
