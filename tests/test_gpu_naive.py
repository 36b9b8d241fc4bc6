"""naive_mla on the matrix cores (csrc/la_naive.hip) at the edges of its
256-position workgroups and 8-head groups, against the float64 oracle at the
fp32 tolerance (products of 16-bit values are exact, sums are fp32)."""

from __future__ import annotations

import pytest
import torch

from conftest import assert_close
from mla_cases import cfg_with_heads, make_cache, make_queries, make_weights, rope, to_np
from oracle import mla_oracle as mo

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S,heads", [(1, 1), (63, 9), (255, 3), (256, 16), (257, 8), (700, 17)])
@pytest.mark.parametrize("dtype,wdtype", [("bf16", "bf16"), ("f16", "f16"), ("bf16", "f16")])
def test_naive_edges(cuda, S, heads, dtype, wdtype):
    from latent_attn import functional as F

    cfg = cfg_with_heads(heads)
    kv = make_cache((S,), cfg, dtype, 1, cuda)
    W_UK, W_UV = make_weights(cfg, wdtype, 2, cuda)
    q_nope, q_rope = make_queries((), cfg, 3, cuda)
    cos, sin = rope(S, cfg, cuda)
    out = F.naive_mla(kv, W_UK, W_UV, q_nope, q_rope, cos, sin, cfg)
    torch.cuda.synchronize()
    d = mo.Dims(cfg.d_model, 512, 128, 64, heads, 128)
    ref = mo.naive_mla(to_np(kv), to_np(W_UK), to_np(W_UV), to_np(q_nope), to_np(q_rope), to_np(cos), to_np(sin), d)
    assert_close(out.cpu().numpy(), ref, "f32", f"naive {dtype}/{wdtype} S={S} H={heads}")
