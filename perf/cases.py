"""Performance cases of the MLA decode library: the calls that programs make, over their range.

Each case is a dict of plain values whose ``kind`` names the public call it makes:

  fused    functional.fused_mla          one absorbed query over one cache
  batched  functional.batched_fused_mla  several absorbed queries over one shared cache
  decode   functional.mla_decode         one query per sequence, equal sequences
  ragged   functional.mla_decode         the same over a packed cache with sequence offsets
  serve    functional.append_kv + mla_decode: one step of a server over a paged cache
  fill     functional.append_kv          a prompt's rows written into the caches
  layer    LatentAttentionLayer.forward_batch: projections, attention, output projection
  naive    functional.naive_mla          decompress, then attend

Head dimensions are DeepSeek-V2's (latent 512, nope 128, rope 64, value 128); ``heads`` is 128, or
fewer where one GPU holds a share of them or a small model runs. Sizes are those of bench.py and of
the tests, and odd ones between. Inputs are normal, as there: weights with standard deviation
1/sqrt(512) (the layer's: its own initialisation), everything else 1.
"""

from __future__ import annotations

import math
import os
import random
import sys

import torch

sys.path.insert(0, os.path.abspath("latent-attn_amd"))

from latent_attn import LatentAttentionLayer, MLAConfig, build_rope_tables  # noqa: E402
from latent_attn import functional as F  # noqa: E402

DTYPE = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32, "fp8": torch.float8_e4m3fn}
SIZE = {"bf16": 2, "f16": 2, "f32": 4, "fp8": 1}
DC, DN, DR, DV = 512, 128, 64, 128
ROW = DC + DR


def listed():
    return [
        # the smallest call: a short conversation, one token, the reference package's own first benchmark size
        {"name": "fused_f16_512", "kind": "fused", "heads": 128, "dtype": "f16", "seq": 512},
        # several drafted or sampled tokens over one cache, as the reference's batched benchmark has them
        {"name": "batched_f16_16x2048", "kind": "batched", "heads": 128, "dtype": "f16", "batch": 16, "seq": 2048},
        # one user's chat at 8K: the single-sequence configuration of bench.py
        {"name": "decode_bf16_1x8192", "kind": "decode", "heads": 128, "dtype": "bf16", "batch": 1, "seq": 8192},
        # the headline: a full batch at 8K
        {"name": "decode_bf16_32x8192", "kind": "decode", "heads": 128, "dtype": "bf16", "batch": 32, "seq": 8192},
        # few users with very long contexts
        {"name": "decode_bf16_4x131072", "kind": "decode", "heads": 128, "dtype": "bf16", "batch": 4, "seq": 131072},
        # a batch as it comes: 64 sequences of 512 to 32768 positions in one packed cache (the largest)
        {"name": "ragged_bf16_64", "kind": "ragged", "heads": 128, "dtype": "bf16", "batch": 64, "min_len": 512,
         "max_len": 32768, "lens_seed": 0},
        # one of eight GPUs that share the heads, an odd length
        {"name": "decode_bf16_h16_32x4099", "kind": "decode", "heads": 16, "dtype": "bf16", "batch": 32, "seq": 4099},
        # a checking or research program in float32, a length that is no multiple of anything
        {"name": "decode_f32_4x1000", "kind": "decode", "heads": 128, "dtype": "f32", "batch": 4, "seq": 1000},
        # a server's step: every sequence's new token goes into its 8-bit paged cache, then attends
        {"name": "serve_fp8_16", "kind": "serve", "heads": 128, "dtype": "fp8", "batch": 16, "min_len": 300,
         "max_len": 6000, "lens_seed": 1, "block": 64},
        # eight prompts written into the cache
        {"name": "fill_bf16_8x1021", "kind": "fill", "dtype": "bf16", "src": "bf16", "batch": 8, "tokens": 1021,
         "block": 0},
        # the module that a model calls: bench.py --layer's batch
        {"name": "layer_bf16_32x8192", "kind": "layer", "heads": 128, "dtype": "bf16", "batch": 32, "seq": 8192},
        # the un-absorbed path, which programs compare the fused one with
        {"name": "naive_f16_8192", "kind": "naive", "heads": 128, "dtype": "f16", "seq": 8192},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choices(["decode", "ragged", "fused", "batched", "serve", "fill", "layer", "naive"],
                       [6, 2, 2, 2, 2, 2, 1, 1])[0]
    if kind == "decode":
        dtype = rng.choices(["bf16", "f16", "f32", "fp8"], [5, 2, 2, 2])[0]
        total = _log_int(rng, 256, 8192 if dtype == "f32" else 524288)
        batch = _log_int(rng, 1, min(64, total // 64))
        return {"kind": kind, "heads": rng.choice([16, 32, 64, 128, 128]), "dtype": dtype, "batch": batch,
                "seq": max(1, total // batch)}
    if kind == "ragged":
        top = _log_int(rng, 256, 16384)
        return {"kind": kind, "heads": rng.choice([16, 128]), "dtype": rng.choice(["bf16", "f16"]),
                "batch": _log_int(rng, 2, 64), "min_len": rng.randint(1, top // 4), "max_len": top,
                "lens_seed": rng.randrange(1 << 20)}
    if kind == "fused":
        return {"kind": kind, "heads": rng.choice([16, 64, 128]), "dtype": rng.choice(["f16", "f16", "bf16"]),
                "seq": _log_int(rng, 64, 32768)}
    if kind == "batched":
        return {"kind": kind, "heads": rng.choice([16, 64, 128, 128]), "dtype": rng.choice(["f16", "f16", "bf16"]),
                "batch": _log_int(rng, 1, 64), "seq": _log_int(rng, 256, 8192)}
    if kind == "serve":
        top = _log_int(rng, 256, 8192)
        return {"kind": kind, "heads": rng.choice([16, 128, 128]), "dtype": rng.choice(["bf16", "fp8"]),
                "batch": _log_int(rng, 1, 64), "min_len": rng.randint(1, top // 2), "max_len": top,
                "lens_seed": rng.randrange(1 << 20), "block": rng.choice([32, 64, 64, 128])}
    if kind == "fill":
        return {"kind": kind, "dtype": rng.choice(["bf16", "f16", "fp8", "f32"]), "src": rng.choice(["bf16", "f32"]),
                "batch": _log_int(rng, 1, 32), "tokens": _log_int(rng, 16, 2048), "block": rng.choice([0, 0, 64])}
    if kind == "layer":
        return {"kind": kind, "heads": 128, "dtype": rng.choice(["bf16", "f16"]), "batch": _log_int(rng, 1, 32),
                "seq": _log_int(rng, 256, 8192)}
    return {"kind": kind, "heads": rng.choice([16, 128]), "dtype": rng.choice(["f16", "bf16"]),
            "seq": _log_int(rng, 128, 8192)}


def _cfg(case):
    return MLAConfig(5120, DC, DN, DR, case.get("heads", 128), DV)


def _lens(case):
    """The lengths of a ragged batch: the case's own, the same for every seed."""
    r = random.Random(case["lens_seed"])
    return [r.randint(case["min_len"], case["max_len"]) for _ in range(case["batch"])]


def _blocks(case):
    return -(-(case["max_len"] + 1) // case["block"])


def _randn(g, *shape, dtype="f32", scale=1.0):
    """Normal values on the GPU in dtype, made in pieces so that no float32 copy of a large cache is held."""
    if dtype == "f32":
        return torch.randn(*shape, generator=g, device="cuda").mul_(scale)
    out = torch.empty(*shape, dtype=DTYPE[dtype], device="cuda")
    flat = out.view(-1)
    for i in range(0, flat.numel(), 1 << 27):
        n = min(1 << 27, flat.numel() - i)
        flat[i:i + n] = torch.randn(n, generator=g, device="cuda").mul_(scale).to(DTYPE[dtype])
    return out


def _weight(g, case, per_head):
    return _randn(g, case["heads"] * per_head, DC, dtype="bf16" if case["dtype"] == "fp8" else case["dtype"],
                  scale=DC ** -0.5)


def _rope(rows):
    cos, sin = build_rope_tables(rows, DR, device="cuda")
    return cos.contiguous(), sin.contiguous()


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    kind, dtype = case["kind"], case["dtype"]
    s = {"case": case, "cfg": _cfg(case)}
    if kind == "fill":
        b, t, block = case["batch"], case["tokens"], case["block"]
        s["c_t"] = _randn(g, b, t, DC, dtype=case["src"])
        s["k_rope"] = _randn(g, b, t, DR, dtype=case["src"])
        if block:
            per = -(-t // block)
            s["kv"] = torch.zeros(b * per * block, ROW, device="cuda").to(DTYPE[dtype])
            s["table"] = torch.randperm(b * per, generator=g, device="cuda").to(torch.int32).view(b, per)
        else:
            s["kv"] = torch.zeros(b, t, ROW, device="cuda").to(DTYPE[dtype])
        s["lens"] = torch.zeros(b, dtype=torch.int32, device="cuda")
        s["status"] = torch.zeros(1, dtype=torch.int32, device="cuda")
        return s
    heads = case["heads"]
    if kind == "layer":
        with torch.device("cuda"):
            layer = LatentAttentionLayer(s["cfg"], case["seq"])
        s["layer"] = layer.cuda()
        with torch.no_grad():
            for name in ("W_Q_absorbed", "W_Q_rope", "W_UK", "W_UV", "W_O"):
                getattr(layer, name).normal_(0.0, 0.02 / math.sqrt(2.0) if name == "W_O" else 0.02, generator=g)
        s["x"] = _randn(g, case["batch"], s["cfg"].d_model)
        s["kv"] = _randn(g, case["batch"], case["seq"], ROW, dtype=dtype)
        return s
    s["W_UV"] = _weight(g, case, DV)
    if kind in ("fused", "batched"):
        lead = (heads,) if kind == "fused" else (case["batch"], heads)
        s["kv"] = _randn(g, case["seq"], ROW, dtype=dtype)
        s["q_abs"] = _randn(g, *lead, DC, scale=0.5)
        s["q_rope"] = _randn(g, *lead, DR)
        s["cos"], s["sin"] = _rope(case["seq"])
        return s
    s["W_UK"] = _weight(g, case, DN)
    if kind == "naive":
        s["kv"] = _randn(g, case["seq"], ROW, dtype=dtype)
        s["q_nope"], s["q_rope"] = _randn(g, heads, DN), _randn(g, heads, DR)
        s["cos"], s["sin"] = _rope(case["seq"])
        return s
    b = case["batch"]
    s["q_nope"], s["q_rope"] = _randn(g, b, heads, DN), _randn(g, b, heads, DR)
    if kind == "decode":
        s["kv"] = _randn(g, b, case["seq"], ROW, dtype=dtype)
        s["cos"], s["sin"] = _rope(case["seq"])
    elif kind == "ragged":
        lens = _lens(case)
        s["kv"] = _randn(g, sum(lens), ROW, dtype=dtype)
        s["offsets"] = torch.tensor([sum(lens[:i]) for i in range(b + 1)], dtype=torch.int32, device="cuda")
        s["cos"], s["sin"] = _rope(max(lens))
    else:  # serve
        per = _blocks(case)
        s["kv"] = _randn(g, b * per * case["block"], ROW, dtype=dtype)
        s["table"] = torch.randperm(b * per, generator=g, device="cuda").to(torch.int32).view(b, per)
        s["lens"] = torch.tensor(_lens(case), dtype=torch.int32, device="cuda")
        s["c_t"], s["k_rope"] = _randn(g, b, 1, DC, dtype="bf16"), _randn(g, b, 1, DR, dtype="bf16")
        s["cos"], s["sin"] = _rope(case["max_len"] + 1)
    return s


def run(s):
    case, cfg = s["case"], s["cfg"]
    kind = case["kind"]
    if kind == "fused":
        return F.fused_mla(s["kv"], s["q_abs"], s["q_rope"], s["W_UV"], s["cos"], s["sin"], cfg)
    if kind == "batched":
        return F.batched_fused_mla(s["kv"], s["q_abs"], s["q_rope"], s["W_UV"], s["cos"], s["sin"], cfg)
    if kind == "decode":
        return F.mla_decode(s["kv"], s["q_nope"], s["q_rope"], s["W_UK"], s["W_UV"], s["cos"], s["sin"], cfg)
    if kind == "ragged":
        return F.mla_decode(s["kv"], s["q_nope"], s["q_rope"], s["W_UK"], s["W_UV"], s["cos"], s["sin"], cfg,
                            seq_offsets=s["offsets"])
    if kind == "layer":
        return s["layer"].forward_batch(s["x"], s["kv"])
    if kind == "naive":
        return F.naive_mla(s["kv"], s["W_UK"], s["W_UV"], s["q_nope"], s["q_rope"], s["cos"], s["sin"], cfg)
    if kind == "fill":
        s["lens"].zero_()  # new sequences in these places
        if case["block"]:
            F.append_kv(s["kv"], s["lens"], s["c_t"], s["k_rope"], cfg, status=s["status"], block_table=s["table"],
                        block_size=case["block"])
        else:
            F.append_kv(s["kv"], s["lens"], s["c_t"], s["k_rope"], cfg, status=s["status"])
        return {"kv": _bytes(s["kv"]), "lens": s["lens"], "status": s["status"]}
    # serve: the step's lengths and its query, which the append advances and rotates in place
    lens, q_rope = s["lens"].clone(), s["q_rope"].clone()
    F.append_kv(s["kv"], lens, s["c_t"], s["k_rope"], cfg, q_rope=q_rope, rope_cos=s["cos"], rope_sin=s["sin"],
                block_table=s["table"], block_size=case["block"])
    out = F.mla_decode(s["kv"], s["q_nope"], q_rope, s["W_UK"], s["W_UV"], s["cos"], s["sin"], cfg, seq_lens=lens,
                       block_table=s["table"], block_size=case["block"])
    return {"out": out, "q_rope": q_rope, "lens": lens, "kv": _bytes(s["kv"])}


def _bytes(kv):
    """A cache as whole numbers, so that it is compared bit by bit."""
    return kv.view({1: torch.uint8, 2: torch.int16, 4: torch.int32}[kv.element_size()])


def work(case):
    kind, size = case["kind"], SIZE[case["dtype"]]
    if kind == "fill":
        rows = case["batch"] * case["tokens"]
        return {"bytes": rows * ROW * (size + SIZE[case["src"]]), "flops": 0}
    heads = case["heads"]
    wsize = 4 if case["dtype"] == "f32" else 2
    if kind in ("ragged", "serve"):
        lens = [n + (kind == "serve") for n in _lens(case)]
    else:
        lens = [case["seq"]] * (1 if kind in ("fused", "batched", "naive") else case["batch"])
    tokens = case["batch"] if kind == "batched" else len(lens)
    rows, longest = sum(lens), max(lens)
    cache = rows * ROW * size
    tables = longest * DR * 4
    out = tokens * heads * DV * 4
    w = heads * 128 * DC
    shared = case["batch"] if kind == "batched" else 1
    attend = 2 * heads * (ROW + DC) * rows * shared
    project = 2 * w * tokens  # the query absorbed, or the output projected
    if kind in ("fused", "batched"):
        return {"bytes": cache + tables + out + w * wsize + tokens * heads * ROW * 4, "flops": attend + project}
    if kind == "naive":
        return {"bytes": cache + tables + out + 2 * w * wsize + tokens * heads * (DN + DR) * 4,
                "flops": 4 * w * rows + 2 * heads * (DN + DR + DV) * rows}
    if kind == "layer":
        d = 5120
        weights = (heads * DC + heads * DR + heads * DV) * d + w  # query, rope and output projections; W_UV
        return {"bytes": cache + tables + 4 * weights + 2 * tokens * d * 4,
                "flops": attend + project + 2 * tokens * d * heads * (DC + DR + DV)}
    new = 2 * tokens * ROW * size + tokens * heads * DR * 4 if kind == "serve" else 0
    return {"bytes": cache + tables + out + 2 * w * wsize + tokens * heads * (DN + DR) * 4 + new,
            "flops": attend + 2 * project}


def tolerance(case):
    """About four times the error against exact() that each type shows."""
    if case["kind"] == "fill":
        return "exact"  # copies and conversions that round to nearest
    if case["kind"] == "naive":
        return {"rel": 6e-6}  # float32 sums of exact 16-bit values
    if case["kind"] == "layer":
        return {"rel": {"bf16": 1.3e-2, "f16": 2e-3}[case["dtype"]]}
    return {"rel": {"bf16": 9e-3, "fp8": 9e-3, "f16": 1.5e-3, "f32": 3e-6}[case["dtype"]]}


def _attend(kv, q_abs, q_rope, cos, sin, w_uv):
    """kv (S, 576), q_abs (H, 512), q_rope (H, 64), w_uv (H, 128, 512) -> (H, 128), all in 64 bits."""
    c, k = kv[:, :DC], kv[:, DC:]
    co, si = cos[:kv.size(0)].double(), sin[:kv.size(0)].double()
    a, b = k[:, :DR // 2], k[:, DR // 2:]
    k = torch.cat([a * co - b * si, a * si + b * co], 1)
    p = torch.softmax((q_abs @ c.T + q_rope @ k.T) / math.sqrt(DN + DR), 1)
    return ((p @ c)[:, None, :] * w_uv).sum(2)


def exact(case, seed):
    kind = case["kind"]
    if kind == "fill":
        return None
    s = prepare(case, seed)
    heads = case["heads"]
    if kind == "layer":
        layer = s["layer"]
        x = s["x"].double()
        q_abs = (x @ layer.W_Q_absorbed.detach().double().T).view(-1, heads, DC)
        q_rope = (x @ layer.W_Q_rope.detach().double().T).view(-1, heads, DR)
        w_uv = layer.W_UV.detach().half().double().view(heads, DV, DC)  # the module's attention takes it in fp16
        o = torch.stack([_attend(s["kv"][i].double(), q_abs[i], q_rope[i], layer.rope_cos, layer.rope_sin, w_uv)
                         for i in range(case["batch"])])
        return o.flatten(1) @ layer.W_O.detach().double().T
    w_uv = s["W_UV"].double().view(heads, DV, DC)
    cos, sin = s["cos"], s["sin"]
    q_rope = s["q_rope"].double()
    if kind == "fused":
        return _attend(s["kv"].double(), s["q_abs"].double(), q_rope, cos, sin, w_uv)
    if kind == "batched":
        kv = s["kv"].double()
        return torch.stack([_attend(kv, s["q_abs"][i].double(), q_rope[i], cos, sin, w_uv)
                            for i in range(case["batch"])])
    w_uk = s["W_UK"].double().view(heads, DN, DC)
    q_abs = (s["q_nope"].double()[..., None] * w_uk).sum(-2) if kind == "naive" else torch.stack(
        [(q.double()[..., None] * w_uk).sum(-2) for q in s["q_nope"]])
    if kind == "naive":
        return _attend(s["kv"].double(), q_abs, q_rope, cos, sin, w_uv)
    if kind == "decode":
        caches = list(s["kv"])
    elif kind == "ragged":
        caches = list(torch.split(s["kv"], _lens(case)))
    else:
        lens, block = _lens(case), case["block"]
        pool = s["kv"].view(-1, block, ROW)
        new = torch.cat([s["c_t"][:, 0], s["k_rope"][:, 0]], 1).float().clamp(-448, 448).to(DTYPE[case["dtype"]])
        caches = [torch.cat([pool[s["table"][i].long()].flatten(0, 1)[:n].double(), new[i:i + 1].double()])
                  for i, n in enumerate(lens)]
        at = torch.tensor(lens, device="cuda")
        co, si = cos[at].double()[:, None], sin[at].double()[:, None]
        a, b = q_rope[..., :DR // 2], q_rope[..., DR // 2:]
        q_rope = torch.cat([a * co - b * si, a * si + b * co], -1)
    out = torch.stack([_attend(kv.double(), q_abs[i], q_rope[i], cos, sin, w_uv) for i, kv in enumerate(caches)])
    return {"out": out, "q_rope": q_rope, "lens": None, "kv": None} if kind == "serve" else out
