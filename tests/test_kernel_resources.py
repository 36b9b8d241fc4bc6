"""CPU check of the compiled hot kernels' registers: none spills to scratch (hipcc, gfx950 assembly;
the 128-head attention kernel is checked in tests/test_lds_waits.py)."""

from __future__ import annotations

import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.parametrize("source,least", [("la_append", 5), ("la_f32", 5), ("la_mfma16", 18), ("la_naive", 8), ("la_proj", 20)])
def test_no_scratch(source, least, tmp_path):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    src = os.path.join(ROOT, "latent-attn_amd", "csrc")
    out = tmp_path / "kernels.s"
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", "-I", os.path.join(ROOT, "include"), "-I", src, "--cuda-device-only", "-S",
                    os.path.join(src, source + ".hip"), "-o", str(out)], check=True, capture_output=True, timeout=600)
    sizes = {}
    for line in out.read_text().splitlines():
        if m := re.match(r"\s*\.amdhsa_kernel (\S+)", line):
            name = m.group(1)
        elif m := re.match(r"\s*\.amdhsa_private_segment_fixed_size (\d+)", line):
            sizes[name] = int(m.group(1))
    assert len(sizes) >= least
    assert {n: b for n, b in sizes.items() if b} == {}
