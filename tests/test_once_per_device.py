"""csrc/la_once.hpp on the host: a kernel's set-up step runs for every device of a process, again
after a failure, and from any thread."""

from __future__ import annotations

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include "la_once.hpp"
#include <thread>
#include <vector>
int main() {
  la::OncePerDevice once;
  int calls = 0;
  auto ok = [&] { ++calls; return 0; };
  if (once.run(0, ok) != 0 || once.run(0, ok) != 0 || calls != 1) return 1;
  if (once.run(1, ok) != 0 || calls != 2) return 2;       // a second device needs its own
  if (once.run(3, [] { return 7; }) != 7) return 3;       // a failure is reported and not kept
  if (once.run(3, ok) != 0 || calls != 3) return 4;
  if (once.run(64, ok) != 0 || once.run(64, ok) != 0 || calls != 5) return 5;  // past the bits: every time
  la::OncePerDevice shared;
  std::atomic<int> n{0};
  std::vector<std::thread> t;
  for (int i = 0; i < 8; ++i)
    t.emplace_back([&] { for (int d = 0; d < 63; ++d) shared.run(d, [&] { ++n; return 0; }); });
  for (auto& x : t) x.join();
  const int after = n;
  for (int d = 0; d < 63; ++d) shared.run(d, [&] { ++n; return 0; });
  return after >= 63 && n == after ? 0 : 6;
}
"""


def test_once_per_device(tmp_path):
    gxx = shutil.which("g++")
    if not gxx:
        pytest.skip("g++ not available")
    src, exe = tmp_path / "once.cpp", tmp_path / "once"
    src.write_text(PROGRAM)
    subprocess.run([gxx, "-std=c++17", "-O2", "-pthread", "-I", os.path.join(ROOT, "latent-attn_amd", "csrc"), str(src),
                    "-o", str(exe)], check=True)
    assert subprocess.run([str(exe)], timeout=60).returncode == 0
