"""latent-attn_amd/phase_profile.py on the host: a workload whose attention kernel leaves no stamps
(decode_mfma16_kernel) has no phase table, and the launch is counted for the kernel that runs."""

from __future__ import annotations

import ctypes
import types

import numpy as np
import pytest

import phase_profile as pp


class StampLib:
    """la_phase_attn_stamps over given stamps (blocks, 4 waves, SLOTS)."""

    def __init__(self, stamps):
        self.stamps = np.ascontiguousarray(stamps, dtype=np.uint64)

    def la_phase_attn_stamps(self, buf, blocks, clear):
        ctypes.memmove(buf, self.stamps.ctypes.data, self.stamps[:blocks].nbytes)
        return 0


def test_no_stamps_no_table():
    assert pp.attn_table(StampLib(np.zeros((8, 4, pp.SLOTS))), 8) is None


def test_stamped_workgroups_are_kept(capsys):
    st = np.zeros((8, 4, pp.SLOTS))
    st[:3, :, :11] = 100 + 10 * np.arange(11)
    st[:3, :, 11:15], st[:3, :, 15] = 40, 4
    n, total, d, per_tile = pp.attn_table(StampLib(st), 8)
    assert n == 3 and (total == 100).all() and (d == 10).all() and (per_tile == 10).all()
    row = (n, total, d, per_tile)
    pp.print_attention({"back to back": row, "in a step": row})
    assert "| total | 100 | 100 | 100 | 100 |" in capsys.readouterr().out


@pytest.mark.parametrize("chunks,heads,per_wg,want", [(64, 128, 16, 512), (256, 128, 128, 256), (4, 128, 16, 32),
                                                      (171, 48, 128, 176), (3, 144, 128, 8)])
def test_workgroups_of_the_launch(chunks, heads, per_wg, want):
    info = types.SimpleNamespace(num_chunks=chunks, heads_per_workgroup=per_wg)
    assert pp.attention_workgroups(info, heads) == want
