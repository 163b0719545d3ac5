"""The auto schedule's lines (DecodeAttention.schedule) on a device of 256 compute units: host arithmetic, no GPU."""
from __future__ import annotations

import pytest


@pytest.mark.parametrize("b,S,fused,want", [
    (80, 4096, True, "stream"),    # a fused call has its row's length before the first tiles: from 5/8 of the CUs
    (79, 4096, True, "split"),
    (80, 4096, False, "split"),    # an unfused call requests its first tiles over the whole row: from 3/4
    (95, 2112, False, "split"),
    (96, 4096, False, "stream"),
    (64, 2048, False, "stream"),   # up to 2048 positions, from half of them either way
    (64, 2048, True, "stream"),
    (63, 2048, False, "split"),
])
def test_long_rows(a8, b, S, fused, want):
    att = a8.DecodeAttention(16 * b, 14, 2, 64, 16, "cpu")
    att.n_cu = 256
    assert att.schedule(b, S, a8.ref_nsplit(b, 2), fused=fused)[0] == want
