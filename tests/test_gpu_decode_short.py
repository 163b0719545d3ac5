"""The fused store + decode over a cache of at most 32 positions (csrc/decode_short.h; the fast AR's passes) against the
two calls it replaces, bit for bit, at and around its limit: caches of 1 .. 33 positions (33 takes the streaming
kernel), lengths of 0, 1 and past the cache, the new key at the end, inside and past the attended keys, ring wrap,
positions outside the tables, slots outside the cache, with and without a row map, a bias and a stored q."""
from __future__ import annotations

import pytest
import torch

from test_gpu_fused import HD, NKV, NQ, _bits_equal, _inputs, _run_both

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S", [1, 2, 10, 15, 16, 17, 31, 32, 33])
@pytest.mark.parametrize("use_rowmap", [True, False])
def test_short_cache_equals_store_then_attend(a8, dev, S, use_rowmap):
    print(f"case: short fused decode S={S} rowmap={use_rowmap}", flush=True)
    g = torch.Generator().manual_seed(S)
    b, ring = 37, max(1, S - 1)
    lens = [int(v) for v in torch.randint(0, S + 3, (b,), generator=g)]
    lens[:4] = [0, 1, S, S + 5]
    pos = [max(0, min(L, S) - 1) for L in lens]
    pos[5:9] = [0, S - 1, 3 * S + 1, ring]                   # inside, at the end, wrapped
    slot = torch.randperm(b + 2, generator=g)[:b].tolist() if use_rowmap else list(range(b))
    slot[10] = b + 40                                        # outside the cache
    for bias, write_q in ((True, True), (False, False)):
        x = _inputs(S, b, b + 2, S, lens, pos, slot, bias=bias, max_pos=4 * S + 8)
        (o0, q0, k0, v0), (o1, q1, k1, v1) = _run_both(a8, dev, x, (1, 1, 2 * b), ring=ring, write_q=write_q,
                                                       use_rowmap=use_rowmap)
        assert _bits_equal(q0, q1) if write_q else not q1.any()
        assert _bits_equal(k0, k1) and _bits_equal(v0, v1)
        live = [i for i in range(b) if not (use_rowmap and i == 10) and lens[i] > 0]
        assert _bits_equal(o0[live], o1[live])
        dead = [i for i in range(b) if i not in live]
        assert torch.isnan(o0[dead].float()).all() and torch.isnan(o1[dead].float()).all()


def test_short_cache_position_outside_the_tables(a8, dev):
    """A row at a position with no table row stores nothing and attends with q = 0: the mean of its values."""
    S, b = 10, 3
    x = _inputs(7, b, b, S, [10, 10, 4], [9, 500, 3], [0, 1, 2], max_pos=16)
    _, (o1, _, k1, v1) = _run_both(a8, dev, x, (1, 1, 2 * b), use_rowmap=False)
    assert _bits_equal(k1[1], x["kc"][1]) and _bits_equal(v1[1], x["vc"][1])
    mean = x["vc"][1].float().mean(1).repeat_interleave(NQ // NKV, 0)
    assert o1.shape == (b, NQ, HD) and (o1[1].float() - mean).abs().max().item() <= 2e-2
