"""Whole-row decode at ragged lengths (k_decode_rows with the second unit chosen by length, k_decode_unit with the
row's own step count): every row served once whatever the lengths and ties, at the edges of the halves (one row,
odd counts, more than 64 and more than 128 rows a wave ranks), of the step counts (empty rows, one key, tile and
step edges, the whole cache) and of the step instances (2 to 16 steps)."""
from __future__ import annotations

import pytest
import torch

from conftest import randn_bf16

pytestmark = pytest.mark.gpu

NQ, NKV, HD = 14, 2, 64
W = (NQ + 2 * NKV) * HD
BF = torch.bfloat16


def _lens(kind, b, S, g):
    if kind == "equal":
        return torch.full((b,), S, dtype=torch.int32)
    edges = torch.tensor([0, 1, 63, 64, 65, 255, 256, 257, S - 1, S, S + 5, S // 2, S // 2], dtype=torch.int32)
    if kind == "ties":
        return edges[torch.randint(0, len(edges), (b,), generator=g)]
    return torch.randint(1, S + 1, (b,), generator=g, dtype=torch.int32)


@pytest.mark.parametrize("b,S,per", [(1, 300, 2), (2, 512, 2), (5, 1100, 2), (67, 320, 2), (131, 2048, 2),
                                     (256, 600, 2), (3, 4096, 2), (33, 700, 1), (9, 4096, 1), (1, 512, 1)])
@pytest.mark.parametrize("kind", ["random", "ties", "equal"])
def test_ragged_rows(a8, ref, dev, b, S, per, kind):
    print(f"case: {b} rows x {S}, {per} unit(s) per workgroup, {kind} lengths", flush=True)
    g = torch.Generator().manual_seed(b * 7 + S)
    lens = _lens(kind, b, S, g)
    pos = (lens - 1).clamp(0, S - 1)
    qkv, bias = randn_bf16(g, b, W), (torch.randn(W, generator=g) * 0.02).to(BF)
    kc, vc = randn_bf16(g, b, NKV, S, HD), randn_bf16(g, b, NKV, S, HD)
    slot = torch.randperm(b, generator=g).int()
    cos, sin = a8.rope_tables(10000.0, HD, S, dev)
    att = a8.DecodeAttention(max(16 * b, 64), NQ, NKV, HD, 16, dev)
    att.force_stream = (4, -(-S // 256), b if per == 2 else 2 * b)
    # the oracle: store, then attend cache row slot[r]
    cr, sr = ref.rope_tables(10000.0, HD, S)
    q_ref, kr, vr = torch.zeros(b, NQ, HD, dtype=BF), kc.clone(), vc.clone()
    ref.bias_rope_store(qkv, bias, cr, sr, pos, slot, q_ref, kr, vr, NQ, NKV, HD)
    want = ref.decode_attention(q_ref, kr, vr, lens.clamp(max=S), nsplit=1, rowmap=slot).float()
    d = [t.to(dev) for t in (qkv, bias, pos, slot, lens)]
    outs = []
    for fused in (True, False):
        k, v = kc.to(dev), vc.to(dev)
        q = torch.zeros(b, NQ, HD, dtype=BF, device=dev)
        out = torch.zeros(b, NQ, HD, dtype=BF, device=dev)
        if fused:
            att.store_and_attend(d[0], d[1], cos, sin, d[2], d[3], q, k, v, d[4], out, rowmap=d[3])
        else:
            a8.bias_rope_store(d[0], d[1], cos, sin, d[2], d[3], q, k, v, NQ, NKV, HD)
            att(q, k, v, d[4], out, rowmap=d[3])
        torch.cuda.synchronize()
        got = out.cpu().float()
        assert torch.equal(k.cpu(), kr) and torch.equal(v.cpu(), vr)
        assert torch.equal(got.isnan(), want.isnan())
        # bf16 weights and outputs, as the other decode tests' bar
        assert (got - want).nan_to_num().abs().max().item() <= 2e-2
        outs.append(out.cpu().view(torch.int16))
    assert torch.equal(outs[0], outs[1])


@pytest.mark.parametrize("b,S,want", [(1, 1024, "unit"), (48, 1024, "unit"), (80, 4096, "unit"), (64, 4096, "split"),
                                      (140, 4096, "pair"), (16, 2048, "split")])
def test_fused_schedule(a8, dev, b, S, want):
    """The auto schedule's lines for a fused call: one workgroup per unit up to 1024 positions and, up to 4096, from
    5/8 of the compute units; two units a workgroup above one per compute unit."""
    att = a8.DecodeAttention(16 * b, NQ, NKV, HD, 16, dev)
    if att.n_cu != 256:
        pytest.skip(f"the lines are stated for 256 compute units, this device has {att.n_cu}")
    kind, shape = att.schedule(b, S, a8.ref_nsplit(b, NKV), fused=True)
    assert (kind, shape[2] if kind == "stream" else 0) == {"unit": ("stream", 2 * b), "pair": ("stream", b),
                                                           "split": ("split", 0)}[want]


@pytest.mark.parametrize("b,S", [(12, 512), (67, 1500), (192, 2048), (33, 4096)])
@pytest.mark.parametrize("fused", [True, False])
def test_a_rows_bits_are_its_own(a8, dev, b, S, fused):
    """A row's output depends on its own length alone: the same bits when every other row's length changes (and with
    it the pairing by length), and the same bits with one unit a workgroup as with two."""
    print(f"case: {b} rows x {S}, fused={fused}, kept rows among changed ones", flush=True)
    g = torch.Generator().manual_seed(b + S)
    kept = torch.arange(0, b, 3)
    first = torch.randint(1, S + 1, (b,), generator=g, dtype=torch.int32)
    qkv, bias = randn_bf16(g, b, W).to(dev), (torch.randn(W, generator=g) * 0.02).to(BF).to(dev)
    kc, vc = randn_bf16(g, b, NKV, S, HD), randn_bf16(g, b, NKV, S, HD)
    q0 = randn_bf16(g, b, NQ, HD).to(dev)
    slot = torch.arange(b, dtype=torch.int32, device=dev)
    cos, sin = a8.rope_tables(10000.0, HD, S, dev)
    att = a8.DecodeAttention(max(16 * b, 64), NQ, NKV, HD, 16, dev)

    def run(lens, per):
        att.force_stream = (4, -(-S // 256), b if per == 2 else 2 * b)
        k, v, out = kc.to(dev), vc.to(dev), torch.zeros(b, NQ, HD, dtype=BF, device=dev)
        n = lens.to(dev)
        if fused:
            att.store_and_attend(qkv, bias, cos, sin, (n - 1), slot, torch.empty_like(q0), k, v, n, out)
        else:
            att(q0, k, v, n, out)
        torch.cuda.synchronize()
        return out.cpu().view(torch.int16)

    want = run(first, 2)
    assert torch.equal(run(first, 1), want)
    for kind in range(3):
        lens = torch.randint(1, S + 1, (b,), generator=g, dtype=torch.int32) if kind else torch.full_like(first, S)
        lens[kept] = first[kept]
        assert torch.equal(run(lens, 2)[kept], want[kept])
