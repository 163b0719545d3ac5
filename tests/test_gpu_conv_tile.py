"""The tile convolution (csrc/conv_tile.hip) behind conv_cl and ru_cl, where its tiles end: row counts one under, at
and over its 128 / 256 rows (64-row waves) and ragged ends of its 192 / 384 (96-row waves), batch rows that divide a
tile, do not, or are longer; one to eight taps and the widest dilations its LDS slices hold (and one past them, which
takes the other kernel); an odd and an even number of 96-channel column groups over one or several phases; K split or
not; inputs with more rows than the call needs. test_conv_tile_edges: against the oracle (fp32 sums), to one fp16 ulp
(sums in another order) or 1e-3 of the scale where a sum cancels; test_conv_tile_instances: against float64, to the
rounding of the result and a bound on the fp32 sums."""
from __future__ import annotations

import pytest
import torch

from test_schedule import conv_tile

pytestmark = pytest.mark.gpu
F16 = torch.float16


def _close(got, want):
    g, w = got.cpu().float(), want.float()
    ulp = (w.abs() * 2 ** -10).clamp(min=2 ** -24)
    return bool((((g - w).abs() <= ulp * 1.01) | ((g - w).abs() <= 1e-3 * w.abs().max().item())).all())


@pytest.mark.parametrize("B,T,extra,Cin,Cout,taps,dil,ph,res,split", [
    (1, 127, 0, 192, 192, 7, 1, 1, False, True),       # one row under a tile, two column halves
    (1, 129, 0, 192, 192, 7, 9, 1, True, True),        # one over, the widest dilation
    (3, 64, 0, 192, 192, 7, 1, 1, True, False),        # few rows and no workspace: the general kernel
    (3, 64, 0, 192, 192, 7, 1, 1, True, True),         # batch rows dividing a tile
    (7, 50, 0, 192, 384, 7, 3, 1, True, True),         # not dividing it
    (5, 70, 3, 192, 192, 7, 3, 1, False, True),        # input rows left over after the last tap's reach
    (37, 4, 0, 512, 192, 7, 1, 1, False, True),        # four-row batch rows: 320-row slices
    (12, 32, 0, 192, 192, 7, 9, 1, False, True),       # 344-row slices
    (12, 32, 0, 192, 192, 8, 9, 1, False, True),       # 381-row slices: past the tile kernel's LDS
    (3, 257, 0, 192, 96, 7, 1, 1, True, True),         # one column group: the 256-row tile
    (2, 385, 0, 224, 96, 7, 5, 1, False, True),        #   and 7 channel slices, ragged, at its widest dilation
    (2, 385, 0, 224, 96, 7, 9, 1, False, True),        #   364-row slices: past the LDS of the narrow tile
    (1, 33, 0, 576, 96, 2, 1, 8, False, True),         # phases in pairs over one column group each
    (2, 65, 0, 416, 192, 3, 2, 3, True, True),         # six column groups over three phases, 13 channel slices
    (1, 5, 0, 1152, 96, 1, 1, 3, True, True),          # one tap, an odd number of column groups, one short tile
    (130, 128, 0, 96, 192, 1, 1, 1, True, False),      # one tap, many tiles (three channel slices)
    (43, 384, 0, 32, 96, 2, 1, 2, False, False),       # one channel slice, two taps
])
def test_conv_tile_edges(a8, dev, B, T, extra, Cin, Cout, taps, dil, ph, res, split):
    from oracle import conv_ref as cref
    print(f"case: conv_cl tile B={B} T={T}+{extra} {Cin}->{Cout} taps={taps} dil={dil} ph={ph} res={res} split={split}",
          flush=True)
    g = torch.Generator().manual_seed(B + T + Cin + Cout + taps)
    Tin = T + (taps - 1) * dil + extra
    x = torch.randn(B, Tin, Cin, generator=g).to(F16)
    w = (torch.randn(ph, taps, Cin, Cout, generator=g) / (taps * Cin) ** 0.5).to(F16)
    bv = torch.randn(Cout, generator=g).to(F16)
    rv = torch.randn(B, T * ph, Cout, generator=g).to(F16) if res else None
    want = cref.conv_cl(x, w, bv, T, taps, dil, ph, Cout, res=rv)
    nws = a8.conv_cl_ws_bytes(B, T, Cin, Cout, taps, ph)
    ws = torch.empty(nws, dtype=torch.uint8, device=dev) if split and nws > 0 else None
    # rows around the output stay as they are
    buf = torch.full((B, T * ph + 2, Cout), 7.0, dtype=F16, device=dev)
    a8.conv_cl(x.to(dev), w.to(dev), bv.to(dev), T, taps, dil, ph, buf[:, 1:T * ph + 1],
               res=rv.to(dev) if res else None, ws=ws)
    torch.cuda.synchronize()
    got = buf.cpu()
    assert _close(got[:, 1:T * ph + 1], want)
    assert (got[:, 0] == 7.0).all() and (got[:, T * ph + 1] == 7.0).all()


@pytest.mark.parametrize("shares", [0, 1, 2, 3, 4.5, 6])
def test_conv_tile_workspace_sizes(a8, dev, shares):
    """K shares as the workspace holds them, down to none (the general kernel then): nothing is written past it."""
    from oracle import conv_ref as cref
    M, Cin, Cout, taps = 250, 384, 384, 7
    nws = int(shares * 4 * M * Cout)
    print(f"case: conv_cl {M} rows, a workspace of {shares} shares", flush=True)
    g = torch.Generator().manual_seed(77)
    x = torch.randn(1, M + 6, Cin, generator=g).to(F16)
    w = (torch.randn(1, taps, Cin, Cout, generator=g) / (taps * Cin) ** 0.5).to(F16)
    bv = torch.randn(Cout, generator=g).to(F16)
    want = cref.conv_cl(x, w, bv, M, taps, 1, 1, Cout)
    ws = torch.full((nws + 4096,), 0x5a, dtype=torch.uint8, device=dev)
    y = torch.empty(1, M, Cout, dtype=F16, device=dev)
    a8.conv_cl(x.to(dev), w.to(dev), bv.to(dev), M, taps, 1, 1, y, ws=ws[:nws] if nws else None)
    torch.cuda.synchronize()
    assert _close(y, want)
    assert (ws[nws:] == 0x5a).all()


def _exact(x, w, b, T, taps, dil, ph, res):
    x, w = x.double(), w.double()
    out = torch.empty(x.shape[0], T * ph, w.shape[3], dtype=torch.float64)
    for p in range(ph):
        out[:, p::ph] = sum(x[:, j * dil:j * dil + T] @ w[p, j] for j in range(taps))
    return out + b.double() + res.double()


@pytest.mark.parametrize("B,T,Cin,Cout,taps,dil,ph,want", [
    (1, 2100, 64, 384, 2, 1, 8, (3, 16, 1)),        # 192-row tiles, one pass
    (21, 100, 64, 384, 7, 8, 8, (3, 22, 1)),        #   over batch rows of 100
    (1, 2710, 512, 768, 7, 1, 1, (3, 16, 4)),       #   K split
    (27, 100, 512, 768, 7, 8, 1, (3, 22, 4)),
    (2, 35001, 32, 96, 3, 9, 1, (3, 28, 1)),        # 384-row tiles, one pass
    (1, 7260, 512, 288, 7, 1, 1, (3, 28, 4)),       #   K split, three column groups
    (130, 128, 96, 192, 1, 1, 1, (2, 12, 1)),       # 128- and 256-row tiles in one pass
    (81, 515, 64, 96, 7, 5, 1, (2, 20, 1)),
])
def test_conv_tile_instances(a8, dev, B, T, Cin, Cout, taps, dil, ph, want):
    """Every instance of the tile kernel, on row counts that its tiles do not divide (want: row groups a wave, KiB of an
    input slice, K shares)."""
    print(f"case: conv_cl tile {want} B={B} T={T} {Cin}->{Cout} taps={taps} dil={dil} ph={ph}", flush=True)
    Tin = T + (taps - 1) * dil
    nws = a8.conv_cl_ws_bytes(B, T, Cin, Cout, taps, ph)
    assert conv_tile(a8, B, Tin, T, Cin, Cout, taps, dil, ph, ws=nws) == want
    g = torch.Generator().manual_seed(B + T + Cin + Cout)
    x = torch.randn(B, Tin, Cin, generator=g).to(F16)
    w = (torch.randn(ph, taps, Cin, Cout, generator=g) / (taps * Cin) ** 0.5).to(F16)
    bv = torch.randn(Cout, generator=g).to(F16)
    rv = torch.randn(B, T * ph, Cout, generator=g).to(F16)
    ws = torch.empty(nws, dtype=torch.uint8, device=dev) if nws > 0 else None
    buf = torch.full((B, T * ph + 2, Cout), 7.0, dtype=F16, device=dev)
    a8.conv_cl(x.to(dev), w.to(dev), bv.to(dev), T, taps, dil, ph, buf[:, 1:T * ph + 1], res=rv.to(dev), ws=ws)
    torch.cuda.synchronize()
    got = buf.cpu()
    assert (got[:, 0] == 7.0).all() and (got[:, T * ph + 1] == 7.0).all()
    exact = _exact(x, w, bv, T, taps, dil, ph, rv)
    # a sum of Cin taps / 16 MFMAs, the shares, the bias and the residual: each step rounds (or cuts) a partial sum,
    # taken as at most twice the largest result, by 2^-23 of it; the 16 products of an MFMA likewise among themselves
    steps = taps * Cin / 16 + 16 + want[2] + 2
    sums = steps * 2 ** -23 * 2 * exact.abs().max().item()
    err = (got[:, 1:T * ph + 1].double() - exact).abs()
    assert (err <= (exact.abs() + sums) * 2 ** -11 + 2 ** -25 + sums).all(), err.max().item()


@pytest.mark.parametrize("B,T,C,dil,want", [
    (161, 128, 192, 9, (2, 12)), (162, 127, 192, 1, (2, 12)),  # 128-row tiles, whole and ragged batch rows
    (65, 511, 192, 1, (3, 16)), (66, 500, 192, 3, (3, 16)),    # 192-row tiles, ragged
    (41, 1000, 96, 3, (2, 20)), (81, 515, 96, 5, (2, 20)),     # 256-row tiles
    (65, 1009, 96, 3, (3, 28)),                                # 384-row tiles
    (81, 515, 96, 9, (0, 0)),                                  # past the narrow tile's LDS: the general kernel
])
def test_ru_tile_edges(a8, dev, B, T, C, dil, want):
    """The residual unit on every instance of the tile kernel that takes one (want: row groups a wave, KiB of an input
    slice): full and ragged tiles, both widths."""
    from oracle import conv_ref as cref
    print(f"case: ru_cl tile B={B} T={T} C={C} dil={dil}", flush=True)
    g = torch.Generator().manual_seed(B * 7 + C + dil)
    taps, ctx = 7, 6 * dil
    assert conv_tile(a8, B, ctx + T, T, C, C, taps, dil, 1, ru=1)[:2] == want
    x = torch.randn(B, T, C, generator=g).half()
    st = torch.randn(B, ctx, C, generator=g).half()
    a1, a2 = torch.rand(C, generator=g) + 0.5, torch.rand(C, generator=g) + 0.5
    ib1, ib2 = 1.0 / (a1 + 1e-9), 1.0 / (a2 + 1e-9)
    w1 = (torch.randn(taps, C, C, generator=g) / (taps * C) ** 0.5).half()
    w2 = (torch.randn(C, C, generator=g) / C ** 0.5).half()
    b1, b2 = (0.1 * torch.randn(C, generator=g)).half(), (0.1 * torch.randn(C, generator=g)).half()
    want = cref.ru_fused(x, st, a1, ib1, w1, b1, a2, ib2, w2, b2, taps, dil)
    xd = x.to(dev)
    xin = torch.empty(B, ctx + T, C, dtype=F16, device=dev)
    a8.snake_cat(xd, st.to(dev), a1.to(dev), ib1.to(dev), xin)
    out = torch.full((B, T, C), 9.0, dtype=F16, device=dev)
    a8.ru_cl(xin, w1.to(dev), b1.to(dev), a2.to(dev), ib2.to(dev), w2.to(dev), b2.to(dev), xd, out, T, taps, dil)
    torch.cuda.synchronize()
    assert _close(out, want)


@pytest.mark.parametrize("B,T,Cin,Cout,cw,taps,split", [
    (130, 128, 96, 192, 192, 1, False), # the tile kernel
    (3, 64, 192, 192, 192, 7, True),    #   K split: in the finish
    (3, 64, 192, 192, 192, 7, False),   # k_conv_cl: four channels a store
    (3, 40, 64, 96, 96, 3, False),
    (3, 40, 64, 30, 32, 3, False),      #   element by element
    (4, 8, 512, 30, 32, 7, True),       #   K split
])
def test_out_snake_equals_a_snake_pass(a8, dev, B, T, Cin, Cout, cw, taps, split):
    """conv_cl with out_snake against conv_cl then the snake over its fp16 outputs (snake_cat without a context; per
    channel, so Cout is padded to whole 16-byte chunks there): the same bits."""
    print(f"case: out_snake B={B} T={T} {Cin}->{Cout} taps={taps} split={split}", flush=True)
    g = torch.Generator().manual_seed(Cin + Cout + taps)
    x = (torch.randn(B, T + taps - 1, Cin, generator=g)).to(F16).to(dev)
    w = (torch.randn(1, taps, Cin, cw, generator=g) / (taps * Cin) ** 0.5).to(F16).to(dev)
    bv = torch.randn(cw, generator=g).to(F16).to(dev)
    oa = torch.rand(cw, generator=g).to(dev) + 0.5
    oib = 1.0 / (oa + 1e-9)
    nws = a8.conv_cl_ws_bytes(B, T, Cin, Cout, taps, 1)
    assert not split or nws > 0
    ws = torch.empty(nws, dtype=torch.uint8, device=dev) if split else None
    y = torch.empty(B, T, Cout, dtype=F16, device=dev)
    plain = torch.zeros(B, T, cw, dtype=F16, device=dev)
    a8.conv_cl(x, w, bv, T, taps, 1, 1, y, ws=ws, out_snake=(oa, oib))
    tight = torch.empty(B, T, Cout, dtype=F16, device=dev)
    a8.conv_cl(x, w, bv, T, taps, 1, 1, tight, ws=ws)
    plain[..., :Cout] = tight
    want = torch.empty_like(plain)
    a8.snake_cat(plain, None, oa, oib, want)
    torch.cuda.synchronize()
    assert torch.equal(y, want[..., :Cout])
