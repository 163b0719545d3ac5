"""The lines between kernels that the host draws, on a device of 256 compute units: the auto schedule's
(DecodeAttention.schedule) and the tile convolution's (a8_conv_tile_query). No GPU."""
from __future__ import annotations

import ctypes

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


def conv_tile(a8, B, Tin, TR, Cin, Cout, taps, dil, ph, ru=0, ws=0):
    """(32-row groups a wave, KiB of an input slice, K shares) of the tile kernel; (0, 0, 1): the general kernel."""
    o = [ctypes.c_int() for _ in range(3)]
    assert a8.load_library().a8_conv_tile_query(B, Tin, TR, Cin, Cout, taps, dil, ph, ru, ws, *map(ctypes.byref, o)) == 0
    return tuple(v.value for v in o)


# Decoder convs and others, (Cin, Cout, taps, phases), and per row count which kernel a call without a workspace was
# measured faster on: k_conv_cl while its 64-row tiles take at most two workgroups a compute unit.
@pytest.mark.parametrize("conv,general,tile", [
    ((1024, 1536, 7, 1), (20, 768, 1280), (1536, 2048, 6144)),
    ((1536, 768, 2, 8), (20, 128, 256), (384, 512, 1536)),
    ((768, 768, 7, 1), (20, 256, 2560), (3072, 6144)),
    ((768, 384, 2, 8), (20, 128, 640, 1024), (896, 1152)),
    ((384, 384, 7, 1), (20, 1024, 5120), (6144, 12288)),
    ((384, 192, 2, 4), (20, 2560, 4096), (4608, 6144)),
    ((192, 192, 7, 1), (20, 4096, 16384), (18432, 49152)),
    ((192, 96, 2, 2), (20, 8192, 16384), (18432, 49152)),
    ((96, 96, 7, 1), (20, 16384, 32768), (36864, 65536)),
    ((768, 768, 1, 1), (20, 3072, 4096), (5120, 12288)),
    ((480, 480, 3, 1), (20, 3072, 6400), (7168, 16384)),
])
def test_conv_without_a_workspace(a8, conv, general, tile):
    cin, cout, taps, ph = conv
    for m in general:
        assert conv_tile(a8, 1, m + taps - 1, m, cin, cout, taps, 1, ph)[0] == 0, m
    for m in tile:
        mt, _, ksplit = conv_tile(a8, 1, m + taps - 1, m, cin, cout, taps, 1, ph)
        assert mt in (2, 3) and ksplit == 1, m


def test_conv_takes_the_shares_its_workspace_holds(a8):
    """A workspace too small for the tile's own choice of shares: as many as it holds, or one pass of the faster kernel
    (256 rows of 768 channels, 7 taps: 62.3 us as one pass of tiles, 22.9 split by the general kernel, 22.4 by tiles)."""
    lib, m, c = a8.load_library(), 256, 768
    need, share = lib.a8_conv_cl_ws_bytes(1, m, c, c, 7, 1), 4 * m * c
    want = conv_tile(a8, 1, m + 6, m, c, c, 7, 1, 1, ws=need)[2]
    assert want > 6 and need >= want * share
    for k in range(3, want + 1):
        for ws in (k * share, (k + 1) * share - 1):
            assert conv_tile(a8, 1, m + 6, m, c, c, 7, 1, 1, ws=ws)[2] == k
    assert conv_tile(a8, 1, m + 6, m, c, c, 7, 1, 1, ws=share)[0] == 0
    # too few steps for k_conv_cl to split, and one pass of it beats the tile's split
    assert conv_tile(a8, 1, 3074, 3072, 480, 480, 3, 1, 1, ws=1 << 30)[0] == 0
