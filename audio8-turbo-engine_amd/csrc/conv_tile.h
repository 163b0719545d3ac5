// The 128 x 192 / 256 x 96 tile convolution (conv_tile.hip) behind a8_conv_cl and a8_ru_cl.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace a8 {

// One launch. Strides in elements; x rows b of Tin rows each lie back to back (s_xb == Tin * s_xt), so the row at
// time t of batch row b is flat row b * Tin + t.
struct ConvTileArgs {
  const uint16_t *x;
  int64_t s_xt;
  const uint16_t *w;  // [phase][tap][k][n]
  int64_t s_wp, s_wt, s_wc;
  const uint16_t *bias, *res;
  int64_t s_rb, s_rt;
  uint16_t *y;
  int64_t s_yb, s_yt;
  int M, TR, Tin, Cin, Cout, taps, dil, ph;
  float *part;  // split-K partials [share][phase][M][Cout] (no bias, residual or rounding), else null
  int ksplit;
  uint32_t x_span, w_span;
  // the residual unit's second half (RU): w2 [k][n], its bias, the snake before it
  const uint16_t *w2, *b2;
  const float *a2, *ib2;
  uint32_t w2_span;
  const float *oa, *oib;  // a snake over the stored (fp16) outputs, or null
};

// mt: 32-row groups of a wave. xkb: KiB of LDS one 32-channel slice of a tile's input rows takes (16 rows a KiB); 0:
// the tile kernel does not take the shape. narrow: tiles of 128 mt rows x 96 channels instead of 64 mt x 192.
struct ConvTilePlan {
  int mt, xkb, ksplit;
  bool narrow;
  int64_t ws_bytes;
};
// ws_bytes: what the caller's workspace holds (K is split no further); other_us: the time the launch would take on
// k_conv_cl in one pass, infinite where that one would split K (its split never beat the tile's, however few shares
// the workspace leaves the tile).
ConvTilePlan conv_tile_plan(int64_t M, int TR, int Tin, int Cin, int Cout, int taps, int dil, int ph, bool ru,
                            int64_t ws_bytes, double other_us);
// The split-K workspace conv_tile_plan would ask for, whatever the input rows.
int64_t conv_tile_ws_bytes(int64_t M, int Cin, int Cout, int taps, int ph);
int conv_tile_launch(const ConvTilePlan &pl, const ConvTileArgs &a, bool ru, hipStream_t stream);

}  // namespace a8
