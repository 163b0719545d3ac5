// Fused store + decode over caches of at most 32 positions (the fast AR's 10), included by decode_stream.hip.
//
// A launch over so few keys is latency alone: its start, the row's metadata, the table rows at its position, then the
// arithmetic. One wave per (row, kv head) with nothing that a longer row needs (no ring, no next chunk, no merge): the
// qkv and bias chunks, which depend on no metadata, and (without a row map) K and V are requested together with the
// metadata, and only the table rows wait for the position; the streaming kernel asked for its 64-key tile first and
// for the qkv chunks after the position. 192 rows x 10 positions in a graph: 5.9 -> 3.8 us per layer; a two-token pass
// and 8 one-token passes of 4 layers 240 -> 169 us (171 with the last 64 bytes of the arguments left cold). Half a
// 64-key tile: the same operand layout, products and sum order as compute_step's first 32 keys (the others would add
// zeros), so the same bits.
#pragma once
#include "fused_qkv.h"

namespace a8 {

constexpr int kShortKeys = 32;

__global__ __launch_bounds__(64) void k_decode_short(uint16_t *kc, uint16_t *vc, int64_t s_kb, int64_t s_kh,
                                                     int cache_rows, int cache_len, const int32_t *__restrict__ lens,
                                                     const int32_t *__restrict__ rowmap, uint16_t *__restrict__ out,
                                                     int64_t s_ob, int64_t s_oh, int b, int nq, int nkv, int group,
                                                     float sl2, StoreIn si) {
  warm_kernargs<208>();  // the explicit arguments above span 0x00-0xcf
  __shared__ __attribute__((aligned(16))) uint16_t vt[kShortKeys * 64];
  const int lane = threadIdx.x, row = blockIdx.x / nkv, kh = blockIdx.x - row * nkv;
  TileLane tl;
  tl.init(lane);
  const int r16 = tl.r16, g = tl.g;
  const uint32_t rb = (uint32_t)b * 4u, ro = (uint32_t)row * 4u;
  int craw = row;
  if (rowmap) craw = bld4(make_rsrc(rowmap, rb), ro);
  const int praw = bld4(make_rsrc(si.pos, rb), ro), sraw = bld4(make_rsrc(si.slot, rb), ro);
  const int lraw = bld4(make_rsrc(lens, rb), ro);
  // the lane's chunks of the row's qkv and of the bias (load_qkv_raw's, the tables apart)
  const int H = nq + 2 * nkv;
  const uint32_t og = 16u * g, ho = (uint32_t)fused_lane_head(r16, kh, group, nq, nkv) * 128u + og;
  const rsrc_t xr = make_rsrc(si.qkv + (int64_t)row * si.s_qkv, (uint32_t)H * 128u);
  const rsrc_t br = make_rsrc(si.bias, si.bias ? (uint32_t)H * 128u : 0u);
  QkvRaw r;
  r.w[0] = bld16(xr, ho);
  r.w[1] = bld16(xr, ho + 64u);
  r.bb[0] = bld16(br, ho);
  r.bb[1] = bld16(br, ho + 64u);
  // K as the score operands (rows 8(r16/4) + 4t + r16%4), V row by row (row 8j + lane/8, chunk lane%8)
  const int crow = __builtin_amdgcn_readfirstlane(craw);
  const bool have = crow >= 0 && crow < cache_rows;
  const int64_t cb = (int64_t)(have ? crow : 0) * s_kb + (int64_t)kh * s_kh;
  const uint32_t span = have ? (uint32_t)cache_len * kRow : 0u;
  const rsrc_t kr = make_rsrc_wave(kc + cb, span), vr = make_rsrc_wave(vc + cb, span);
  u32x4 ka[2][2], va[4];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    ka[t][0] = bld16(kr, tl.kb0 + 4u * t * kRow);
    ka[t][1] = bld16(kr, tl.kb0 + 4u * t * kRow + 64u);
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) va[j] = bld16(vr, (uint32_t)(8 * j + (lane >> 3)) * kRow + 16u * (lane & 7));
  const int p = __builtin_amdgcn_readfirstlane(praw);
  const bool pv = p >= 0 && p < si.n_tab;
  const rsrc_t cr = make_rsrc_wave(si.cos_tab + (int64_t)(pv ? p : 0) * si.s_cs, pv ? 128u : 0u);
  const rsrc_t sr = make_rsrc_wave(si.sin_tab + (int64_t)(pv ? p : 0) * si.s_cs, pv ? 128u : 0u);
  r.cs[0] = bld16(cr, og);
  r.cs[1] = bld16(cr, og + 64u);
  r.sn[0] = bld16(sr, og);
  r.sn[1] = bld16(sr, og + 64u);
  const int srow = __builtin_amdgcn_readfirstlane(sraw);
  const int hi = have ? min(max(__builtin_amdgcn_readfirstlane(lraw), 0), cache_len) : 0;
  u32x4 q0, q1;
  KVPatch pt;
  apply_qkv_raw(si, r, true, row, kh, p, srow, crow, cache_rows, cache_len, group, kc, vc, s_kb, s_kh, 64, true, tl, q0,
                q1, pt);
  f32x4 o[4];
#pragma unroll
  for (int dt = 0; dt < 4; ++dt) o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  float ps = 0.f;
  if (hi > 0) {  // (uniform)
    if (pt.col >= 0) {  // the new key (uniform): its K row from lane kLaneK of the group
      const int src = 16 * g + kLaneK, ts = (pt.col >> 2) & 1;
      const bool mine = r16 == 4 * (pt.col >> 3) + (pt.col & 3);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t klo = (uint32_t)__shfl((int)pt.lo[e], src), khi = (uint32_t)__shfl((int)pt.hi[e], src);
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          ka[t][0][e] = mine && t == ts ? klo : ka[t][0][e];
          ka[t][1][e] = mine && t == ts ? khi : ka[t][1][e];
        }
      }
    }
    // V into LDS in load_tile's layout, rows past the length as zeros, the new row from the kLaneV lanes
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int vrow = 8 * j + (lane >> 3), s = (vrow & 3) ^ (j & 1);
      const u32x4 z{0u, 0u, 0u, 0u};
      st16(vt + vrow * 64 + 8 * ((lane & 7) ^ (2 * s)), vrow < hi ? va[j] : z);
    }
    wave_lds_fence();
    if (pt.col >= 0 && pt.col < hi && r16 == kLaneV) {
      const int s = (pt.col & 3) ^ ((pt.col >> 3) & 1);
      st16(vt + pt.col * 64 + 8 * (g ^ (2 * s)), pt.lo);
      st16(vt + pt.col * 64 + 8 * ((4 + g) ^ (2 * s)), pt.hi);
    }
    f32x4 sc[2];
    float mt = kNegInf;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      f32x4 a = mfma16x16x32(ka[t][0], q0, f32x4{0.f, 0.f, 0.f, 0.f});
      a = mfma16x16x32(ka[t][1], q1, a);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (8 * g + 4 * t + i >= hi) a[i] = kNegInf;
      mt = fmaxf(mt, fmaxf(fmaxf(a[0], a[1]), fmaxf(a[2], a[3])));
      sc[t] = a;
    }
    mt = max_over_groups(mt);
    const float mc = mt * sl2;
    u32x4 pB;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      float pr[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        pr[i] = fast_exp2(__builtin_fmaf(sc[t][i], sl2, -mc));
        ps += pr[i];
      }
      pB[2 * t] = pack_bf16x2(pr[0], pr[1]);
      pB[2 * t + 1] = pack_bf16x2(pr[2], pr[3]);
    }
    wave_lds_fence();
    const char *vb = reinterpret_cast<const char *>(vt);
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) {
      const u32x2 lo = lds_tr16(vb + tl.vt[dt]), h2 = lds_tr16(vb + tl.vt[dt] + 4 * kRow);
      o[dt] = mfma16x16x32(u32x4{lo[0], lo[1], h2[0], h2[1]}, pB, o[dt]);
    }
  }
  const float den = sum_over_groups(ps);  // (no key: 0 / 0, as every schedule writes)
  if (r16 >= group) return;
  uint16_t *op = out + (int64_t)row * s_ob + (int64_t)(kh * group + r16) * s_oh + 4 * g;
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
    st8(op + 16 * dt, u32x2{pack_bf16x2(o[dt][0] / den, o[dt][1] / den), pack_bf16x2(o[dt][2] / den, o[dt][3] / den)});
}

}  // namespace a8
