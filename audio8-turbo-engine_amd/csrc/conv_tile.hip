// The tile convolution behind a8_conv_cl / a8_ru_cl where the channel counts divide its tiles: an implicit GEMM
// (M = B * TR rows, N = Cout, K = taps * Cin) as Y^T = W^T . X^T on v_mfma_f32_32x32x16_f16.
//
// A workgroup is four waves of 64 or 96 rows x 96 channels each (2 or 3 x 3 MFMA tiles), either 2 x 2 (128 / 192 rows
// x 192 channels) or 4 x 1 (256 / 384 x 96, where the 96-channel groups of all phases are odd in number); two
// workgroups per compute unit. A column half is one 96-channel group of one phase, so a transposed conv's phases share
// their input rows. K runs channel slice by channel slice (32 channels), and within a slice tap by tap, so a slice of
// the tile's input rows is brought into LDS once and every tap reads it there, j * dil rows further down:
//   * X slice: the tile's flat rows f0 .. (its own, the gaps between batch rows, the last tap's reach), 64 bytes a
//     row, the 16-byte chunk c of row r at position c ^ (r / 4 % 4): any 16 consecutive rows of one chunk then fall
//     on distinct banks. Two areas: the next slice is requested at the slice's first tap.
//   * W slice: 32 k rows x 96 channels per column half, 192 bytes (48 banks) a row: the 4 rows x 32 channels that
//     half a wave's ds_read_b64_tr_b16 touches fall on 64 distinct banks with no padding. A ring of three, requested
//     two steps ahead.
// Both come by DMA (buffer_load ... lds). The DMA is written as asm: the compiler does not see that it writes LDS,
// so it does not drain it before the operand reads; the waits are counted by hand (requests complete in order).
// One barrier a step (12 or 18 MFMAs a wave).
//
// What bounds it: LDS and the MFMAs, not fully overlapped at two waves per SIMD. Skipping parts of the 64-row form
// (384 channels, 7 taps, 49152 rows: 108-114 us): no LDS operand reads 87, no W requests 95, no MFMAs 82, MFMAs alone
// 60. Hence the 96-row wave: a third fewer W requests and 12 KB of operand reads per 18 MFMAs instead of 10 per 12,
// 94 us. Steps in pairs (half the barriers) and a raised wave priority over the MFMAs changed nothing.
// Against k_conv_cl (each wave the whole column width of 16 or 32 rows, X operands from memory again for every tap;
// graph replays, 192 batch rows of 4 frames): 384 channels k 7 131 -> 94 us (1.08 PFLOP/s; a large fp16 matrix product
// on this card: 1.45), 768 channels k 7 92 -> 72, the stride-8 transposed convs 78 -> 46 and 83 -> 61, stride 4
// 96 -> 70, stride 2 77 -> 48, the input conv 51 -> 37; the residual units of 192 / 96 channels 172 -> 135 and
// 114 -> 88 (64-row waves, the two column halves' whole rows exchanged at once: 141 and 92). 24 batch rows: 37 -> 32, 25 -> 24, 20 -> 20, 34 -> 25, 28 -> 17, 14 -> 12.6, 25.5 -> 20.
#include "conv_tile.h"

#include "fp16_ops.h"

namespace a8 {

namespace {

constexpr int kHalf = 32 * 96 * 2;  // bytes of a W slice's column half

typedef uint32_t rsrc_words_t __attribute__((ext_vector_type(4)));

// Raw buffer descriptor as four words (asm operands; same fields as make_rsrc).
__device__ __forceinline__ rsrc_words_t rsrc_words(const void *base, uint32_t bytes) {
  const uint64_t p = reinterpret_cast<uint64_t>(base);
  return rsrc_words_t{(uint32_t)p, (uint32_t)(p >> 32) & 0xffffu, bytes, 0x00020000u};
}

// bld16_lds as asm (see the head of the file). M0 is an operand, so the compiler knows what the asm needs there and
// sees to it again if it uses M0 itself. s_nop: the wait states a vector-written scalar operand and M0 need, which the
// compiler does not add inside asm.
__device__ __forceinline__ void dma16(rsrc_words_t r, uint32_t lds, uint32_t voff, uint32_t soff) {
  lds = __builtin_amdgcn_readfirstlane(lds);  // (uniform; the compiler may have computed them in vector registers)
  soff = __builtin_amdgcn_readfirstlane(soff);
  asm volatile(
      "s_nop 4\n\t"
      "buffer_load_dwordx4 %1, %2, %3 offen lds"
      :
      : "{m0}"(lds), "v"(voff), "s"(r), "s"(soff)
      : "memory");
}

__device__ __forceinline__ void swap32(uint32_t &a, uint32_t &b) {
  const auto s = __builtin_amdgcn_permlane32_swap(a, b, false, false);
  a = s[0];
  b = s[1];
}

}  // namespace

// WMW: waves along the rows (2: 128 x 192 tile, 4: 256 x 96). XKB: KiB of one X slice area. RU: a residual unit, as
// k_conv_cl's: h = acc + bias (fp32), the snake with a2 / ib2 (one fp16 rounding), then out = h . w2 + b2 + res; the
// tile holds the whole row (Cout = BN).
template <int WMW, int MT, int XKB, bool RU>
__global__ __launch_bounds__(256, 2) void k_conv_tile(const ConvTileArgs a) {
  constexpr int NH = 4 / WMW, BM = 32 * MT * WMW;
  constexpr int kW = NH * kHalf, kWI = NH * 6;          // a W slice: bytes, DMA instructions
  constexpr int WR = (kWI + 3) / 4, XI = (XKB + 3) / 4;  // instructions per wave and slice (the last repeated)
  constexpr int kMainLds = 3 * kW + 2 * XKB * 1024, kRuLds = (NH == 2 ? 2 * 8 * MT * 1024 : 0) + 2 * kW;
  constexpr int kLds = RU && kRuLds > kMainLds ? kRuLds : kMainLds;
  static_assert(kLds <= 80 * 1024, "two workgroups per compute unit");
  __shared__ __attribute__((aligned(16))) char smem[kLds];
  const uint32_t lds0 = (uint32_t)reinterpret_cast<uintptr_t>(smem);
  constexpr int kXOff = 3 * kW;  // W ring, then the two X areas
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = NH == 2 ? wv >> 1 : wv, wn = NH == 2 ? wv & 1 : 0;
  const int r32 = lane & 31, h = lane >> 5, l15 = lane & 15;
  // tile: rows m0 .., column groups of 96 channels cg .. (of ph * Cout / 96: phase by phase), k share ks
  const int ng = a.Cout / 96;
  const int nmt = (a.M + BM - 1) / BM, ct = blockIdx.x / nmt, mt = blockIdx.x - ct * nmt;
  const int ks = blockIdx.y, m0 = mt * BM, cg = ct * NH;
  const int KC = a.Cin >> 5, taps = a.taps;
  const int kb = (int)((int64_t)KC * ks / a.ksplit), ke = (int)((int64_t)KC * (ks + 1) / a.ksplit);
  const int f0 = (m0 / a.TR) * a.Tin + m0 % a.TR;

  const rsrc_words_t xr = rsrc_words(a.x, a.x_span), wr = rsrc_words(a.w, a.w_span);
  // X: instruction q fills rows 16 q .. + 15 of an area (lane: row lane / 4, chunk position lane % 4)
  const uint32_t xvo = (uint32_t)(((int64_t)(f0 + (lane >> 2)) * a.s_xt + 8 * ((lane & 3) ^ (lane >> 4))) * 2);
  auto issue_x = [&](int kc, int area) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < XI; ++i) {
      const int q = 4 * i + wv < XKB ? 4 * i + wv : XKB - 1;
      // (the rows in the vector offset: the range check subtracts the scalar one from the size, and rows past a
      // short input could leave it negative)
      dma16(xr, lds0 + kXOff + area * (XKB * 1024) + q * 1024, xvo + (uint32_t)(q * 32 * (int)a.s_xt),
            (uint32_t)kc * 64);
    }
  };
  // W: instruction q covers chunks 64 (q % 6) .. of column half q / 6: k row chunk / 12, channels 8 (chunk % 12)
  uint32_t wvo[WR];
  int wq[WR];
#pragma unroll
  for (int i = 0; i < WR; ++i) {
    wq[i] = 4 * i + wv < kWI ? 4 * i + wv : kWI - 1;
    const int c = (wq[i] % 6) * 64 + lane, g = cg + wq[i] / 6, pg = g / ng;
    wvo[i] = (uint32_t)(((int64_t)pg * a.s_wp + (int64_t)(c / 12) * a.s_wc + (g - pg * ng) * 96 + 8 * (c % 12)) * 2);
  }
  auto issue_w = [&](rsrc_words_t r, uint32_t off, uint32_t so) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < WR; ++i) dma16(r, lds0 + off + wq[i] * 1024, wvo[i], so);
  };
  auto w_off = [&](int kc, int j) __attribute__((always_inline)) -> uint32_t {
    return (uint32_t)(((int64_t)j * a.s_wt + (int64_t)kc * 32 * a.s_wc) * 2);
  };
  // this lane's rows: LDS row of tap 0 (rows past M read row 0)
  int rb[MT], mrow[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    mrow[i] = m0 + (wm * MT + i) * 32 + r32;
    rb[i] = mrow[i] < a.M ? (mrow[i] / a.TR) * a.Tin + mrow[i] % a.TR - f0 : 0;
  }
  f32x16 acc[3][MT];
#pragma unroll
  for (int nt = 0; nt < 3; ++nt)
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[nt][i][e] = 0.f;

  // A operand (W^T): k rows 8h + l15 / 4 (+4), channels 16 (lane / 16 % 2) + 4 (l15 % 4) of a 32-channel tile
  const int aoff = wn * kHalf + (8 * h + (l15 >> 2)) * 192 + (16 * ((lane >> 4) & 1) + 4 * (l15 & 3)) * 2;
  auto next = [&](int &kc, int &j) __attribute__((always_inline)) {  // the step after (past the end: the last again)
    if (j + 1 < taps) {
      ++j;
    } else if (kc + 1 < ke) {
      j = 0;
      ++kc;
    }
  };
  issue_x(kb, 0);
  issue_w(wr, 0, w_off(kb, 0));
  int kc2 = kb, j2 = 0;  // the step requested last
  next(kc2, j2);
  issue_w(wr, kW, w_off(kc2, j2));
  uint32_t cur = 0, nxt = 2 * kW;  // ring offsets: this step's slice, the one to fill
  for (int kc = kb; kc < ke; ++kc) {
    const bool more = kc + 1 < ke;
    const char *xs = smem + kXOff + ((kc - kb) & 1) * (XKB * 1024);
    for (int j = 0; j < taps; ++j) {
      // this step's W slice (and at j = 0 its X slice) has landed when only what was requested after it is
      // outstanding: the next step's W slice, and at j = 1 the next X slice, requested before that
      if (j == 1 && more)
        wait_vmcnt<WR + XI>();
      else
        wait_vmcnt<WR>();
      lds_barrier();
      const char *wp = smem + cur + aoff;
      uint32_t xa[MT];
      u32x4 bx[2][MT], av[2][3];
      auto read = [&](int u) __attribute__((always_inline)) {
#pragma unroll
        for (int nt = 0; nt < 3; ++nt) {
          const u32x2 lo = lds_tr16(wp + u * 16 * 192 + nt * 64), hi = lds_tr16(wp + u * 16 * 192 + nt * 64 + 4 * 192);
          av[u][nt] = u32x4{lo[0], lo[1], hi[0], hi[1]};
        }
#pragma unroll
        for (int i = 0; i < MT; ++i) bx[u][i] = lds_ld16(xs + (xa[i] ^ (u << 5)));
      };
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        const int row = rb[i] + j * a.dil;
        xa[i] = (uint32_t)(row * 64 + ((h ^ ((row >> 2) & 3)) << 4));
      }
      read(0);  // (the requests below are issued while these reads return)
      if (j == 0 && more) issue_x(kc + 1, (kc + 1 - kb) & 1);
      next(kc2, j2);
      issue_w(wr, nxt, w_off(kc2, j2));
      read(1);
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int nt = 0; nt < 3; ++nt)
#pragma unroll
          for (int i = 0; i < MT; ++i) acc[nt][i] = mfma32x32x16_f16(av[u][nt], bx[u][i], acc[nt][i]);
      nxt = cur;  // the slot just read is filled next
      cur = cur == 2 * kW ? 0 : cur + kW;
    }
  }
  wait_vmcnt<0>();  // the last steps' repeated requests still write LDS
  const uint16_t *bias = a.bias;
  if constexpr (RU) {
    // h in B-operand order: of 16-channel step s = 2 nt + q, slot 8h' + e of this wave's channels is channel
    // 32 nt + 16 q + 8 (e / 4) + 4 h' + e % 4, which lane half h' already holds; w2's rows are read in that order.
    u32x4 hb[6][MT];
#pragma unroll
    for (int nt = 0; nt < 3; ++nt)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int n = wn * 96 + 32 * nt + 8 * q + 4 * h;
        const u32x2 bv = *reinterpret_cast<const u32x2 *>(bias + n);
        const f32x4 av = *reinterpret_cast<const f32x4 *>(a.a2 + n), iv = *reinterpret_cast<const f32x4 *>(a.ib2 + n);
        const float bb[4] = {h_lo(bv[0]), h_hi(bv[0]), h_lo(bv[1]), h_hi(bv[1])};
#pragma unroll
        for (int i = 0; i < MT; ++i) {
          float hv[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float v = acc[nt][i][4 * q + e] + bb[e];
            const float sv = sin_hw(v * av[e]);
            hv[e] = v + iv[e] * sv * sv;
          }
          hb[2 * nt + (q >> 1)][i][2 * (q & 1)] = pack_f16x2(hv[0], hv[1]);
          hb[2 * nt + (q >> 1)][i][2 * (q & 1) + 1] = pack_f16x2(hv[2], hv[3]);
        }
      }
#pragma unroll
    for (int nt = 0; nt < 3; ++nt)
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[nt][i][e] = 0.f;
    const rsrc_words_t w2r = rsrc_words(a.w2, a.w2_span);
    const int aoff2 = wn * kHalf + (4 * h + (l15 >> 2)) * 192 + (16 * ((lane >> 4) & 1) + 4 * (l15 & 3)) * 2;
    constexpr int S2 = 3 * NH;  // 32-channel steps over the row
    // Two column halves: a wave holds half of its rows' channels, its partner (wave ^ 1) the other half. It starts
    // with its own three slices, from registers, then takes the partner's through LDS, a 32-channel slice at a time
    // (two slice areas: the third goes out once the first has been read everywhere). So in step s2 column half hh
    // multiplies w2's rows of slice 3 hh + s2, then of slice 3 (1 - hh) + s2 - 3.
    constexpr int kEx = 8 * MT * 1024, kH = NH == 2 ? 2 * kEx : 0;
    auto issue_w2 = [&](int s2, int slot) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < WR; ++i) {
        const int half = wq[i] / 6;
        const int slice = NH == 1 ? s2 : s2 < 3 ? 3 * half + s2 : 3 * (1 - half) + s2 - 3;
        dma16(w2r, lds0 + kH + slot * kW + wq[i] * 1024, wvo[i], (uint32_t)((int64_t)slice * 32 * a.s_wc * 2));
      }
    };
    auto ex_at = [&](int c, int wave, int u, int i) __attribute__((always_inline)) {
      return smem + (c & 1) * kEx + (((wave * 2 + u) * MT + i) * 64 + lane) * 16;
    };
    auto ex_put = [&](int c) __attribute__((always_inline)) {
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int i = 0; i < MT; ++i)
          *(__attribute__((address_space(3))) u32x4 *)ex_at(c, wv, u, i) = hb[2 * c + u][i];
    };
    lds_barrier();  // every wave is done with the ring
    issue_w2(0, 0);
    if constexpr (NH == 2) {
      ex_put(0);
      ex_put(1);
    }
#pragma unroll
    for (int s2 = 0; s2 < S2; ++s2) {
      wait_vmcnt<0>();
      lds_barrier();
      if (s2 + 1 < S2) issue_w2(s2 + 1, (s2 + 1) & 1);
      if (NH == 2 && s2 == 4) ex_put(2);
      const char *wp = smem + kH + (s2 & 1) * kW + aoff2;
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        u32x4 bx[MT];
#pragma unroll
        for (int i = 0; i < MT; ++i) bx[i] = s2 < 3 ? hb[(2 * s2 + u) % 6][i] : lds_ld16(ex_at(s2 - 3, wv ^ 1, u, i));
#pragma unroll
        for (int nt = 0; nt < 3; ++nt) {
          const u32x2 lo = lds_tr16(wp + u * 16 * 192 + nt * 64), hi = lds_tr16(wp + u * 16 * 192 + nt * 64 + 8 * 192);
          const u32x4 av = u32x4{lo[0], lo[1], hi[0], hi[1]};
#pragma unroll
          for (int i = 0; i < MT; ++i) acc[nt][i] = mfma32x32x16_f16(av, bx[i], acc[nt][i]);
        }
      }
    }
    bias = a.b2;
  }
  // acc[nt][i]: lane (r32, h) holds row mrow[i], channels nb + 32 nt + 8 q + 4 h + e (element 4 q + e)
  const int p = (cg + wn) / ng, nb = (cg + wn - p * ng) * 96;
  if (a.part) {
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      if (mrow[i] >= a.M) continue;
      float *prow = a.part + ((int64_t)(ks * a.ph + p) * a.M + mrow[i]) * a.Cout + nb + 4 * h;
#pragma unroll
      for (int nt = 0; nt < 3; ++nt)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          *reinterpret_cast<f32x4 *>(prow + 32 * nt + 8 * q) =
              f32x4{acc[nt][i][4 * q], acc[nt][i][4 * q + 1], acc[nt][i][4 * q + 2], acc[nt][i][4 * q + 3]};
    }
    return;
  }
  // Two 8-channel groups (16 qq and 16 qq + 8) at a time: swapping between the lane halves leaves lane half h with
  // all eight channels of group 16 qq + 8 h, one 16-byte store (and residual load) a lane.
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const bool ok = mrow[i] < a.M;
    const int m = ok ? mrow[i] : a.M - 1;
    const int b = m / a.TR;
    const int64_t orow = (int64_t)(m - b * a.TR) * a.ph + p;
    uint16_t *yrow = a.y + (int64_t)b * a.s_yb + orow * a.s_yt + nb + 8 * h;
    const uint16_t *rrow = a.res ? a.res + (int64_t)b * a.s_rb + orow * a.s_rt + nb + 8 * h : nullptr;
#pragma unroll
    for (int nt = 0; nt < 3; ++nt)
#pragma unroll
      for (int qq = 0; qq < 2; ++qq) {
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = acc[nt][i][8 * qq + e];
        if (bias) {
          const u32x2 b0 = *reinterpret_cast<const u32x2 *>(bias + nb + 32 * nt + 16 * qq + 4 * h);
          const u32x2 b1 = *reinterpret_cast<const u32x2 *>(bias + nb + 32 * nt + 16 * qq + 8 + 4 * h);
          v[0] += h_lo(b0[0]), v[1] += h_hi(b0[0]), v[2] += h_lo(b0[1]), v[3] += h_hi(b0[1]);
          v[4] += h_lo(b1[0]), v[5] += h_hi(b1[0]), v[6] += h_lo(b1[1]), v[7] += h_hi(b1[1]);
        }
        if (rrow) {
          u32x4 rv = *reinterpret_cast<const u32x4 *>(rrow + 32 * nt + 16 * qq);
          uint32_t r0 = rv[0], r1 = rv[1], r2 = rv[2], r3 = rv[3];
          swap32(r0, r2);
          swap32(r1, r3);
          v[0] += h_lo(r0), v[1] += h_hi(r0), v[2] += h_lo(r1), v[3] += h_hi(r1);
          v[4] += h_lo(r2), v[5] += h_hi(r2), v[6] += h_lo(r3), v[7] += h_hi(r3);
        }
        uint32_t o0 = pack_f16x2(v[0], v[1]), o1 = pack_f16x2(v[2], v[3]);
        uint32_t o2 = pack_f16x2(v[4], v[5]), o3 = pack_f16x2(v[6], v[7]);
        swap32(o0, o2);
        swap32(o1, o3);
        u32x4 o = u32x4{o0, o1, o2, o3};
        if (a.oa) o = snake8(o, a.oa + nb + 32 * nt + 16 * qq + 8 * h, a.oib + nb + 32 * nt + 16 * qq + 8 * h);
        if (ok) st16(yrow + 32 * nt + 16 * qq, o);
      }
  }
}

// Input rows (flat) a BM-row tile reaches: its own, the gaps of the batch-row boundaries inside it, the last tap's.
static int64_t tile_rows(int BM, int TR, int Tin, int taps, int dil) {
  const int64_t nb = TR % BM == 0 ? 0 : BM % TR == 0 ? BM / TR - 1 : (BM - 2) / TR + 1;
  return BM + nb * (Tin - TR) + (int64_t)(taps - 1) * dil;
}

// X slice area (KiB, 16 rows each) of tiles of mt row groups a wave; 0: two of them do not fit beside the W ring in
// half a compute unit's LDS.
static int tile_xkb(int TR, int Tin, int taps, int dil, bool narrow, bool ru, int mt) {
  const int64_t kib = (tile_rows((narrow ? 128 : 64) * mt, TR, Tin, taps, dil) + 15) / 16;
  const int small = narrow ? (mt == 3 ? 28 : 20) : mt == 3 ? 16 : 12, large = narrow || ru ? small : 22;
  return kib <= small ? small : kib <= large ? large : 0;
}

static int64_t tile_count(int64_t M, int Cout, int ph, int mt) {
  const int cols = ph * (Cout / 96), BM = (cols % 2 ? 128 : 64) * mt;
  return (M + BM - 1) / BM * (cols % 2 ? cols : cols / 2);
}

// The K shares of tiles of mt row groups, and the launch's time (us) by a model of the measured times (192 .. 1 batch
// rows through every conv of the decoder, k = 1 .. 16): 6.5 us, the steps (one 32-channel slice of one tap) of a
// share at the time a step takes with the compute unit's number of workgroups (mt 2: 0.40 us alone, 0.68 with a
// second; mt 3: 0.56 and 1.05; further rounds in proportion), and for split K the finish: 4 us and 0.35 us per MB of
// partials. It lies within 10 % of the measured times from 15 to 100 us; shares under 6 steps never paid. kmax: the
// shares the caller's workspace holds.
static int tile_split(int64_t M, int Cin, int Cout, int taps, int ph, int mt, int64_t kmax, double *us) {
  const int64_t tiles = tile_count(M, Cout, ph, mt), steps = (int64_t)(Cin / 32) * taps;
  const double mb = (double)ph * M * Cout * 4e-6;
  int best = 1;
  const bool split = steps >= 36 && (int64_t)ph * M * (Cout / 4) < ((int64_t)1 << 31);  // k_conv_fin
  for (int k = 1; k <= (split ? 16 : 1) && (k == 1 || k <= kmax); ++k) {
    if (k > 1 && (k > Cin / 32 || steps / k < 6)) break;
    const int64_t n = (tiles * k + 255) / 256;
    const double step = mt == 2 ? (n == 1 ? 0.40 : n == 2 ? 0.68 : 0.36 * n) : n == 1 ? 0.56 : 0.53 * n;
    const double t = 6.5 + (double)((steps + k - 1) / k) * step + (k > 1 ? 4 + 0.35 * mb * k : 0);
    if (k == 1 || t < *us) *us = t, best = k;
  }
  return best;
}

int64_t conv_tile_ws_bytes(int64_t M, int Cin, int Cout, int taps, int ph) {
  if (Cin % 32 || Cout % 96) return 0;
  int k = 1;
  double us;
  for (int mt = 2; mt <= 3; ++mt) {
    const int km = tile_split(M, Cin, Cout, taps, ph, mt, 16, &us);
    k = km > k ? km : k;
  }
  return k > 1 ? (int64_t)k * ph * M * Cout * 4 : 0;
}

ConvTilePlan conv_tile_plan(int64_t M, int TR, int Tin, int Cin, int Cout, int taps, int dil, int ph, bool ru,
                            int64_t ws_bytes, double other_us) {
  const ConvTilePlan none{0, 0, 1, false, 0};
  if (Cin % 32 || Cout % 96 || TR <= 0 || M <= 0 || (ru && Cout != 96 && Cout != 192)) return none;
  ConvTilePlan pl = none;
  pl.narrow = ph * (Cout / 96) % 2 != 0;
  double best = 0;
  for (int mt = 2; mt <= 3; ++mt) {
    const int xkb = tile_xkb(TR, Tin, taps, dil, pl.narrow, ru, mt);
    if (!xkb) continue;
    double us;
    const int k = tile_split(M, Cin, Cout, taps, ph, mt, ru ? 1 : ws_bytes / (ph * M * Cout * 4), &us);
    if (!pl.mt || us < best) pl.mt = mt, pl.xkb = xkb, pl.ksplit = k, best = us;
  }
  if (!pl.mt) return none;
  // Few tiles leave the chip idle. Split, that is in the model; in one pass k_conv_cl's 64-row tiles are then faster
  // (its time: other_us), as they are with few tiles and nothing for the taps to share or little to do: 1x1 of 24, 12
  // and 48 steps, 112 tiles 18.4 against 17.3, 12.9 against 12.0 and 29.9 against 28.6 us, 144 tiles 18.8 against
  // 19.7, 13.2 against 13.8 and 30.4 against 33.2. Residual units of 192 and 96 channels: 128 tiles 28.9 against 26.0
  // and 19.2 against 15.7, 160 tiles 29.9 against 35.6 and 19.7 against 20.0.
  const int64_t tiles = tile_count(M, Cout, ph, 2);
  if (ru ? tiles < 160
         : best >= other_us || (pl.ksplit == 1 && tiles < 128 && (taps == 1 || (int64_t)(Cin / 32) * taps < 36)))
    return none;
  if (pl.ksplit > 1) pl.ws_bytes = (int64_t)pl.ksplit * ph * M * Cout * 4;
  return pl;
}

template <int WMW, int MT, int XKB, bool RU>
static int launch(const ConvTileArgs &a, hipStream_t stream) {
  constexpr int BM = 32 * MT * WMW, NH = 4 / WMW;
  const dim3 grid((unsigned)((a.M + BM - 1) / BM) * (unsigned)(a.ph * (a.Cout / 96) / NH), (unsigned)a.ksplit);
  hipLaunchKernelGGL((k_conv_tile<WMW, MT, XKB, RU>), grid, dim3(256), 0, stream, a);
  return (int)hipGetLastError();
}

int conv_tile_launch(const ConvTilePlan &pl, const ConvTileArgs &a, bool ru, hipStream_t stream) {
  if (pl.narrow) {
    if (ru) return pl.mt == 3 ? launch<4, 3, 28, true>(a, stream) : launch<4, 2, 20, true>(a, stream);
    return pl.mt == 3 ? launch<4, 3, 28, false>(a, stream) : launch<4, 2, 20, false>(a, stream);
  }
  if (ru) return pl.mt == 3 ? launch<2, 3, 16, true>(a, stream) : launch<2, 2, 12, true>(a, stream);
  if (pl.mt == 3) return pl.xkb == 16 ? launch<2, 3, 16, false>(a, stream) : launch<2, 3, 22, false>(a, stream);
  return pl.xkb == 12 ? launch<2, 2, 12, false>(a, stream) : launch<2, 2, 22, false>(a, stream);
}

}  // namespace a8
