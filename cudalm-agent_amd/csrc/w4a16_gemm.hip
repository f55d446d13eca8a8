// Prefill-chunk W4A16 GEMM (MI355X, gfx950): the kernels on 32 x 32 MFMA tiles
// (one per call, and the K = 1024 one whose groups two wave sets share), the unit
// GEMM on 16 x 16 tiles with its forms for a group of projections and for SwiGLU,
// and launch_prefill and its like, which choose among them and the wide kernel
// (w4a16_gemm_wide.hip). This header describes the 32 x 32 kernels; the unit GEMM
// has its own further down.
//
// Contract (reference: tests/cuda/test_int4_gemv_bf16.cpp:54-69 applied row
// by row; the reference itself runs prefill one token at a time,
// src/runtime/qwen35_generator.cpp:107-125):
//   y[m,n] = bf16_rne( sum_k q[n,k] * f32(s[n,k/128]) * f32(x[m,k]) ).
//
// Matrix-core mapping. v_mfma_f32_32x32x16_bf16 multiplies 32 activation
// rows (A, m) by 32 weight rows (B, n) over 16 k: lane l = 32h + j holds
// A row j / B column j at k-block h (8 k) of the instruction, and D rows
// 8(r/4) + 4h + r%4 of column j in its 16 accumulators. One decoded weight
// dword (8 nibbles -> 4 bf16 pairs) therefore feeds 32 activation rows per
// instruction, twice as many as the 16 x 16 x 32 tiles of the decode
// kernels, and a wave that owns MT 32-row activation tiles feeds it to MT
// instructions: the decode VALU per FLOP is 1/(2 MT) of the 16 x 16 path.
//
// Same bits as every other kernel of the library. A 16 x 16 x 32 step over
// the k-blocks (b0, b1, b2, b3) of its four lane rows gives exactly the fp32
// result of two 32 x 32 x 16 steps, the first over (b0, b1) and the second
// over (b2, b3) (measured on gfx950: 0 of 1,048,576 outputs differ, random
// bf16 A, 1.5 + q/16 weights, zero and nonzero accumulators). So group g's
// chain runs, for each 16 x 16 step d = 0..3 of the decode kernels (lane
// row a holds k = 32a + 8d .. +7), the two halves e = 0, 1 over k-blocks
// 32(2e) + 8d and 32(2e+1) + 8d; it is seeded with the same offset chain
// (-1.5 * sum x per row and group, computed with the decode kernels' four
// 16 x 16 x 32 MFMAs into an LDS table); the epilogue is the canonical
// part = fma(s[n, g], tmp, part) in group order from 0 within an 8-group
// unit, total = 0 + part_u in unit order, y = bf16_rne(16 * total).
//
// Work decomposition. A workgroup of WVN waves owns TN = 32 WVN weight rows
// and TM = 32 MT activation rows. Per 8-group unit (1024 k): the tile's x
// is staged once into LDS in pair order, the waves split the offset chains
// of the unit's (group, 16-row) pairs into an LDS table, and each wave
// decodes its 32 rows' weights once per k-block and runs MT chains per
// group. Weights of the unit are loaded before the x staging completes.
// At K = 1024 (one unit) w4a16_gemm32_split_kernel runs instead: the
// unit's groups are split over two wave sets, which hand the canonical fma
// chain from one to the other through LDS.

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "cudalm_w4a16.h"
#include "hip_common.h"
#include "w4a16_device.h"

namespace cudalm_hip {
namespace {

constexpr int kPB = kUnit * 16 + 1;  // LDS row pitch of one unit of x, 16-byte blocks (padded)

template <int WVN, int MT>
constexpr size_t gemm32_lds_bytes() {
  return static_cast<size_t>(32 * MT) * kPB * 16 + static_cast<size_t>(kUnit) * 32 * MT * 4;
}

// WVN waves along n, each owning NB 32-row weight tiles; MT 32-row
// activation tiles per workgroup (every wave runs all of them).
template <class Act, int WVN, int MT, int NB, bool PACKED, bool SVEC>
__global__ __launch_bounds__(WVN * 64) void w4a16_gemm32_kernel(
    const uint8_t* __restrict__ W, const uint16_t* __restrict__ S,
    const uint16_t* __restrict__ X, uint16_t* __restrict__ Y, int N, int K, int M) {
  constexpr int NT = WVN * 64;
  constexpr int TM = 32 * MT;
  extern __shared__ u32x4_t lds[];  // x [TM][kPB], then the offset table [8 groups][TM] f32
  u32x4_t* xs = lds;
  float* corr = reinterpret_cast<float*>(lds + TM * kPB);

  const int G = K >> 7;
  const int U = (G + kUnit - 1) / kUnit;
  const int lane = threadIdx.x & 63;
  const int wave = wave_id();
  const int tid = static_cast<int>(threadIdx.x);
  const int j = lane & 31, h = lane >> 5;      // 32 x 32 operand lane: row / column j, k-block h
  const int i16 = lane & 15, a16 = lane >> 4;  // 16 x 16 operand lane (offset chains)
  const int m0 = blockIdx.y * TM;
  const int mrows = min(TM, M - m0);
  const int nbase = (blockIdx.x * WVN + wave) * 32 * NB;  // this wave's first weight row
  const bool wave_ok = nbase < N;

  // lane addresses at group 0 of weight row n = nbase + 32 nb + j: chunk
  // a = h (k 32h .. 32h+31 of a group) and chunk a = 2 + h
  const uint8_t* w_lo[NB];
  const uint8_t* w_hi[NB];
  const uint8_t* s_row[NB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    const int n = nbase + 32 * nb + j;
    if constexpr (PACKED) {
      const int t16 = min(n, N - 1) >> 4, r16 = n & 15;
      const uint8_t* tile = W + static_cast<size_t>(t16) * packed_tile_bytes(G);
      w_lo[nb] = tile + 16 * (16 * h + r16);
      w_hi[nb] = tile + 16 * (16 * (2 + h) + r16);
      s_row[nb] = tile + static_cast<size_t>(G) * 1024 + r16 * packed_scale_pitch(G);
    } else {
      const int row = min(n, N - 1);
      w_lo[nb] = W + static_cast<size_t>(row) * (K >> 1) + 16 * h;
      w_hi[nb] = w_lo[nb] + 32;
      s_row[nb] = reinterpret_cast<const uint8_t*>(S + static_cast<size_t>(row) * G);
    }
  }
  constexpr int kStep = PACKED ? 1024 : 64;  // bytes between groups of one lane

  const f32x16_t zero16 = {};
  f32x16_t acc[NB][MT];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[nb][mt] = zero16;

  constexpr int NBLK = TM * kUnit * 16;  // 16-byte x blocks of one unit
  static_assert(NBLK % NT == 0, "staging covers the tile exactly");
  constexpr int BPT = NBLK / NT;         // x blocks staged per thread per unit
  constexpr int RS = NT / (kUnit * 16);  // rows staged per pass (a thread keeps one block column)
  static_assert(NT % (kUnit * 16) == 0, "a thread keeps one block column");
  constexpr int NCH = kUnit * 2 * MT;    // offset chains per unit (group, 16-row tile)
  constexpr int CPW = (NCH + WVN - 1) / WVN;  // offset chains per wave

  for (int u = 0; u < U; ++u) {
    const int g0 = u * kUnit;
    const int gn = min(kUnit, G - g0);
    // the unit's activations first (staged, then the offset table), then
    // this wave's weights and scales; loads return in issue order
    const int b = tid & (kUnit * 16 - 1);
    const int r0 = tid / (kUnit * 16);
    u32x4_t v[BPT];
    {
      const uint16_t* xcol = X + static_cast<size_t>(m0) * K + min(g0 * kGroup + 8 * b, K - 8);
#pragma unroll
      for (int q = 0; q < BPT; ++q)
        v[q] = *reinterpret_cast<const u32x4_t*>(
            xcol + static_cast<size_t>(min(r0 + q * RS, mrows - 1)) * K);
    }
    u32x4_t wl[NB][kUnit], wh[NB][kUnit];
    uint32_t sc[NB][kUnit / 2];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
#pragma unroll
      for (int gg = 0; gg < kUnit; ++gg) {
        const size_t off = static_cast<size_t>(min(g0 + gg, G - 1)) * kStep;
        wl[nb][gg] = *reinterpret_cast<const u32x4_t*>(w_lo[nb] + off);
        wh[nb][gg] = *reinterpret_cast<const u32x4_t*>(w_hi[nb] + off);
      }
      if constexpr (PACKED || SVEC) {
        const u32x4_t sv = *reinterpret_cast<const u32x4_t*>(s_row[nb] + 2 * g0);
#pragma unroll
        for (int q = 0; q < 4; ++q) sc[nb][q] = sv[q];
      } else {
        const uint16_t* srow = reinterpret_cast<const uint16_t*>(s_row[nb]);
#pragma unroll
        for (int q = 0; q < 4; ++q)
          sc[nb][q] = static_cast<uint32_t>(srow[min(g0 + 2 * q, G - 1)]) |
                      (static_cast<uint32_t>(srow[min(g0 + 2 * q + 1, G - 1)]) << 16);
      }
    }
    if (u > 0) __syncthreads();  // the previous unit's readers are done
    {
      u32x4_t* xdst = xs + r0 * kPB + b;
#pragma unroll
      for (int q = 0; q < BPT; ++q) xdst[q * RS * kPB] = pair_order(v[q]);
    }
    __syncthreads();
    // offset table: chains (group, 16-row activation tile) split over the
    // waves, the decode kernels' four 16 x 16 x 32 MFMAs each; a wave's
    // chains are independent and run side by side
    {
      u32x4_t xo[CPW][4];
#pragma unroll
      for (int q = 0; q < CPW; ++q) {
        const int c = min(wave + q * WVN, NCH - 1);
        const int gg = c / (2 * MT), st = c - gg * (2 * MT);
        const u32x4_t* xg = xs + (st * 16 + i16) * kPB + gg * 16 + 4 * a16;
#pragma unroll
        for (int d = 0; d < 4; ++d) xo[q][d] = xg[d];
      }
#pragma unroll
      for (int q = 0; q < CPW; ++q) {
        const int c = wave + q * WVN;
        const f32x4_t o = group_offset_t<Act>(xo[q]);
        if (c < NCH && i16 == 0) {
          const int gg = c / (2 * MT), st = c - gg * (2 * MT);
          *reinterpret_cast<f32x4_t*>(corr + gg * TM + st * 16 + 4 * a16) = o;
        }
      }
    }
    __syncthreads();
    if (!wave_ok) continue;

    f32x16_t part[NB][MT];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) part[nb][mt] = zero16;
    // one group: offset-seeded chains, then the scale fma into part
    auto group = [&](int gg) {
      u32x4_t xa[4][2][MT];
#pragma unroll
      for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
            xa[d][e][mt] = xs[(mt * 32 + j) * kPB + gg * 16 + 4 * (2 * e + h) + d];
      f32x16_t t[NB][MT];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        // seed: D row 8(r/4) + 4h + r%4 of column j holds that row's offset
        const float* cr = corr + gg * TM + mt * 32 + 4 * h;
        f32x16_t o;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const f32x4_t o4 = *reinterpret_cast<const f32x4_t*>(cr + 8 * q);
#pragma unroll
          for (int r = 0; r < 4; ++r) o[4 * q + r] = o4[r];
        }
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) t[nb][mt] = o;
      }
#pragma unroll
      for (int d = 0; d < 4; ++d) {
#pragma unroll
        for (int e = 0; e < 2; ++e) {
#pragma unroll
          for (int nb = 0; nb < NB; ++nb) {
            const u32x4_t B = Act::template decode<PACKED>(e == 0 ? wl[nb][gg][d] : wh[nb][gg][d]);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) t[nb][mt] = mfma32<Act>(xa[d][e][mt], B, t[nb][mt]);
          }
        }
      }
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        const float s = half_bits_to_f32((sc[nb][gg >> 1] >> (16 * (gg & 1))) & 0xFFFFu);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            part[nb][mt][r] = __builtin_fmaf(s, t[nb][mt][r], part[nb][mt][r]);
      }
    };
    if (gn == kUnit) {
#pragma unroll
      for (int gg = 0; gg < kUnit; ++gg) group(gg);
    } else {
#pragma unroll
      for (int gg = 0; gg < kUnit; ++gg)
        if (gg < gn) group(gg);
    }
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) acc[nb][mt] = acc[nb][mt] + part[nb][mt];
  }
  if (!wave_ok) return;
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    const int n = nbase + 32 * nb + j;
    if (n >= N) continue;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int m = mt * 32 + 8 * (r >> 2) + 4 * h + (r & 3);
        if (m < mrows) {
          // a NaN sum (infinite or NaN activations, overflow) is recomputed
          // by the reference loop, which keeps the reference's semantics
          float v = Act::kUnit * acc[nb][mt][r];
          if (__builtin_expect(v != v, 0))
            v = w4a16_ref_dot<PACKED, std::is_same<Act, ActF16>::value>(W, S, K, n, X + static_cast<size_t>(m0 + m) * K);
          Y[static_cast<size_t>(m0 + m) * N + n] = static_cast<uint16_t>(Act::round(v));
        }
      }
  }
}

// K = 1024 (one 8-group unit): the unit's groups split over two wave sets.
// A workgroup of 2 x WVN waves owns 32 WVN weight rows and 32 activation
// rows; wave (ks, wn) loads and decodes the weights of groups 4 ks .. 4 ks + 3
// of rows 32 wn .. 32 wn + 31 and runs their offset-seeded chains. Set 0
// folds its four chain results into part = fma(s, tmp, part) in group order
// and hands part to set 1 through LDS; set 1 holds its four results in
// registers and continues the same fma chain with groups 4..7, then stores.
// The arithmetic is that of w4a16_gemm32_kernel, step for step; each wave
// has half the weight loads and half the chains on its critical path.
constexpr int kSplitHalf = kUnit / 2;  // groups per wave set

// File layout: each wave loads its rows' 256-byte run of the set's four
// groups in whole lines (load q: rows 4q .. 4q + 3, lane l: bytes 16 (l % 16)
// of row 4q + l / 16) and re-lays them out for the MFMA lanes through a
// per-wave LDS staging area, half the run at a time (rows of 144 bytes).
// With 2-wave sets the staging would leave room for one workgroup per CU
// instead of two, so those keep 32-byte loads straight into the lanes.
constexpr int kSplitStagePitch = 144;

template <int WVN, bool PACKED>
constexpr bool split_staged() {
  return !PACKED && WVN >= 4;
}

// 4-wave sets without staging hand part over through the activation buffer
// (after a barrier every reader of it has passed): 67 KB of LDS, two
// workgroups per CU.
template <int WVN, bool PACKED>
constexpr bool split_alias() {
  return WVN == 4 && !split_staged<WVN, PACKED>();
}

template <int WVN, bool PACKED>
constexpr size_t gemm32_split_lds_bytes() {
  // the part hand-over (WVN x 4 KB) reuses the file layout's staging area
  return gemm32_lds_bytes<WVN, 1>() +
         (split_staged<WVN, PACKED>() ? static_cast<size_t>(2 * WVN) * 32 * kSplitStagePitch
          : split_alias<WVN, PACKED>() ? static_cast<size_t>(0)
                                       : static_cast<size_t>(WVN) * 64 * 16 * 4);
}

template <class Act, int WVN, bool PACKED, bool SVEC>
__global__ __launch_bounds__(WVN * 2 * 64) void w4a16_gemm32_split_kernel(
    const uint8_t* __restrict__ W, const uint16_t* __restrict__ S,
    const uint16_t* __restrict__ X, uint16_t* __restrict__ Y, int N, int M) {
  constexpr int K = kUnit * kGroup;
  constexpr int G = kUnit;
  constexpr int NW = 2 * WVN;  // waves per workgroup
  constexpr int NT = NW * 64;
  constexpr int TM = 32;
  constexpr bool STAGED = split_staged<WVN, PACKED>();
  extern __shared__ u32x4_t lds[];  // x [TM][kPB], offset table [8][TM] f32, part exchange
  u32x4_t* xs = lds;
  float* corr = reinterpret_cast<float*>(lds + TM * kPB);
  uint8_t* stage = reinterpret_cast<uint8_t*>(corr + kUnit * TM);
  constexpr bool ALIAS = split_alias<WVN, PACKED>();
  f32x4_t* xchg = reinterpret_cast<f32x4_t*>(ALIAS ? reinterpret_cast<uint8_t*>(lds) : stage);

  const int lane = threadIdx.x & 63;
  const int wave = wave_id();
  const int ks = wave / WVN, wn = wave - ks * WVN;
  const int tid = static_cast<int>(threadIdx.x);
  const int j = lane & 31, h = lane >> 5;
  const int i16 = lane & 15, a16 = lane >> 4;
  const int m0 = blockIdx.y * TM;
  const int mrows = min(TM, M - m0);
  const int n = (blockIdx.x * WVN + wn) * 32 + j;
  const bool wave_ok = (blockIdx.x * WVN + wn) * 32 < N;
  const int gb = ks * kSplitHalf;  // this wave set's first group

  // activations first (loads return in issue order), then the weights and
  // scales of this wave set's groups
  constexpr int NBLK = TM * kUnit * 16;
  static_assert(NBLK % NT == 0 && NT % (kUnit * 16) == 0, "staging covers the tile exactly");
  constexpr int BPT = NBLK / NT;
  constexpr int RS = NT / (kUnit * 16);
  const int b = tid & (kUnit * 16 - 1);
  const int r0 = tid / (kUnit * 16);
  u32x4_t v[BPT];
  {
    const uint16_t* xcol = X + static_cast<size_t>(m0) * K + 8 * b;
#pragma unroll
    for (int q = 0; q < BPT; ++q)
      v[q] = *reinterpret_cast<const u32x4_t*>(xcol +
                                               static_cast<size_t>(min(r0 + q * RS, mrows - 1)) * K);
  }
  u32x4_t wl[kSplitHalf], wh[kSplitHalf];
  u32x4_t raw[8];  // file layout: the whole-line loads, before the re-layout
  uint32_t sc[kSplitHalf / 2];
  {
    const int row = min(n, N - 1);
    const uint8_t* s_row;
    if constexpr (PACKED) {
      const uint8_t* tile = W + static_cast<size_t>(row >> 4) * packed_tile_bytes(G);
      const uint8_t* w_lo = tile + 16 * (16 * h + (row & 15));
      s_row = tile + static_cast<size_t>(G) * 1024 + (row & 15) * packed_scale_pitch(G);
#pragma unroll
      for (int gg = 0; gg < kSplitHalf; ++gg) {
        wl[gg] = *reinterpret_cast<const u32x4_t*>(w_lo + (gb + gg) * 1024);
        wh[gg] = *reinterpret_cast<const u32x4_t*>(w_lo + 16 * 32 + (gb + gg) * 1024);
      }
    } else if constexpr (!STAGED) {
      const uint8_t* w_lo = W + static_cast<size_t>(row) * (K >> 1) + 16 * h;
      s_row = reinterpret_cast<const uint8_t*>(S + static_cast<size_t>(row) * G);
#pragma unroll
      for (int gg = 0; gg < kSplitHalf; ++gg) {
        wl[gg] = *reinterpret_cast<const u32x4_t*>(w_lo + (gb + gg) * 64);
        wh[gg] = *reinterpret_cast<const u32x4_t*>(w_lo + 32 + (gb + gg) * 64);
      }
    } else {
      s_row = reinterpret_cast<const uint8_t*>(S + static_cast<size_t>(row) * G);
      const int rbase = (blockIdx.x * WVN + wn) * 32 + (lane >> 4);
      const uint8_t* wcol = W + gb * 64 + 16 * (lane & 15);
#pragma unroll
      for (int q = 0; q < 8; ++q)
        raw[q] = *reinterpret_cast<const u32x4_t*>(
            wcol + static_cast<size_t>(min(rbase + 4 * q, N - 1)) * (K >> 1));
    }
    if constexpr (PACKED || SVEC) {
      const uint2 sv = *reinterpret_cast<const uint2*>(s_row + 2 * gb);
      sc[0] = sv.x;
      sc[1] = sv.y;
    } else {
      const uint16_t* srow = reinterpret_cast<const uint16_t*>(s_row);
#pragma unroll
      for (int q = 0; q < kSplitHalf / 2; ++q)
        sc[q] = static_cast<uint32_t>(srow[gb + 2 * q]) |
                (static_cast<uint32_t>(srow[gb + 2 * q + 1]) << 16);
    }
  }
  {
    u32x4_t* xdst = xs + r0 * kPB + b;
#pragma unroll
    for (int q = 0; q < BPT; ++q) xdst[q * RS * kPB] = pair_order(v[q]);
  }
  __syncthreads();
  // offset table: 16 chains (group, 16-row tile) split over the waves
  {
    constexpr int NCH = kUnit * 2;
    constexpr int CPW = (NCH + NW - 1) / NW;
    u32x4_t xo[CPW][4];
#pragma unroll
    for (int q = 0; q < CPW; ++q) {
      const int c = min(wave + q * NW, NCH - 1);
      const u32x4_t* xg = xs + ((c & 1) * 16 + i16) * kPB + (c >> 1) * 16 + 4 * a16;
#pragma unroll
      for (int d = 0; d < 4; ++d) xo[q][d] = xg[d];
    }
#pragma unroll
    for (int q = 0; q < CPW; ++q) {
      const int c = wave + q * NW;
      const f32x4_t o = group_offset_t<Act>(xo[q]);
      if (c < NCH && i16 == 0)
        *reinterpret_cast<f32x4_t*>(corr + (c >> 1) * TM + (c & 1) * 16 + 4 * a16) = o;
    }
  }
  __syncthreads();

  if constexpr (STAGED) {
    // re-lay the wave's rows out for the MFMA lanes: lane (j, h) takes
    // 16-byte chunks 4 gq + h (groups' k 32h .. 32h + 31) and 4 gq + 2 + h
    // of row j
    uint8_t* st = stage + wave * 32 * kSplitStagePitch;
#pragma unroll
    for (int hh = 0; hh < 2; ++hh) {
      if (((lane >> 3) & 1) == hh) {
#pragma unroll
        for (int q = 0; q < 8; ++q)
          *reinterpret_cast<u32x4_t*>(st + (4 * q + (lane >> 4)) * kSplitStagePitch +
                                      (lane & 7) * 16) = raw[q];
      }
      wave_lds_sync();
#pragma unroll
      for (int g2 = 0; g2 < 2; ++g2) {
        wl[2 * hh + g2] =
            *reinterpret_cast<const u32x4_t*>(st + j * kSplitStagePitch + (4 * g2 + h) * 16);
        wh[2 * hh + g2] =
            *reinterpret_cast<const u32x4_t*>(st + j * kSplitStagePitch + (4 * g2 + 2 + h) * 16);
      }
      wave_lds_sync();
    }
  }

  // chain results of this wave set's groups
  f32x16_t t[kSplitHalf];
  if (wave_ok) {
#pragma unroll
    for (int gq = 0; gq < kSplitHalf; ++gq) {
      const int gg = gb + gq;
      u32x4_t xa[4][2];
#pragma unroll
      for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int e = 0; e < 2; ++e) xa[d][e] = xs[j * kPB + gg * 16 + 4 * (2 * e + h) + d];
      const float* cr = corr + gg * TM + 4 * h;
      f32x16_t acc;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x4_t o4 = *reinterpret_cast<const f32x4_t*>(cr + 8 * q);
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[4 * q + r] = o4[r];
      }
#pragma unroll
      for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int e = 0; e < 2; ++e)
          acc = mfma32<Act>(xa[d][e], Act::template decode<PACKED>(e == 0 ? wl[gq][d] : wh[gq][d]), acc);
      t[gq] = acc;
    }
  }
  const auto scale = [&](int gq) {
    return half_bits_to_f32((sc[gq >> 1] >> (16 * (gq & 1))) & 0xFFFFu);
  };
  f32x4_t* slot = xchg + wn * 4 * 64 + lane;
  f32x16_t part = {};
  if (ks == 0 && wave_ok) {
#pragma unroll
    for (int gq = 0; gq < kSplitHalf; ++gq) {
      const float s = scale(gq);
#pragma unroll
      for (int r = 0; r < 16; ++r) part[r] = __builtin_fmaf(s, t[gq][r], part[r]);
    }
  }
  // every wave is done with its staging rows / the activations
  if constexpr (STAGED || ALIAS) __syncthreads();
  if (ks == 0 && wave_ok) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
      slot[q * 64] = f32x4_t{part[4 * q], part[4 * q + 1], part[4 * q + 2], part[4 * q + 3]};
  }
  __syncthreads();
  if (ks == 0 || !wave_ok || n >= N) return;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const f32x4_t p4 = slot[q * 64];
#pragma unroll
    for (int r = 0; r < 4; ++r) part[4 * q + r] = p4[r];
  }
#pragma unroll
  for (int gq = 0; gq < kSplitHalf; ++gq) {
    const float s = scale(gq);
#pragma unroll
    for (int r = 0; r < 16; ++r) part[r] = __builtin_fmaf(s, t[gq][r], part[r]);
  }
  // one unit: total = 0 + part
  const f32x16_t zero16 = {};
  const f32x16_t total = zero16 + part;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int m = 8 * (r >> 2) + 4 * h + (r & 3);
    if (m < mrows) {
      float val = Act::kUnit * total[r];
      if (__builtin_expect(val != val, 0))
        val = w4a16_ref_dot<PACKED, std::is_same<Act, ActF16>::value>(W, S, K, n, X + static_cast<size_t>(m0 + m) * K);
      Y[static_cast<size_t>(m0 + m) * N + n] = static_cast<uint16_t>(Act::round(val));
    }
  }
}

template <class Act, int WVN, bool PACKED>
int launch_gemm32_split(const uint8_t* W, const uint16_t* S, const uint16_t* X, uint16_t* Y, int N,
                        int M, hipStream_t stream) {
  const size_t lds = gemm32_split_lds_bytes<WVN, PACKED>();
  const int gx = (N + 32 * WVN - 1) / (32 * WVN);
  const int gy = (M + 31) / 32;
  if (gy > 65535) return CUDALM_W4A16_ERANGE;
  const bool svec = !PACKED && aligned(S, 8);
  auto kern = svec ? w4a16_gemm32_split_kernel<Act, WVN, PACKED, true>
                   : w4a16_gemm32_split_kernel<Act, WVN, PACKED, false>;
  if (!allow_lds(kern, lds)) return CUDALM_W4A16_ELAUNCH;
  hipLaunchKernelGGL(kern, dim3(gx, gy), dim3(WVN * 2 * 64), lds, stream, W, S, X, Y, N, M);
  return launch_status();
}

template <class Act, int WVN, int MT, int NB, bool PACKED>
int launch_gemm32(const uint8_t* W, const uint16_t* S, const uint16_t* X, uint16_t* Y, int N,
                  int K, int M, hipStream_t stream) {
  const size_t lds = gemm32_lds_bytes<WVN, MT>();
  const int gx = (N + 32 * WVN * NB - 1) / (32 * WVN * NB);
  const int gy = (M + 32 * MT - 1) / (32 * MT);
  if (gy > 65535) return CUDALM_W4A16_ERANGE;
  const bool svec = !PACKED && (K / kGroup) % 8 == 0 && aligned(S, 16);
  auto kern = svec ? w4a16_gemm32_kernel<Act, WVN, MT, NB, PACKED, true>
                   : w4a16_gemm32_kernel<Act, WVN, MT, NB, PACKED, false>;
  if (!allow_lds(kern, lds)) return CUDALM_W4A16_ELAUNCH;
  hipLaunchKernelGGL(kern, dim3(gx, gy), dim3(WVN * 64), lds, stream, W, S, X, Y, N, K, M);
  return launch_status();
}

// ---------------------------------------------------------------------------
// Unit GEMM kernel (prefill chunks): a k-slice of WV waves owns
// TN = WV * RB * 16 weight rows and TM = CT * 16 activation rows. K is walked
// one 8-group unit (1024 k) at a time: the unit's activations are staged
// once into LDS (pair order), the slice computes the unit's offset table
// once (waves split the chains), and every weight is decoded once, by the
// wave that owns its rows, and feeds CT MFMA column tiles. Weights of a unit
// are fetched up front (while the activations are staged). The per-output
// operation sequence is the stream kernel's, so the bits are the same.
//
// KS > 1 k-slices split the units of the same output tile: slice s takes
// units s, s + KS, ... with its own LDS buffers, keeps each unit partial,
// and at the end the partials meet in LDS and are summed in unit order, so
// the bits do not depend on KS. This serves few-tile, long-K shapes
// (N = 1024, K = 2048 / 3584), where one slice would walk every unit alone.
// ---------------------------------------------------------------------------

constexpr int kSliceMaxUnits = 4;  // units per k-slice kept as partials (KS > 1)

// GLU: RB = 2, the wave's tiles are the same rows of gate (W, S) and up (W2,
// S2), and y = silu(gate) * up is stored.
template <class Act, int RB, int CT, int WV, bool PACKED, bool SVEC, int KS = 1, bool IOFF = false,
          bool GLU = false>
__device__ __forceinline__ void gemm_unit_tile(const uint8_t* __restrict__ W,
                                               const uint16_t* __restrict__ S,
                                               const uint16_t* __restrict__ X,
                                               uint16_t* __restrict__ Y, int N, int K, int M,
                                               int bx, const uint8_t* __restrict__ W2 = nullptr,
                                               const uint16_t* __restrict__ S2 = nullptr) {
  static_assert(!GLU || RB == 2, "a gate and an up tile");
  constexpr int TR = GLU ? 1 : RB;  // output tiles per wave
  constexpr int NT = WV * 64;  // threads of one k-slice
  constexpr int TM = CT * 16;
  constexpr int PB = x_pitch(kUnit * kGroup);  // LDS row pitch in 16-byte blocks (padded)
  constexpr int NBLK = TM * kUnit * 16;  // 16-byte x blocks per unit
  static_assert(NBLK % NT == 0, "staging must cover the tile exactly");
  constexpr int BPT = NBLK / NT;  // x blocks staged per thread per unit
  constexpr int XB = TM * PB;     // 16-byte blocks of one slice's x buffer
  constexpr int NPART = KS == 1 ? 1 : kSliceMaxUnits;
  extern __shared__ u32x4_t lds[];  // [KS][TM][PB] x, then [KS] offset tables

  const int G = K >> 7;
  const int U = (G + kUnit - 1) / kUnit;
  const int ntiles = (N + kTileRows - 1) / kTileRows;
  const int lane = threadIdx.x & 63;
  const int slice = KS == 1 ? 0 : wave_id() / WV;
  const int wave = wave_id() - slice * WV;  // wave within the slice
  const int tid = static_cast<int>(threadIdx.x) - slice * NT;
  const int i = lane & 15, a = lane >> 4;
  const int m0 = blockIdx.y * TM;
  const int mrows = min(TM, M - m0);
  u32x4_t* xs = lds + slice * XB;
  float* corr = reinterpret_cast<float*>(lds + KS * XB) + slice * (kUnit * CT * 16);

  int rt[RB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) rt[rb] = min((bx * WV + wave) * TR + (GLU ? 0 : rb), ntiles - 1);
  const bool any_ok = (bx * WV + wave) * TR < ntiles;

  // lane addresses of each owned tile at group 0
  const uint8_t* wbase[RB];
  const uint8_t* sbase[RB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    if constexpr (PACKED) {
      const uint8_t* tile = (GLU && rb == 1 ? W2 : W) + static_cast<size_t>(rt[rb]) * packed_tile_bytes(G);
      wbase[rb] = tile + lane * 16;
      sbase[rb] = tile + static_cast<size_t>(G) * 1024 + i * packed_scale_pitch(G);
    } else {
      const int row = min(rt[rb] * kTileRows + i, N - 1);
      wbase[rb] = (GLU && rb == 1 ? W2 : W) + static_cast<size_t>(row) * (K >> 1) + a * 16;
      sbase[rb] = reinterpret_cast<const uint8_t*>((GLU && rb == 1 ? S2 : S) + static_cast<size_t>(row) * G);
    }
  }
  constexpr int kStep = PACKED ? 1024 : 64;  // bytes between groups of one lane

  const f32x4_t zero = {0.0f, 0.0f, 0.0f, 0.0f};
  // KS == 1: the running unit sum; KS > 1: this slice's unit partials
  f32x4_t acc[NPART][RB][CT];
#pragma unroll
  for (int q = 0; q < NPART; ++q)
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) acc[q][rb][ct] = zero;

  const int iters = (U + KS - 1) / KS;
  for (int it = 0; it < iters; ++it) {
    const int u = it * KS + slice;
    const int uc = min(u, U - 1);  // a slice past the last unit re-reads it and skips the math
    const int g0 = uc * kUnit;
    const int gn = u < U ? min(kUnit, G - g0) : 0;
    // the unit's activations first: they are staged and feed the offset
    // table before any weight is used, and loads return in issue order
    constexpr int RS = NT / (kUnit * 16);
    static_assert(NT % (kUnit * 16) == 0, "a thread keeps one block column");
    const int b = tid & (kUnit * 16 - 1);  // thread tid stages block b of rows tid / 128 + q * RS
    const int r0 = tid / (kUnit * 16);
    u32x4_t v[BPT];
    {
      const uint16_t* xcol = X + static_cast<size_t>(m0) * K + min(g0 * kGroup + 8 * b, K - 8);
#pragma unroll
      for (int q = 0; q < BPT; ++q)
        v[q] = *reinterpret_cast<const u32x4_t*>(
            xcol + static_cast<size_t>(min(r0 + q * RS, mrows - 1)) * K);
    }
    // then this unit's weights and scales (group indices clamped to G - 1)
    u32x4_t w[RB][kUnit];
    uint32_t sc[RB][kUnit / 2];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
#pragma unroll
      for (int gg = 0; gg < kUnit; ++gg)
        w[rb][gg] = *reinterpret_cast<const u32x4_t*>(
            wbase[rb] + static_cast<size_t>(min(g0 + gg, G - 1)) * kStep);
      if constexpr (PACKED || SVEC) {
        const u32x4_t sv = *reinterpret_cast<const u32x4_t*>(sbase[rb] + 2 * g0);
#pragma unroll
        for (int q = 0; q < 4; ++q) sc[rb][q] = sv[q];
      } else {
        const uint16_t* srow = reinterpret_cast<const uint16_t*>(sbase[rb]);
#pragma unroll
        for (int q = 0; q < 4; ++q)
          sc[rb][q] = static_cast<uint32_t>(srow[min(g0 + 2 * q, G - 1)]) |
                      (static_cast<uint32_t>(srow[min(g0 + 2 * q + 1, G - 1)]) << 16);
      }
    }
    if (it > 0) __syncthreads();  // previous unit's readers are done
    {
      u32x4_t* xdst = xs + r0 * PB + x_slot(b);
#pragma unroll
      for (int q = 0; q < BPT; ++q) xdst[q * RS * PB] = pair_order(v[q]);
    }
    __syncthreads();
    // offset table of the unit: chains (group, column tile) split over waves
    // (IOFF: each wave runs the chains of its own groups inline instead, the
    // same operands, and the table and its barrier are skipped)
    if constexpr (!IOFF) {
      for (int c = wave; c < kUnit * CT; c += WV) {
        const int gg = c / CT, ct = c - gg * CT;
        u32x4_t xa[4];
        load_group_x(xa, xs + (ct * 16 + i) * PB + gg * 16, a);
        const f32x4_t o = group_offset_t<Act>(xa);
        if (i == 0) *reinterpret_cast<f32x4_t*>(corr + c * 16 + 4 * a) = o;
      }
      __syncthreads();
    }
    if (!any_ok) continue;

    f32x4_t part[RB][CT];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) part[rb][ct] = zero;
    // one group: offset-seeded weight chains, then the scale fma into part
    auto group = [&](int gg) {
      u32x4_t xa[CT][4];
      f32x4_t t[RB][CT];
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) {
        load_group_x(xa[ct], xs + (ct * 16 + i) * PB + gg * 16, a);
        const f32x4_t o = IOFF ? group_offset_t<Act>(xa[ct])
                               : *reinterpret_cast<const f32x4_t*>(corr + (gg * CT + ct) * 16 + 4 * a);
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) t[rb][ct] = o;
      }
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          const u32x4_t B = Act::template decode<PACKED>(w[rb][gg][d]);
#pragma unroll
          for (int ct = 0; ct < CT; ++ct) t[rb][ct] = Act::mma(xa[ct][d], B, t[rb][ct]);
        }
      }
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        const float s = half_bits_to_f32((sc[rb][gg >> 1] >> (16 * (gg & 1))) & 0xFFFFu);
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            part[rb][ct][r] = __builtin_fmaf(s, t[rb][ct][r], part[rb][ct][r]);
      }
    };
    if (gn == kUnit) {
      // full unit: straight-line, so independent group chains interleave
#pragma unroll
      for (int gg = 0; gg < kUnit; ++gg) group(gg);
    } else {
#pragma unroll
      for (int gg = 0; gg < kUnit; ++gg)
        if (gg < gn) group(gg);
    }
    if constexpr (KS == 1) {
#pragma unroll
      for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) acc[0][rb][ct] = acc[0][rb][ct] + part[rb][ct];
    } else {
#pragma unroll
      for (int q = 0; q < NPART; ++q)
        if (q == it)
#pragma unroll
          for (int rb = 0; rb < RB; ++rb)
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) acc[q][rb][ct] = part[rb][ct];
    }
  }

  f32x4_t total[RB][CT];
  if constexpr (KS == 1) {
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) total[rb][ct] = acc[0][rb][ct];
  } else {
    // unit partials meet in LDS (over the x buffers): slot [u][wave][rb][ct][lane]
    __syncthreads();
    f32x4_t* slots = reinterpret_cast<f32x4_t*>(lds);
    if (any_ok) {
#pragma unroll
      for (int q = 0; q < NPART; ++q) {
        const int u = q * KS + slice;
        if (q < iters && u < U)
#pragma unroll
          for (int rb = 0; rb < RB; ++rb)
#pragma unroll
            for (int ct = 0; ct < CT; ++ct)
              slots[(((u * WV + wave) * RB + rb) * CT + ct) * 64 + lane] = acc[q][rb][ct];
      }
    }
    __syncthreads();
    if (slice != 0) return;
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) {
        total[rb][ct] = zero;
        for (int u = 0; u < U; ++u)
          total[rb][ct] = total[rb][ct] + slots[(((u * WV + wave) * RB + rb) * CT + ct) * 64 + lane];
      }
  }
  if (!any_ok) return;
  if constexpr (GLU) {
    const int n = rt[0] * kTileRows + i;
    if (n >= N) return;
    uint16_t* col = Y + static_cast<size_t>(m0 + 4 * a) * N + n;
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (ct * 16 + 4 * a + r < mrows) {
          const uint16_t* xrow = X + static_cast<size_t>(m0 + ct * 16 + 4 * a + r) * K;
          const uint32_t gt = Act::round(out_value<Act, PACKED>(total[0][ct][r], W, S, K, n, xrow));
          const uint32_t up = Act::round(out_value<Act, PACKED>(total[1][ct][r], W2, S2, K, n, xrow));
          col[static_cast<size_t>(ct * 16 + r) * N] = static_cast<uint16_t>(silu_mul_bits(gt, up));
        }
    return;
  }
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    const int n = ((bx * WV + wave) * RB + rb) * kTileRows + i;
    if (n >= N) continue;
    uint16_t* col = Y + static_cast<size_t>(m0 + 4 * a) * N + n;
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (ct * 16 + 4 * a + r < mrows)
          col[static_cast<size_t>(ct * 16 + r) * N] = static_cast<uint16_t>(Act::round(
              out_value<Act, PACKED>(total[rb][ct][r], W, S, K, n,
                                         X + static_cast<size_t>(m0 + ct * 16 + 4 * a + r) * K)));
  }
}

template <class Act, int RB, int CT, int WV, bool PACKED, bool SVEC, int KS = 1, bool IOFF = false>
__global__ __launch_bounds__(WV * KS * 64) void w4a16_gemm_unit_kernel(
    const uint8_t* __restrict__ W, const uint16_t* __restrict__ S,
    const uint16_t* __restrict__ X, uint16_t* __restrict__ Y, int N, int K, int M) {
  gemm_unit_tile<Act, RB, CT, WV, PACKED, SVEC, KS, IOFF>(W, S, X, Y, N, K, M, blockIdx.x);
}

template <int WV, bool PACKED, bool SVEC, int KS, bool IOFF>
__global__ __launch_bounds__(WV * KS * 64) void w4a16_gemm_unit_swiglu_kernel(
    const uint8_t* __restrict__ Wg, const uint8_t* __restrict__ Wu, const uint16_t* __restrict__ X,
    int N, int K, int M, const uint16_t* __restrict__ Sg, const uint16_t* __restrict__ Su,
    uint16_t* __restrict__ Y) {
  gemm_unit_tile<ActBf16, 2, 2, WV, PACKED, SVEC, KS, IOFF, true>(Wg, Sg, X, Y, N, K, M, blockIdx.x,
                                                                 Wu, Su);
}

// Projections sharing x: blockIdx.x numbers the row tiles of all of them in
// turn (P.end).
template <int WV, bool PACKED, bool SVEC, int KS, bool IOFF>
__global__ __launch_bounds__(WV * KS * 64) void w4a16_gemm_unit_group_kernel(PrefillGroup P, int K,
                                                                             int M) {
  int bx = blockIdx.x;
  const PrefillProj v = prefill_proj(P, bx);
  gemm_unit_tile<ActBf16, 1, 2, WV, PACKED, SVEC, KS, IOFF>(v.w, v.s, P.x, v.y, v.n, K, M, bx);
}

template <class Act, int RB, int CT, int WV, bool PACKED, int KS = 1, bool IOFF = false>
int launch_gemm_unit(const uint8_t* W, const uint16_t* S, const uint16_t* X, uint16_t* Y, int N,
                     int K, int M, hipStream_t stream) {
  constexpr int TM = CT * 16;
  const size_t xbytes = static_cast<size_t>(TM) * x_pitch(kUnit * kGroup) * 16;
  const size_t lds = KS * (xbytes + static_cast<size_t>(kUnit) * CT * 16 * sizeof(float));
  const int G = K / kGroup;
  if constexpr (KS > 1) {
    // every slice keeps at most kSliceMaxUnits partials, and all of them
    // must fit the x buffers they are parked in
    const int U = (G + kUnit - 1) / kUnit;
    if (U > KS * kSliceMaxUnits ||
        static_cast<size_t>(U) * WV * RB * CT * 64 * 16 > KS * xbytes)
      return launch_gemm_unit<Act, RB, CT, WV, PACKED, 1, IOFF>(W, S, X, Y, N, K, M, stream);
  }
  const int ntiles = (N + kTileRows - 1) / kTileRows;
  const int gx = (ntiles + WV * RB - 1) / (WV * RB);
  const int gy = (M + TM - 1) / TM;
  if (gy > 65535) return CUDALM_W4A16_ERANGE;
  const bool svec = !PACKED && G % 8 == 0 && aligned(S, 16);
  auto kern = svec ? w4a16_gemm_unit_kernel<Act, RB, CT, WV, PACKED, true, KS, IOFF>
                   : w4a16_gemm_unit_kernel<Act, RB, CT, WV, PACKED, false, KS, IOFF>;
  if (!allow_lds(kern, lds)) return CUDALM_W4A16_ELAUNCH;
  hipLaunchKernelGGL(kern, dim3(gx, gy), dim3(WV * KS * 64), lds, stream, W, S, X, Y, N, K, M);
  return launch_status();
}

// Waves per wave set of the K = 1024 split kernel: the narrowest of 2, 4
// and 8 (64, 128 or 256 weight rows per workgroup) whose workgroups fill
// between half and one round of the CUs. M = 512: 512 x 1024 takes 2
// (5.20-5.25 against 5.51-5.56 us for the 64 x 32 unit GEMM), 2048 x 1024
// takes 4 (6.57 against 6.68-6.75 us for the 128 x 32 one), 3584 and 4096
// x 1024 take 8. When none fits, prepacked weights take 4-wave sets (two
// workgroups per CU) from one to 1.5 rounds of those: 6144 x 1024 13.48-13.61
// against 14.37-14.63 us for the unit GEMM; the file layout, whose 4-wave
// sets stage their loads and run one workgroup per CU, keeps the unit GEMM
// (15.9-16.0 against 19.1-19.3 us). 0: the unit GEMM.
int prefill_split_waves(int N, int M, int cus, bool packed) {
  const long long gy = (M + 31) / 32;
  for (int wv = 2; wv <= 8; wv *= 2) {
    const long long wgs = gy * ((N + 32 * wv - 1) / (32 * wv));
    if (2 * wgs >= cus && wgs <= cus) return wv;
  }
  const long long wgs4 = gy * ((N + 127) / 128);
  if (packed && wgs4 >= cus && wgs4 <= 3LL * cus) return 4;
  return 0;
}

}  // namespace

template <class Act, bool PACKED>
int launch_prefill32(const uint8_t* W, const uint16_t* S, const uint16_t* X, uint16_t* Y, int N,
                     int K, int M, hipStream_t stream) {
  if (K == kUnit * kGroup) {
    switch (prefill_split_waves(N, M, cu_count(), PACKED)) {
      case 2: return launch_gemm32_split<Act, 2, PACKED>(W, S, X, Y, N, M, stream);
      case 4: return launch_gemm32_split<Act, 4, PACKED>(W, S, X, Y, N, M, stream);
      default: return launch_gemm32_split<Act, 8, PACKED>(W, S, X, Y, N, M, stream);
    }
  }
  return launch_gemm32<Act, 8, 1, 1, PACKED>(W, S, X, Y, N, K, M, stream);
}

// Prefill chunks (M >= 33, and 17 to 32 rows of long K). Shapes with enough 64 x
// 256 output tiles that pad little take the wide kernel (wide_serves), few tiles of
// long K its k-slices (wide_slices_serve). The 32 x 32 MFMA GEMM (32 activation rows x
// 256 weight rows per 8-wave workgroup) serves K <= 1024
// when its workgroups fill between 3/4 and all of the CUs in one round
// (3584x1024 and 4096x1024 at M = 512: 10.3 -> 9.6-9.9 us, 10.7 -> 9.5-10.0 us);
// elsewhere the 16 x 16 unit GEMM is faster (one round of 32 x 256 tiles
// leaves too many CUs idle below that, and past one round it takes two).
// Unit GEMM tiles: 128 x 32 of 8 waves while they fill most of the CUs,
// else 64 x 32 of 4 waves, with two k-slices of 4 waves when K spans
// several units (1024x3584 at M = 512: 16.7 -> 14.6 us). The 4-wave tiles
// run their offset chains inline (512x1024x512 5.8 -> 5.5 us, 1024x3584x512
// 14.4 -> 13.8 us); inline chains cost the 8-wave tiles 0.6 us at
// 3584x1024x512, so those keep the table.
template <class Act, bool PACKED>
int launch_prefill(const uint8_t* W, const uint16_t* S, const uint16_t* X, uint16_t* Y, int N, int K,
                   int M, hipStream_t stream) {
  const int cus = cu_count();
  if (wide_serves<PACKED>(N, K, M)) return launch_wide<Act, PACKED>(W, S, X, Y, N, K, M, stream);
  if (wide_slices_serve<PACKED>(S, N, K, M))
    return launch_wide_slices<Act, PACKED>(W, S, X, Y, N, K, M, stream);
  if (K == kUnit * kGroup && prefill_split_waves(N, M, cus, PACKED) != 0)
    return launch_prefill32<Act, PACKED>(W, S, X, Y, N, K, M, stream);
  if (K < kUnit * kGroup) {
    const long long wgs32 = static_cast<long long>((N + 255) / 256) * ((M + 31) / 32);
    if (4 * wgs32 >= 3LL * cus && wgs32 <= cus)
      return launch_prefill32<Act, PACKED>(W, S, X, Y, N, K, M, stream);
  }
  const long long wgs = static_cast<long long>((N + 127) / 128) * ((M + 31) / 32);
  // (crossover measured between 128 and 168 workgroups of 128 x 32:
  // 2048x1024x256 5.7 vs 6.9 us, 3584x1024x192 7.4 vs 6.9 us)
  if (5 * wgs >= 3LL * cus) return launch_gemm_unit<Act, 1, 2, 8, PACKED>(W, S, X, Y, N, K, M, stream);
  if (K > kUnit * kGroup)
    return launch_gemm_unit<Act, 1, 2, 4, PACKED, 2, true>(W, S, X, Y, N, K, M, stream);
  return launch_gemm_unit<Act, 1, 2, 4, PACKED, 1, true>(W, S, X, Y, N, K, M, stream);
}

namespace {

template <int WV, bool PACKED, int KS, bool IOFF>
int launch_unit_group(PrefillGroup P, int K, int M, hipStream_t stream) {
  const int U = (K / kGroup + kUnit - 1) / kUnit;
  const size_t xbytes = static_cast<size_t>(32) * x_pitch(kUnit * kGroup) * 16;
  if constexpr (KS > 1)
    if (U > KS * kSliceMaxUnits || static_cast<size_t>(U) * WV * 2 * 64 * 16 > KS * xbytes)
      return launch_unit_group<WV, PACKED, 1, IOFF>(P, K, M, stream);
  const int gy = (M + 31) / 32;
  if (gy > 65535) return CUDALM_W4A16_ERANGE;
  bool svec = !PACKED && (K / kGroup) % 8 == 0;
  int tiles = 0;
  for (int j = 0; j < P.count; ++j) {
    tiles += (P.n[j] + WV * kTileRows - 1) / (WV * kTileRows);
    P.end[j] = tiles;
    svec = svec && aligned(P.s[j], 16);
  }
  const size_t lds = KS * (xbytes + static_cast<size_t>(kUnit) * 32 * sizeof(float));
  auto kern = svec ? w4a16_gemm_unit_group_kernel<WV, PACKED, !PACKED, KS, IOFF>
                   : w4a16_gemm_unit_group_kernel<WV, PACKED, false, KS, IOFF>;
  if (!allow_lds(kern, lds)) return CUDALM_W4A16_ELAUNCH;
  hipLaunchKernelGGL(kern, dim3(tiles, gy), dim3(WV * KS * 64), lds, stream, P, K, M);
  return launch_status();
}

template <int WV, bool PACKED, int KS, bool IOFF>
int launch_unit_swiglu_t(const uint8_t* Wg, const uint16_t* Sg, const uint8_t* Wu,
                         const uint16_t* Su, const uint16_t* X, uint16_t* Y, int N, int K, int M,
                         hipStream_t stream) {
  const int U = (K / kGroup + kUnit - 1) / kUnit;
  const size_t xbytes = static_cast<size_t>(32) * x_pitch(kUnit * kGroup) * 16;
  if constexpr (KS > 1)
    if (U > KS * kSliceMaxUnits || static_cast<size_t>(U) * WV * 4 * 64 * 16 > KS * xbytes)
      return launch_unit_swiglu_t<WV, PACKED, 1, IOFF>(Wg, Sg, Wu, Su, X, Y, N, K, M, stream);
  const int gx = (N + WV * kTileRows - 1) / (WV * kTileRows), gy = (M + 31) / 32;
  if (gy > 65535) return CUDALM_W4A16_ERANGE;
  const bool svec = !PACKED && (K / kGroup) % 8 == 0 && aligned(Sg, 16) && aligned(Su, 16);
  const size_t lds = KS * (xbytes + static_cast<size_t>(kUnit) * 32 * sizeof(float));
  auto kern = svec ? w4a16_gemm_unit_swiglu_kernel<WV, PACKED, !PACKED, KS, IOFF>
                   : w4a16_gemm_unit_swiglu_kernel<WV, PACKED, false, KS, IOFF>;
  if (!allow_lds(kern, lds)) return CUDALM_W4A16_ELAUNCH;
  hipLaunchKernelGGL(kern, dim3(gx, gy), dim3(WV * KS * 64), lds, stream, Wg, Wu, X, N, K, M, Sg, Su,
                     Y);
  return launch_status();
}

}  // namespace

// Projections sharing x, M >= 33, in one launch: the wide kernel or the unit
// GEMM's tiles by the rules of launch_prefill on the tiles of all of them.
// One call per projection took a launch of 5 us or more for each, the two of
// 16 rows too. us, those calls first: qkv/z/b/a (6144, 2048, 16, 16 x 1024)
// prepacked M = 33 18.1 / 6.6, 128 19.3 / 9.8, 512 28.0 / 19.2, 1024 41.4 / 29.1;
// q/k/v (4096, 512, 512) M = 128 14.0 / 8.2, 777 23.8 / 18.4; gate/up (3584
// twice) M = 64 9.4 / 7.2, 512 15.8 / 13.0, file layout 18.1 / 14.1; K = 4096
// qkv/z/b/a M = 1024 128 / 101. No shape from M = 33 to 1024 and K = 512 to
// 4096 measured slower.
template <bool PACKED>
int launch_prefill_group(const PrefillGroup& P, int K, int M, hipStream_t stream) {
  if (wide_group_serves<PACKED>(P, K, M)) return launch_wide_group<PACKED>(P, K, M, stream);
  long long wgs = 0;
  for (int j = 0; j < P.count; ++j) wgs += (P.n[j] + 127) / 128;
  wgs *= (M + 31) / 32;
  if (5 * wgs >= 3LL * cu_count()) return launch_unit_group<8, PACKED, 1, false>(P, K, M, stream);
  if (K > kUnit * kGroup) return launch_unit_group<4, PACKED, 2, true>(P, K, M, stream);
  return launch_unit_group<4, PACKED, 1, true>(P, K, M, stream);
}
template int launch_prefill_group<true>(const PrefillGroup&, int, int, hipStream_t);
template int launch_prefill_group<false>(const PrefillGroup&, int, int, hipStream_t);

// SwiGLU of M > 32 rows: GEMM tiles against the chunked kernels, whose 16 x 32
// tiles take a workgroup each. Theirs / the unit GEMM's tiles, us, by their
// workgroups on 256 CUs, prepacked: K = 1024: 128 (512, M = 128) 6.3 / 6.6, 256
// (1024, M = 128) 6.7 / 6.8, 448 (3584, M = 64) 11.8 / 7.0, 896 (M = 128) 21.9 /
// 7.3; K = 512: 376 (3001, M = 64) 7.1 / 5.9, file layout 7.1 / 6.6, M = 40 6.3 /
// 6.7; K = 2048: 192 (1024, M = 96) 8.5 / 10.2, 256 (M = 128) 15.4 / 10.3; K =
// 3584: 128 (1024, M = 64) 13.2 / 15.6, 192 (M = 96) 24.7 / 15.7. (At K <= 1024 the
// line lies where hardly a shape loses, not where the gains begin: M = 64 gains
// from fewer tiles than M = 40.) A second chunk of at most 16 rows costs half, and
// of the file layout, whose scales the GEMM loads one by one below K = 1024, the
// chunks keep those while a row tile has a CU: K = 768, M = 33 to 48 6.2 to 6.7 /
// 7.2, K = 640 6.1 to 6.6 / 7.0, K = 384 and 512 1 to 10 % (K = 256 level, K = 128
// and 896 the other way by 6 and 25 %).
//
// Past K = 1024 a chunk's workgroups have a CU each, and while all of them fit
// one round the chunks are the faster: 1024 x 1152, M = 109 file layout, 256
// workgroups, 7.8 / 11.4, 306 x 2304, M = 359 15.2 / 20.3, 434 x 2816, M = 221
// prepacked 13.9 / 15.6. (How many rows a chunk has, and so how many workgroups
// there are, follows from the LDS: 25 to 32 up to K = 2304, 17 at K = 4096.) Of 1,500
// random shapes past K = 1024 three lose by 4 to 14 %, where the last chunk has
// two to four rows.
bool swiglu_gemm_serves(int N, int K, int M, int chunks, bool packed) {
  if (M <= 32) return false;
  const long long cols = (N + 15) / 16, tiles = cols * ((M + 31) / 32);
  const long long cus = cu_count();
  if (!packed && M <= 48 && cols <= cus && K > 2 * kGroup && K <= 6 * kGroup) return false;
  if (K <= kUnit * kGroup) return 2 * tiles >= 3 * cus;
  if (cols * chunks <= cus) return false;
  return K <= 2 * kUnit * kGroup ? tiles >= cus : 4 * tiles >= 3 * cus;
}

// The unit GEMM's 128 x 32 tiles (a gate and an up tile per wave) while they
// make one round, then the wide kernel (3584 x 1024: M = 256, 224 tiles, 9.4 us
// against 13.1; M = 384, 336 tiles, 17.0 / 13.4; M = 1000 22.3 for the wide one,
// 143.5 in chunks; K = 2048: M = 256 14.4 / 23, M = 512 27.7 / 23.0). Below 3/5
// of a round 64 x 32 tiles, with two k-slices past K = 1024, as in
// launch_prefill.
template <bool PACKED>
int launch_gemm_swiglu(const uint8_t* Wg, const uint16_t* Sg, const uint8_t* Wu,
                       const uint16_t* Su, const uint16_t* X, uint16_t* Y, int N, int K, int M,
                       hipStream_t stream) {
  const long long wgs = static_cast<long long>((N + 127) / 128) * ((M + 31) / 32);
  const long long cus = cu_count();
  if (wgs > cus && wide_swiglu_fits(N, K, M))
    return launch_wide_swiglu<PACKED>(Wg, Sg, Wu, Su, X, Y, N, K, M, stream);
  if (5 * wgs >= 3 * cus)
    return launch_unit_swiglu_t<8, PACKED, 1, false>(Wg, Sg, Wu, Su, X, Y, N, K, M, stream);
  if (K > kUnit * kGroup)
    return launch_unit_swiglu_t<4, PACKED, 2, true>(Wg, Sg, Wu, Su, X, Y, N, K, M, stream);
  return launch_unit_swiglu_t<4, PACKED, 1, true>(Wg, Sg, Wu, Su, X, Y, N, K, M, stream);
}
template int launch_gemm_swiglu<true>(const uint8_t*, const uint16_t*, const uint8_t*,
                                      const uint16_t*, const uint16_t*, uint16_t*, int, int, int,
                                      hipStream_t);
template int launch_gemm_swiglu<false>(const uint8_t*, const uint16_t*, const uint8_t*,
                                       const uint16_t*, const uint16_t*, uint16_t*, int, int, int,
                                       hipStream_t);

int prefill32_regs() { return regs_of(w4a16_gemm32_split_kernel<ActBf16, 8, true, false>); }
int prefill_unit_regs() { return regs_of(w4a16_gemm_unit_kernel<ActBf16, 1, 2, 8, true, false>); }

#define W4A16_PREFILL(ACT, PACKED)                                                             \
  template int launch_prefill32<ACT, PACKED>(const uint8_t*, const uint16_t*, const uint16_t*, \
                                             uint16_t*, int, int, int, hipStream_t);           \
  template int launch_prefill<ACT, PACKED>(const uint8_t*, const uint16_t*, const uint16_t*,   \
                                           uint16_t*, int, int, int, hipStream_t)
W4A16_PREFILL(ActBf16, true);
W4A16_PREFILL(ActBf16, false);
W4A16_PREFILL(ActF16, true);
W4A16_PREFILL(ActF16, false);
#undef W4A16_PREFILL

}  // namespace cudalm_hip
