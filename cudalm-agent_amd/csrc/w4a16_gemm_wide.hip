// W4A16 GEMM on 64 x 64 wave tiles (MI355X, gfx950): prefill chunks and
// scoring calls whose outputs fill the chip with 64 x 256 tiles, and the
// SwiGLU front half of an MLP for such chunks.
//
// Contract (reference: tests/cuda/test_int4_gemv_bf16.cpp:54-69 applied row
// by row):  y[m,n] = rne( sum_k q[n,k] * f32(s[n,k/128]) * f32(x[m,k]) ).
//
// What bounds it. One decoded weight dword (7-8 VALU) feeds MT = 2 MFMAs of
// 32 x 32 x 16, and one 16-byte activation read feeds NT = 2; per group a
// wave issues 32 MFMAs (1056 cycles at the measured 33 cycles each) beside
// ~220 VALU, 28 LDS reads and 4 LDS writes. With two workgroups of 4 waves
// per CU (<= 256 registers) a pair of groups takes ~4850 cycles for both, 87%
// of the matrix cores' issue rate; one workgroup alone takes ~4280, so the
// kernel needs both. The rest of a workgroup's ~26,000 cycles at K = 1024 is
// the first loads (~2,900) and the stores (~3,500), which overlap the other
// workgroup's groups. Under this load the part lowers its clock to ~1.65 GHz
// (the same launch on all-zero data runs 1.24x faster), as it does for a
// large library GEMM (1.42 PFLOP/s measured for 8192^3 bf16).
//
// Measured against the 128 x 32 unit GEMM and the split 32 x 32 kernel, which
// serve the smaller shapes (same box, prepacked / file layout, us):
//   6144 x 1024, M = 2048:  42.3 -> 29.8 / 46.8 -> 32.3
//   4096 x 1024, M = 1024:  16.0 -> 13.4 / 17.4 -> 14.3
//   248320 x 1024, M = 256:  292 -> 147 / 279 -> 175
//   4096 x 4096, M = 1024:  55.5 -> 45.6 (64 x 32 wave tiles)
//   SwiGLU 3584 x 1024, M = 1000: 143.5 (32-row chunks) -> 22.3 / 143 -> 23.0
// Wave tiles of 128 x 64 and 64 x 128 outputs with one wave per SIMD (400-470
// registers) measured 1.4-1.5x slower: nothing covers a wave's own latencies.
// 128 x 32 tiles of 8 waves: 1.2x slower (one activation read per MFMA).
//
// Same bits as every other kernel of the library: per group the offset chain
// (four 16 x 16 x 32 MFMAs of x against -1.5) seeds the weight chain, run as
// 32 x 32 x 16 half steps in the order of w4a16_gemm.hip, then
// part = fma(s[n, g], tmp, part) in group order from 0 within an 8-group unit
// and total = 0 + part_u in unit order.
//
// Work decomposition. A workgroup of WV waves owns 32 MT activation rows and
// WV x 32 NT weight rows, each wave its own weight rows. x of a group is
// staged into one of four LDS buffers two groups ahead (loads to registers
// three ahead), with one barrier per two groups; the wave that stages 16 rows
// also runs their offset chains. Weights and scales are loaded one group
// ahead into registers. The operands of a 16-k step are read and decoded
// during the step before, pinned there by scheduling barriers: left alone
// the compiler reads them just in time. With KS k-slices a workgroup has KS
// such wave sets, each on one 8-group unit of the same outputs with buffers
// of its own; the unit partials meet in LDS and are summed in unit order.

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include <type_traits>

#include "cudalm_w4a16.h"
#include "hip_common.h"
#include "w4a16_device.h"

namespace cudalm_hip {
namespace {

// A buffer resource over everything from a uniform base on: loads take a
// 32-bit lane offset and a scalar offset, so walking the groups costs no
// vector address arithmetic and no 64-bit lane pointers. Every offset used
// is inside the operand it addresses.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, 0xFFFFFFFFu, 0x00020000);
}
__device__ __forceinline__ u32x4_t load_b128(__amdgpu_buffer_rsrc_t r, int off, int soff) {
  return __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(r, off, soff, 0));
}

constexpr int kWidePitch = 17;  // 16-byte blocks per LDS row of one group (padded)

template <int MT>
constexpr size_t wide_lds_bytes() {
  return static_cast<size_t>(4) * 32 * MT * (kWidePitch * 16 + 4);
}

// What a wave multiplies: one weight matrix, or the gate and up matrices.
struct WideArgs {
  const uint8_t* w[2];
  const uint16_t* s[2];
  const uint16_t* x;
  uint16_t* y;
  int N, K, M;
  int tiles_m, tiles_n;
};

struct WideGroupArgs {
  PrefillGroup g;
  int K, M;
  int tiles_m, tiles_n;
};

// The operands of column tile bn, made relative to its projection.
__device__ __forceinline__ const WideArgs& wide_view(const WideArgs& a, int&) { return a; }
__device__ __forceinline__ WideArgs wide_view(const WideGroupArgs& a, int& bn) {
  const PrefillProj v = prefill_proj(a.g, bn);
  return WideArgs{{v.w, v.w}, {v.s, v.s}, a.g.x, v.y, v.n, a.K, a.M, a.tiles_m, a.tiles_n};
}

// SVEC: 4-byte aligned scale pairs (prepacked, or G even and S 4 B aligned)
template <class Act, int MT, int NT, int WV, int OCC, bool PACKED, bool SVEC, bool MULTI, bool GLU,
          int KS = 1, class Args = WideArgs>
__global__ __launch_bounds__(WV * KS * 64, OCC) void w4a16_gemm_wide_kernel(Args args) {
  static_assert(!GLU || NT == 2, "a wave holds a gate and an up tile");
  static_assert(KS == 1 || (!GLU && !MULTI), "a k-slice is one unit");
  constexpr int BM = 32 * MT;
  constexpr int BNW = GLU ? 32 : 32 * NT;  // output columns per wave
  constexpr int NS = BM / 16;              // 16-row staging slices
  constexpr int SPW = (NS + WV - 1) / WV;  // slices per wave
  extern __shared__ u32x4_t lds[];
  constexpr int XB = BM * kWidePitch;  // 16-byte blocks of one group's x
  const int slice = KS == 1 ? 0 : wave_id() / WV;
  u32x4_t* const xs = lds + slice * (wide_lds_bytes<MT>() / 16);
  float* const ob = reinterpret_cast<float*>(xs + 4 * XB);

  const int K = args.K;
  const int G = K >> 7;
  // this slice's groups: [gb, ge), all of them or one 8-group unit
  const int gb = slice * kUnit, ge = KS == 1 ? G : min(G, gb + kUnit);
  const int lane = threadIdx.x & 63;
  const int wave = wave_id() - slice * WV;
  const int j = lane & 31, h = lane >> 5;
  const int i16 = lane & 15, a16 = lane >> 4;

  // tile order: each XCD (workgroup L runs on XCD L % 8) takes a contiguous
  // run of tiles, in bands of 8 tile rows walked column by column
  int bm, bn;
  {
    const int total = args.tiles_m * args.tiles_n;
    const int per = (total + 7) >> 3;
    const int L = blockIdx.x;
    const int idx = (L & 7) * per + (L >> 3);
    if ((L >> 3) >= per || idx >= total) return;
    const int band = 8 * args.tiles_n;
    const int bi = idx / band;
    const int rem = idx - bi * band;
    const int rows = min(8, args.tiles_m - bi * 8);
    bn = rem / rows;
    bm = bi * 8 + rem - bn * rows;
  }
  const WideArgs p = wide_view(args, bn);
  const int N = p.N;
  const int m0 = bm * BM;
  const int mrows = min(BM, p.M - m0);
  const int nbase = (bn * WV + wave) * BNW;
  const bool wave_ok = nbase < N;

  // staging: wave w stages slices w, w + WV, ...: load q of slice s reads
  // row 16 s + 4 q + lane / 16, block lane % 16 of the group
  const auto xsrc = make_rsrc(p.x + static_cast<size_t>(m0) * K);
  int xoff[SPW][4];
#pragma unroll
  for (int sl = 0; sl < SPW; ++sl)
#pragma unroll
    for (int q = 0; q < 4; ++q)
      xoff[sl][q] = min(16 * (wave + sl * WV) + 4 * q + a16, mrows - 1) * K * 2 + 16 * i16;

  // weights: a base per wave (uniform) and 32-bit lane offsets from it
  const int nfirst = min(nbase, N - 1);
  const size_t wfirst = PACKED ? static_cast<size_t>(nfirst >> 4) * packed_tile_bytes(G)
                               : static_cast<size_t>(nfirst) * (K >> 1);
  const auto wsrc0 = make_rsrc(p.w[0] + wfirst);
  const auto wsrc1 = make_rsrc((GLU ? p.w[1] : p.w[0]) + wfirst);
  const auto ssrc0 = PACKED ? wsrc0 : make_rsrc(p.s[0] + static_cast<size_t>(nfirst) * G);
  const auto ssrc1 = PACKED ? wsrc1 : make_rsrc((GLU ? p.s[1] : p.s[0]) + static_cast<size_t>(nfirst) * G);
  int woff[NT], soff[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const int n = min(nbase + (GLU ? 0 : 32 * nt) + j, N - 1);
    if constexpr (PACKED) {
      const int tile = ((n >> 4) - (nfirst >> 4)) * static_cast<int>(packed_tile_bytes(G));
      woff[nt] = tile + 16 * (16 * h + (n & 15));
      soff[nt] = tile + G * 1024 + (n & 15) * packed_scale_pitch(G);
    } else {
      woff[nt] = (n - nfirst) * (K >> 1) + 16 * h;
      soff[nt] = (n - nfirst) * G * 2;
    }
  }
  constexpr int kStep = PACKED ? 1024 : 64;  // bytes between groups of one lane
  constexpr int kHi = PACKED ? 512 : 32;     // lane chunk 2 + h after chunk h

  u32x4_t xr[SPW][4];
  auto load_x = [&](int g) {
#pragma unroll
    for (int sl = 0; sl < SPW; ++sl)
#pragma unroll
      for (int q = 0; q < 4; ++q) xr[sl][q] = load_b128(xsrc, xoff[sl][q], g * (kGroup * 2));
  };
  // Staging of the next group's x, in pieces that the group loop places
  // between its steps: the wave's slice rows go to LDS in pair order
  // (stage_write), come back in MFMA operand layout (stage_read; only this
  // wave writes and reads them here), feed the offset chain one step at a
  // time (stage_chain), and the chain's result goes to the table.
  u32x4_t xo[SPW][2];
  f32x4_t oc[SPW];
  auto slice_ok = [&](int sl) { return NS % WV == 0 || wave + sl * WV < NS; };
  auto stage_write = [&](u32x4_t* xb) {
#pragma unroll
    for (int sl = 0; sl < SPW; ++sl)
      if (slice_ok(sl))
#pragma unroll
        for (int q = 0; q < 4; ++q)
          xb[(16 * (wave + sl * WV) + 4 * q + a16) * kWidePitch + i16] = pair_order(xr[sl][q]);
  };
  auto stage_read = [&](const u32x4_t* xb, int d) {
    if (d == 0) wave_lds_sync();
#pragma unroll
    for (int sl = 0; sl < SPW; ++sl)
      xo[sl][d & 1] = xb[(16 * min(wave + sl * WV, NS - 1) + i16) * kWidePitch + 4 * a16 + d];
  };
  auto stage_chain = [&](int d) {
    const u32x4_t neg = {Act::kNegOffsetPair, Act::kNegOffsetPair, Act::kNegOffsetPair,
                         Act::kNegOffsetPair};
    const f32x4_t zero = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int sl = 0; sl < SPW; ++sl) oc[sl] = Act::mma(xo[sl][d & 1], neg, d == 0 ? zero : oc[sl]);
  };
  auto stage_table = [&](float* ob) {
#pragma unroll
    for (int sl = 0; sl < SPW; ++sl)
      if (slice_ok(sl))  // every column of the chain's tile holds the same values
        *reinterpret_cast<f32x4_t*>(ob + 16 * (wave + sl * WV) + 4 * a16) = oc[sl];
  };

  struct WBuf {
    u32x4_t lo[NT], hi[NT];
  };
  auto load_w = [&](WBuf& b, int g) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      b.lo[nt] = load_b128(nt == 0 || !GLU ? wsrc0 : wsrc1, woff[nt], g * kStep);
      b.hi[nt] = load_b128(nt == 0 || !GLU ? wsrc0 : wsrc1, woff[nt] + kHi, g * kStep);
    }
  };
  // scales of groups g, g + 1 (g even)
  auto load_s = [&](uint32_t (&sc)[NT], int g) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const auto src = nt == 0 || !GLU ? ssrc0 : ssrc1;
      if constexpr (PACKED || SVEC)
        sc[nt] = __builtin_amdgcn_raw_buffer_load_b32(src, soff[nt], 2 * g, 0);
      else
        sc[nt] = __builtin_amdgcn_raw_buffer_load_b16(src, soff[nt], 2 * g, 0) |
                 (static_cast<uint32_t>(
                      __builtin_amdgcn_raw_buffer_load_b16(src, soff[nt], 2 * min(g + 1, G - 1), 0))
                  << 16);
    }
  };

  const f32x16_t zero16 = {};
  f32x16_t part[MT][NT];
  f32x16_t acc[MULTI ? MT : 1][NT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      part[mt][nt] = zero16;
      if constexpr (MULTI) acc[mt][nt] = zero16;
    }

  // One group: eight 16-k steps, the operands of a step read and decoded
  // during the step before. between(s) runs beside step s.
  auto group = [&](const u32x4_t* xb, const float* ob, const WBuf& b, const uint32_t (&sc)[NT],
                   int odd, auto&& between, auto&& tail) {
    const u32x4_t* xa = xb + j * kWidePitch + 4 * h;
    u32x4_t A[2][MT], B[2][NT];
    auto fetch = [&](int s) {
      const int d = s >> 1, e = s & 1;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) A[s & 1][mt] = xa[mt * 32 * kWidePitch + 8 * e + d];
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
        B[s & 1][nt] = Act::template decode<PACKED>(e == 0 ? b.lo[nt][d] : b.hi[nt][d]);
    };
    fetch(0);
    f32x16_t t[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const float* cr = ob + mt * 32 + 4 * h;
      f32x16_t o;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x4_t o4 = *reinterpret_cast<const f32x4_t*>(cr + 8 * q);
#pragma unroll
        for (int r = 0; r < 4; ++r) o[4 * q + r] = o4[r];
      }
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) t[mt][nt] = o;
    }
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      __builtin_amdgcn_sched_barrier(0);
      if (s < 7) fetch(s + 1);
      between(s);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) t[mt][nt] = mfma32<Act>(A[s & 1][mt], B[s & 1][nt], t[mt][nt]);
    }
    __builtin_amdgcn_sched_barrier(0);
    tail();
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      float s = half_bits_to_f32((sc[nt] >> (16 * odd)) & 0xFFFFu);
      asm("" : "+v"(s));  // keeps v_fma_f32: v_fma_mix_f32 on the fp16 bits issues at a lower rate
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          part[mt][nt][r] = __builtin_fmaf(s, t[mt][nt][r], part[mt][nt][r]);
    }
  };

  WBuf w0, w1;
  uint32_t sc[NT], scn[NT];
  const auto fold = [&] {
    if constexpr (MULTI) {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
          acc[mt][nt] = acc[mt][nt] + part[mt][nt];
          part[mt][nt] = zero16;
        }
    }
  };
  // prologue: the first two groups of x, then the first weights
  {
    load_x(min(gb, G - 1));
    u32x4_t x0[SPW][4];
#pragma unroll
    for (int sl = 0; sl < SPW; ++sl)
#pragma unroll
      for (int q = 0; q < 4; ++q) x0[sl][q] = xr[sl][q];
    load_x(min(gb + 1, G - 1));
    u32x4_t x1[SPW][4];
#pragma unroll
    for (int sl = 0; sl < SPW; ++sl)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        x1[sl][q] = xr[sl][q];
        xr[sl][q] = x0[sl][q];
      }
    load_w(w0, min(gb, G - 1));
    load_s(sc, min(gb, (G - 1) & ~1));
    stage_write(xs);
#pragma unroll
    for (int sl = 0; sl < SPW; ++sl)
#pragma unroll
      for (int q = 0; q < 4; ++q) xr[sl][q] = x1[sl][q];
    stage_write(xs + XB);
    load_x(min(gb + 2, G - 1));
    // both groups' offset chains side by side, all their reads ahead
    wave_lds_sync();
    u32x4_t xq[2][SPW][4];
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int sl = 0; sl < SPW; ++sl)
#pragma unroll
        for (int d = 0; d < 4; ++d)
          xq[q][sl][d] = xs[q * XB + (16 * min(wave + sl * WV, NS - 1) + i16) * kWidePitch + 4 * a16 + d];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
#pragma unroll
      for (int sl = 0; sl < SPW; ++sl) oc[sl] = group_offset_t<Act>(xq[q][sl]);
      stage_table(ob + q * BM);
    }
  }
  __syncthreads();
  int g = gb, cur = 0;
  // (k-slices all walk whole units: they share the barriers)
  for (; KS == 1 ? g + 1 < G : g < gb + kUnit; g += 2, cur ^= 2) {
    // groups g and g + 1 from one buffer pair, g + 2 and g + 3 staged into
    // the other meanwhile
    const int nxt = cur ^ 2;
    const auto even = [&] { group(xs + cur * XB, ob + cur * BM, w0, sc, 0, [&](int s) {
      if (s == 0) stage_write(xs + nxt * XB);
      if (s == 1) load_x(min(g + 3, G - 1));
      if (s == 1) load_w(w1, KS == 1 ? g + 1 : min(g + 1, G - 1));
      if (s == 1) load_s(scn, min(g + 2, (G - 1) & ~1));
      if (s >= 3 && s < 7) stage_chain(s - 3);
      if (s >= 2 && s < 6) stage_read(xs + nxt * XB, s - 2);
      if (s == 7) stage_table(ob + nxt * BM);
    }, [] {}); };
    const auto odd = [&] { group(xs + cur * XB + XB, ob + cur * BM + BM, w1, sc, 1, [&](int s) {
      if (s == 0) stage_write(xs + nxt * XB + XB);
      if (s == 1) load_x(min(g + 4, G - 1));
      if (s == 1) load_w(w0, min(g + 2, G - 1));
      if (s >= 3 && s < 7) stage_chain(s - 3);
      if (s >= 2 && s < 6) stage_read(xs + nxt * XB + XB, s - 2);
      if (s == 7) stage_table(ob + nxt * BM + BM);
    }, [] { if (KS == 1) __syncthreads(); }); };
    if constexpr (KS == 1) {
      even();
      odd();
    } else {
      if (g < ge) even();
      if (g + 1 < ge) odd();
      __syncthreads();
    }
    if (MULTI && (g & 7) == 6) fold();
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) sc[nt] = scn[nt];
  }
  if (KS == 1 && g < G) group(xs + cur * XB, ob + cur * BM, w0, sc, 0, [](int) {}, [] {});
  if (MULTI && (G & 7) != 0) fold();
  // every wave is done with the staged x; from here on each wave has its own
  // part of the LDS
  __syncthreads();
  if constexpr (KS > 1) {
    // unit partials meet in LDS and slice 0 sums them in unit order
    f32x4_t* const slots = reinterpret_cast<f32x4_t*>(lds) + (wave * MT * NT * 4) * 64 + lane;
    constexpr int SLICE = WV * MT * NT * 4 * 64;  // f32x4 slots per slice
    static_assert(static_cast<size_t>(KS - 1) * SLICE * 16 <= KS * wide_lds_bytes<MT>(), "fits");
    if (slice > 0) {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
          for (int q = 0; q < 4; ++q)
            slots[(slice - 1) * SLICE + ((mt * NT + nt) * 4 + q) * 64] =
                f32x4_t{part[mt][nt][4 * q], part[mt][nt][4 * q + 1], part[mt][nt][4 * q + 2],
                        part[mt][nt][4 * q + 3]};
    }
    __syncthreads();
    if (slice == 0) {
      const int U = (G + kUnit - 1) / kUnit;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) part[mt][nt] = zero16 + part[mt][nt];
      for (int u = 1; u < U; ++u)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              const f32x4_t o = slots[(u - 1) * SLICE + ((mt * NT + nt) * 4 + q) * 64];
#pragma unroll
              for (int r = 0; r < 4; ++r) part[mt][nt][4 * q + r] = part[mt][nt][4 * q + r] + o[r];
            }
    }
    __syncthreads();
    if (slice != 0) return;
  }
  if (!wave_ok) return;
  constexpr bool F16 = std::is_same<Act, ActF16>::value;
  constexpr int kOutPitch = BNW + kOutPad;  // 16-bit elements per LDS output row
  static_assert(static_cast<size_t>(WV) * BM * kOutPitch * 2 <= wide_lds_bytes<MT>(), "fits");
  uint16_t* const ot = reinterpret_cast<uint16_t*>(lds) + wave * BM * kOutPitch;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    // one unit: total = 0 + part; kUnit * total in one exact fma
    f32x16_t v[NT];
    bool bad = false;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      v[nt] = MULTI ? acc[MULTI ? mt : 0][nt] : part[mt][nt];
#pragma unroll
      for (int r = 0; r < 16; ++r) v[nt][r] = __builtin_fmaf(Act::kUnit, v[nt][r], 0.0f);
#pragma unroll
      for (int r = 0; r < 16; r += 2) bad |= __builtin_isunordered(v[nt][r], v[nt][r + 1]);
    }
    uint16_t* const pair = ot + (mt * 32 + 4 * h + (j & 1)) * kOutPitch + (j & ~1);
#pragma unroll
    for (int r = 0; r < 16; r += 2)
#pragma unroll
      for (int nt = 0; nt < (GLU ? 1 : NT); ++nt) {
        uint32_t own;
        if constexpr (GLU)
          own = silu_mul_bits(f32_to_bf16_rne(v[0][r]), f32_to_bf16_rne(v[1][r])) |
                silu_mul_bits(f32_to_bf16_rne(v[0][r + 1]), f32_to_bf16_rne(v[1][r + 1])) << 16;
        else
          own = Act::round2(v[nt][r], v[nt][r + 1]);
        put_row_pair(pair + (8 * (r >> 2) + (r & 3)) * kOutPitch + 32 * nt, own, j);
      }
    if (__builtin_expect(bad, 0)) {
      // outputs whose fast sum is NaN: the reference loop's value instead
      wave_lds_sync();
      for (int q = 0; q < 16 * NT; ++q) {
        const int r = q & 15, nt = q >> 4;
        const int m = mt * 32 + 8 * (r >> 2) + 4 * h + (r & 3);
        const int n = nbase + (GLU ? 0 : 32 * nt) + j;
        if (m >= mrows || n >= N) continue;
        float f[NT];
#pragma unroll
        for (int c = 0; c < NT; ++c) {
          f[c] = v[c][0];
#pragma unroll
          for (int e = 1; e < 16; ++e) f[c] = r == e ? v[c][e] : f[c];
        }
        const uint16_t* xrow = p.x + static_cast<size_t>(m0 + m) * K;
        if constexpr (GLU) {
          const float own = nt == 0 ? f[0] : f[1];
          if (own == own) continue;
          // (no dynamic index into the argument copy: that would live in scratch)
          const float e = w4a16_ref_dot<PACKED>(nt == 0 ? p.w[0] : p.w[1], nt == 0 ? p.s[0] : p.s[1],
                                                K, n, xrow);
          // gate first (q ascending): up's turn recomputes gate if it was NaN too
          float g = nt == 0 ? e : f[0];
          const float u = nt == 0 ? f[1] : e;
          if (g != g && nt == 1) g = w4a16_ref_dot<PACKED>(p.w[0], p.s[0], K, n, xrow);
          ot[m * kOutPitch + j] =
              static_cast<uint16_t>(silu_mul_bits(f32_to_bf16_rne(g), f32_to_bf16_rne(u)));
        } else {
          float own = f[0];
#pragma unroll
          for (int c = 1; c < NT; ++c) own = nt == c ? f[c] : own;
          if (own != own)
            ot[m * kOutPitch + 32 * nt + j] = static_cast<uint16_t>(
                Act::round(w4a16_ref_dot<PACKED, F16>(p.w[0], p.s[0], K, n, xrow)));
        }
      }
    }
  }
  wave_lds_sync();
  store_rows<BM, BNW>(p.y + static_cast<size_t>(m0) * N + nbase, N, ot, mrows, min(BNW, N - nbase),
                      lane, (N & 7) == 0 && (reinterpret_cast<uintptr_t>(p.y) & 15) == 0);
}

template <class Act, int MT, int NT, int WV, int OCC, bool PACKED, bool SVEC, bool MULTI, bool GLU,
          int KS = 1>
int launch_wide_t(WideArgs p, hipStream_t stream) {
  constexpr int BN = WV * (GLU ? 32 : 32 * NT);
  p.tiles_m = (p.M + 32 * MT - 1) / (32 * MT);
  p.tiles_n = (p.N + BN - 1) / BN;
  auto kern = w4a16_gemm_wide_kernel<Act, MT, NT, WV, OCC, PACKED, SVEC, MULTI, GLU, KS>;
  const size_t lds = KS * wide_lds_bytes<MT>();
  if (!allow_lds(kern, lds)) return CUDALM_W4A16_ELAUNCH;
  const int grid = 8 * ((p.tiles_m * p.tiles_n + 7) / 8);  // an equal run of tiles per XCD
  hipLaunchKernelGGL(kern, dim3(grid), dim3(WV * KS * 64), lds, stream, p);
  return launch_status();
}

WideArgs wide_args(const uint8_t* W0, const uint16_t* S0, const uint8_t* W1, const uint16_t* S1,
                   const uint16_t* X, uint16_t* Y, int N, int K, int M) {
  return WideArgs{{W0, W1}, {S0, S1}, X, Y, N, K, M, 0, 0};
}

// Tiles of BM x BN outputs, -1 beyond the kernel's index ranges (32-bit thread
// numbers and lane offsets; M as in the other prefill kernels' grids). A y of
// about 275 GB reaches the first past K = 1024, in tiles of 64 x 128; the unit
// GEMM's two-dimensional grid holds it.
long long wide_tiles(int N, int K, int M, int bm, int bn) {
  if (K > (1 << 20) || M > 65535 * 32) return -1;
  const long long t = static_cast<long long>((M + bm - 1) / bm) * ((N + bn - 1) / bn);
  return t <= kMaxGemmTiles ? t : -1;
}

// Where the wide kernel beats the smaller-tiled prefill kernels. Two lines, in
// us below, theirs first.
//
// A fill line on 64 x 256 tiles (t of them on 256 CUs). Prepacked: 25/32 of a
// tile per CU: K = 1024 t = 182 12.2 / 12.4, 192 12.2 / 12.5, 208 15.0 / 12.8,
// 768 42.3 / 29.8; K = 3584 t = 112 25.2 / 25.6, 208 44.6 / 35.0. File layout,
// whose loads the smaller tiles repeat more often: 5/8 at K <= 1024 (t = 128
// 9.6 / 9.7, 182 14.1 / 13.2, 768 46.8 / 32.3) and 3/8 beyond (K = 2048 t = 96
// 17.0 / 15.5, 64 11.5 / 13.8; K = 3584 t = 104 33.6 / 25.7).
//
// Both sides then step by rounds of one workgroup per CU: w of this kernel's
// tiles (64 x 256, 64 x 128 past K = 1024) and s of the 128 x 32 ones, and a
// ragged M or N, which this kernel pads further, costs it rounds they do not
// take. Medians over 2,000 random shapes by round, K = 1024 prepacked: s = 2 9.8,
// 3 15, 4 21, 5 24, 6 30, 7 34; w = 1 13.5, 2 23, 3 32. File layout s = 2 11, 3
// 16, 4 20, 5 24, 6 28, 7 34; w = 1 14.5, 2 25, 3 35. So at K <= 1024 s > 2 w
// (K = 1024 file layout N = 20342, M = 80 10.0 / 13.9; N = 41863, M = 65 19.2 /
// 23.4); at most K = 256 prepacked, 512 file layout, where s = 4 equals w = 2,
// s >= 2 w, and K <= 256 file layout keeps the fill line alone (s = 2 8.3, w = 1
// 7.3). Past K = 1024, K = 2048 prepacked: s = 2 17.5, 3 24.8, 4 34, 5 40, 6 47, 7
// 54; w = 1 17, 2 26, 3 39, 4 50: 2 s >= 3 w (N = 50045, M = 72 39.9 / 48.4),
// which also holds for file-layout scales that are loaded a unit at a time
// (K a multiple of 1024: N = 19595, M = 65 19.1 / 24.4). Those loaded one by
// one slow the smaller tiles (K = 3584: s = 2 35, 3 51, 4 67, 5 81; w = 1 26.5,
// 2 39.5, 3 61, 4 78): 3 s >= 4 w.
//
// A narrow matrix (N <= 64) leaves half of a 128 x 32 tile's waves or more
// without rows, and counts half a tile (K = 1024 prepacked N = 19, M = 16391
// 9.4 / 18.1; file layout K = 2048 N = 17, M = 7735 8.0 / 16.6); in a group, where
// the other projections' tiles share the CU with it, three quarters, and a whole
// one at K <= 512 (K = 1024 file layout (18, 23, 33), M = 11605: one call per
// projection 20.1 / 29.1).
bool wide_rounds_pay(bool packed, int K, long long wide, long long small8) {
  const long long cus = cu_count();
  const long long w = (wide + cus - 1) / cus;
  const long long s = (small8 + 8 * cus - 1) / (8 * cus);  // small8: eighths of a tile
  if (K > kUnit * kGroup)
    return packed || (K / kGroup) % kUnit == 0 ? 2 * s >= 3 * w : 3 * s >= 4 * w;
  if (!packed && K <= 2 * kGroup) return true;
  if (K <= (packed ? 2 : 4) * kGroup) return s >= 3 && s >= 2 * w;
  return s > 2 * w;
}

// 32nds of a 64 x 256 tile per CU that make the fill line
template <bool PACKED>
int wide_fill(int K) {
  return PACKED ? 25 : K <= kUnit * kGroup ? 20 : 12;
}

int wide_tile_cols(int K) { return K <= kUnit * kGroup ? 256 : 128; }

}  // namespace

template <bool PACKED>
bool wide_serves(int N, int K, int M) {
  const long long t = wide_tiles(N, K, M, 64, 256), wide = wide_tiles(N, K, M, 64, wide_tile_cols(K));
  if (t < 0 || wide < 0 || 32 * t < wide_fill<PACKED>(K) * cu_count()) return false;
  const long long cols8 = N <= 64 ? 4 : 8LL * ((N + 127) / 128);
  return wide_rounds_pay(PACKED, K, wide, (M + 31) / 32 * cols8);
}

// Projections sharing x: the same lines on the tiles of all of them (their
// single calls reach them later, if at all).
template <bool PACKED>
bool wide_group_serves(const PrefillGroup& P, int K, int M) {
  long long t = 0, wide = 0, cols8 = 0;
  for (int j = 0; j < P.count; ++j) {
    const int N = P.n[j], bn = wide_tile_cols(K);
    if (wide_tiles(N, K, M, 64, bn) < 0) return false;
    t += static_cast<long long>((M + 63) / 64) * ((N + 255) / 256);
    wide += static_cast<long long>((M + 63) / 64) * ((N + bn - 1) / bn);
    cols8 += N <= 64 && K > 4 * kGroup ? 6 : 8LL * ((N + 127) / 128);
  }
  if (wide > kMaxGemmTiles || 32 * t < wide_fill<PACKED>(K) * cu_count()) return false;
  return wide_rounds_pay(PACKED, K, wide, (M + 31) / 32 * cols8);
}

template <int NT, bool PACKED, bool SVEC, bool MULTI>
int launch_wide_group_t(WideGroupArgs a, hipStream_t stream) {
  constexpr int BN = 4 * 32 * NT;
  a.tiles_m = (a.M + 63) / 64;
  a.tiles_n = 0;
  for (int j = 0; j < a.g.count; ++j) {
    a.tiles_n += (a.g.n[j] + BN - 1) / BN;
    a.g.end[j] = a.tiles_n;
  }
  auto kern = w4a16_gemm_wide_kernel<ActBf16, 2, NT, 4, 2, PACKED, SVEC, MULTI, false, 1, WideGroupArgs>;
  const size_t lds = wide_lds_bytes<2>();
  if (!allow_lds(kern, lds)) return CUDALM_W4A16_ELAUNCH;
  const int grid = 8 * ((a.tiles_m * a.tiles_n + 7) / 8);
  hipLaunchKernelGGL(kern, dim3(grid), dim3(256), lds, stream, a);
  return launch_status();
}

template <bool PACKED>
int launch_wide_group(const PrefillGroup& P, int K, int M, hipStream_t stream) {
  const WideGroupArgs a = {P, K, M, 0, 0};
  if constexpr (!PACKED) {
    bool svec = (K / kGroup) % 2 == 0;
    for (int j = 0; j < P.count; ++j) svec = svec && aligned(P.s[j], 4);
    if (!svec)
      return K <= kUnit * kGroup ? launch_wide_group_t<2, PACKED, false, false>(a, stream)
                                 : launch_wide_group_t<1, PACKED, false, true>(a, stream);
  }
  return K <= kUnit * kGroup ? launch_wide_group_t<2, PACKED, true, false>(a, stream)
                             : launch_wide_group_t<1, PACKED, true, true>(a, stream);
}
template bool wide_group_serves<true>(const PrefillGroup&, int, int);
template bool wide_group_serves<false>(const PrefillGroup&, int, int);
template int launch_wide_group<true>(const PrefillGroup&, int, int, hipStream_t);
template int launch_wide_group<false>(const PrefillGroup&, int, int, hipStream_t);

template <class Act, bool PACKED>
int launch_wide(const uint8_t* W, const uint16_t* S, const uint16_t* X, uint16_t* Y, int N, int K,
                int M, hipStream_t stream) {
  const WideArgs p = wide_args(W, S, W, S, X, Y, N, K, M);
  const bool svec = PACKED || ((K / kGroup) % 2 == 0 && aligned(S, 4));
  if (K <= kUnit * kGroup) {
    if constexpr (!PACKED)
      if (!svec) return launch_wide_t<Act, 2, 2, 4, 2, PACKED, false, false, false>(p, stream);
    return launch_wide_t<Act, 2, 2, 4, 2, PACKED, true, false, false>(p, stream);
  }
  if constexpr (!PACKED)
    if (!svec) return launch_wide_t<Act, 2, 1, 4, 2, PACKED, false, true, false>(p, stream);
  return launch_wide_t<Act, 2, 1, 4, 2, PACKED, true, true, false>(p, stream);
}

// Few tiles of long K (a down projection): four k-slices of one unit each per
// 32 x 128 tile, 16 waves, where the unit GEMM's 64 x 32 tiles no longer fill
// one round and its 128 x 32 tiles, one slice of 8 waves, walk every unit
// alone. 1024 x 3584 prepacked / file layout, unit GEMM first: M = 777 18.7 ->
// 15.5 / 22.4 -> 18.4 us, M = 1000 20.0 -> 16.2 / 23.4 -> 18.7; 2048 x 4096, M =
// 500 19.0 -> 17.8 / 21.1 -> 22.0, so the file layout takes it only where the
// unit GEMM cannot load a unit's scales at once (K / 128 not a multiple of 8).
// Below one round of 64 x 32 tiles (M = 512: 12.9 against 14.7 us) and at
// short K the unit GEMM is faster (K = 2048, two slices, M = 777 9.9 against
// 10.6 us; prepacked 4096 x 2304, M = 256 11.1 against 11.5, file layout 14.7
// against 12.6). Three units (prepacked 2560 < K <= 3072) leave one slice idle,
// and where the 128 x 32 tiles are what the unit GEMM would run, it is as fast or
// faster when the column tiles are even in number: they are numbered first, so a
// workgroup's XCD (its number % 8) then keeps to half, a quarter or an eighth of
// the weights. Slices / unit GEMM, median and range over 2,200 random shapes:
// odd 0.92 (0.80 - 1.07), even 1.02 (0.84 - 1.12), from 25/32 of a round 0.95;
// multiples of four 1.06 (0.82 - 1.18; 3050 x 3072, M = 276 15.2 / 13.1 us). What
// bounds the slices is VALU: at 32 rows a decoded dword feeds one MFMA.
template <bool PACKED>
bool wide_slices_serve(const uint16_t* S, int N, int K, int M) {
  if (K <= (PACKED ? 20 * kGroup : 2 * kUnit * kGroup) || K > 4 * kUnit * kGroup) return false;
  if (!PACKED && (K / kGroup) % 8 == 0 && aligned(S, 16)) return false;
  const long long rows = (M + 31) / 32, cols = (N + 127) / 128, cus = cu_count();
  if (rows * ((N + 63) / 64) <= cus || rows * cols > cus) return false;
  if (!PACKED || K > 3 * kUnit * kGroup || 5 * rows * cols < 3 * cus) return true;
  return cols % 2 != 0 || (cols % 4 != 0 && 32 * rows * cols >= 25 * cus);
}

template <class Act, bool PACKED>
int launch_wide_slices(const uint8_t* W, const uint16_t* S, const uint16_t* X, uint16_t* Y, int N,
                       int K, int M, hipStream_t stream) {
  const WideArgs p = wide_args(W, S, W, S, X, Y, N, K, M);
  if constexpr (!PACKED)
    if ((K / kGroup) % 2 != 0 || !aligned(S, 4))
      return launch_wide_t<Act, 1, 1, 4, 1, PACKED, false, false, false, 4>(p, stream);
  return launch_wide_t<Act, 1, 1, 4, 1, PACKED, true, false, false, 4>(p, stream);
}

bool wide_swiglu_fits(int N, int K, int M) { return wide_tiles(N, K, M, 64, 128) >= 0; }

template <bool PACKED>
int launch_wide_swiglu(const uint8_t* Wg, const uint16_t* Sg, const uint8_t* Wu,
                       const uint16_t* Su, const uint16_t* X, uint16_t* Y, int N, int K, int M,
                       hipStream_t stream) {
  const WideArgs p = wide_args(Wg, Sg, Wu, Su, X, Y, N, K, M);
  const bool svec = PACKED || ((K / kGroup) % 2 == 0 && aligned(Sg, 4) && aligned(Su, 4));
  if (K <= kUnit * kGroup) {
    if constexpr (!PACKED)
      if (!svec) return launch_wide_t<ActBf16, 2, 2, 4, 2, PACKED, false, false, true>(p, stream);
    return launch_wide_t<ActBf16, 2, 2, 4, 2, PACKED, true, false, true>(p, stream);
  }
  if constexpr (!PACKED)
    if (!svec) return launch_wide_t<ActBf16, 2, 2, 4, 1, PACKED, false, true, true>(p, stream);
  return launch_wide_t<ActBf16, 2, 2, 4, 1, PACKED, true, true, true>(p, stream);
}

#define W4A16_WIDE(ACT, PACKED)                                                          \
  template int launch_wide_slices<ACT, PACKED>(const uint8_t*, const uint16_t*,          \
                                               const uint16_t*, uint16_t*, int, int, int, \
                                               hipStream_t);                             \
  template int launch_wide<ACT, PACKED>(const uint8_t*, const uint16_t*, const uint16_t*, \
                                        uint16_t*, int, int, int, hipStream_t)
W4A16_WIDE(ActBf16, true);
W4A16_WIDE(ActBf16, false);
W4A16_WIDE(ActF16, true);
W4A16_WIDE(ActF16, false);
#undef W4A16_WIDE
#define W4A16_WIDE_SWIGLU(PACKED)                                                          \
  template bool wide_serves<PACKED>(int, int, int);                                       \
  template bool wide_slices_serve<PACKED>(const uint16_t*, int, int, int);                \
  template int launch_wide_swiglu<PACKED>(const uint8_t*, const uint16_t*, const uint8_t*, \
                                          const uint16_t*, const uint16_t*, uint16_t*, int, int, \
                                          int, hipStream_t)
W4A16_WIDE_SWIGLU(true);
W4A16_WIDE_SWIGLU(false);
#undef W4A16_WIDE_SWIGLU

}  // namespace cudalm_hip
