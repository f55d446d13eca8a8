// bf16 GEMM for M > 32 activation rows (the tied LM head of a large decode
// batch or of scored text) on MI355X (gfx950); dispatched by
// bf16_gemv_kernels.hip, which serves M <= 32.
//
// Contract (reference: src/kernels/batch_decode.cu:195-236):
//   y[m,n] = bf16_rne( sum_k f32(W[n,k]) * f32(x[m,k]) ), fp32 accumulation.
//
// What bounds it. Up to M = 64 the weight stream: 508.6 MB of a 248320 x 1024
// head, read once (5.1 TB/s packed at M = 64 with 31.8 MB of outputs beside
// it; a 1 GiB copy reaches 5.1 TB/s, a fill 6.8). Beyond, LDS and the matrix
// cores: per 64-k stage a workgroup of 128 x 128 outputs spends ~540 LDS
// cycles (8 writes and 16 reads of 1 KB per wave) beside 528 MFMA cycles.
// 248320 x 1024, file layout / tile-major copy, us, against 32-row chunks that
// each stream the weights again (same box):
//   M = 33 180 -> 102 / 174 -> 93, M = 64 188 -> 110 / 187 -> 100,
//   M = 128 372 -> 126 / 367 -> 115, M = 256 744 -> 199 / 728 -> 193.
// Three register sets of loads in flight instead of two (D = 3): 5 % slower (fewer
// waves resident); 64-wide n per wave at M <= 64: 4x (spills); 256 x 128 tiles of 8
// waves: level at M = 256, 174 us at M = 128.
//
// Same bits as the decode kernel: a 16 x 16 x 32 MFMA step over k-blocks
// (b0, b1, b2, b3) equals two 32 x 32 x 16 steps over (b0, b1) and (b2, b3),
// so every output is one chain over k in ascending 16-wide steps from zero;
// the zeros that pad the last stage leave a sum as it is.
//
// Work decomposition. A workgroup of 4 waves owns 64 x 128 outputs (M <= 64:
// 64 x 32 per wave) or 128 x 128 (64 x 64 per wave). Both operands go through
// double-buffered LDS in 64-k stages, in whole 128-byte lines (tile-major copy:
// whole 1 KB slabs). Two register sets of loads are in flight (D = 2): a stage is
// requested three stages before its turn and put into LDS one before it. Tiles of one
// weight row block run on neighbouring workgroups of one XCD, so that its
// second reader finds it in that XCD's L2.

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "bf16_gemm.h"
#include "hip_common.h"
#include "w4a16_device.h"

namespace cudalm_hip {
namespace {

constexpr int kBK = 64;           // k per stage
constexpr int kBlocks = kBK / 8;  // 16-byte blocks per row and stage

// LDS block of logical block c of row r: rows are 128 B, so 16 consecutive
// rows' blocks land in the 16 different 16-byte slots of the 64 banks.
__device__ __forceinline__ int slot(int r, int c) { return r * kBlocks + (c ^ ((r >> 1) & 7)); }

template <int BM, int BN>
constexpr size_t gemm_lds_bytes() {
  return static_cast<size_t>(2) * (BM + BN) * kBlocks * 16;
}

template <int MT, int NT, int WM, int WN, int OCC, int D, bool PACKED>
__global__ __launch_bounds__(WM * WN * 64, OCC) void bf16_gemm_kernel(
    const uint16_t* __restrict__ W, const uint16_t* __restrict__ X, uint16_t* __restrict__ Y, int N,
    int K, int M, int tiles_m, int tiles_n) {
  constexpr int BM = 32 * MT * WM, BN = 32 * NT * WN, NTH = WM * WN * 64;
  constexpr int XL = BM * kBlocks / NTH, WL = BN * kBlocks / NTH;  // 16-byte loads per thread
  static_assert(BM * kBlocks % NTH == 0 && BN * kBlocks % NTH == 0, "whole loads");
  constexpr int BUF = (BM + BN) * kBlocks;
  extern __shared__ u32x4_t lds[];

  int bm, bn;
  {
    const int total = tiles_m * tiles_n;
    const int per = (total + 7) >> 3;
    const int L = blockIdx.x;
    const int idx = (L & 7) * per + (L >> 3);
    if ((L >> 3) >= per || idx >= total) return;
    bn = idx / tiles_m;
    bm = idx - bn * tiles_m;
  }
  const int tid = static_cast<int>(threadIdx.x);
  const int lane = tid & 63, wave = wave_id();
  const int j = lane & 31, h = lane >> 5;
  const int wm = wave / WN, wn = wave - wm * WN;
  const int m0 = bm * BM, n0 = bn * BN;
  const int mrows = min(BM, M - m0);

  // load q of a thread: x row tid / 8 + q * NTH / 8, block tid % 8 of the
  // stage; W the same, or (packed) row 16 t + l % 16 of its tile-major slabs
  const uint16_t* xsrc[XL];
#pragma unroll
  for (int q = 0; q < XL; ++q)
    xsrc[q] = X + static_cast<size_t>(m0 + min(tid / 8 + q * (NTH / 8), mrows - 1)) * K + 8 * (tid & 7);
  const uint16_t* wsrc[WL];
  int wdst[WL];
#pragma unroll
  for (int q = 0; q < WL; ++q) {
    if constexpr (PACKED) {
      // wave-load = one slab (16 rows x 32 k): slab s of the stage's
      // BN / 16 x 2, tile s / 2, half s % 2
      const int s = wave + q * (NTH / 64);
      const int t = min((n0 >> 4) + (s >> 1), (N >> 4) - 1);
      wsrc[q] = W + static_cast<size_t>(t) * 16 * K + (s & 1) * 512 + lane * 8;
      wdst[q] = slot(16 * (s >> 1) + (lane & 15), 4 * (s & 1) + (lane >> 4));
    } else {
      const int r = tid / 8 + q * (NTH / 8);
      wsrc[q] = W + static_cast<size_t>(min(n0 + r, N - 1)) * K + 8 * (tid & 7);
      wdst[q] = slot(r, tid & 7);
    }
  }
  const int S = (K + kBK - 1) / kBK;
  struct Regs {
    u32x4_t x[XL], w[WL];
  };
  const u32x4_t zero4 = {0u, 0u, 0u, 0u};
  auto load = [&](Regs& r, int s) {
    s = min(s, S - 1);
    const int k = s * kBK;
    const int kx = min(k, K - 8 - 8 * (tid & 7));  // clamped: zeroed when written
#pragma unroll
    for (int q = 0; q < XL; ++q) r.x[q] = *reinterpret_cast<const u32x4_t*>(xsrc[q] + kx);
#pragma unroll
    for (int q = 0; q < WL; ++q) {
      const u32x4_t* p =
          reinterpret_cast<const u32x4_t*>(wsrc[q] + (PACKED ? static_cast<size_t>(s) * 1024 : kx));
      r.w[q] = tiles_m == 1 ? __builtin_nontemporal_load(p) : *p;
    }
  };
  auto put = [&](const Regs& r, int s) {
    u32x4_t* xb = lds + (s & 1) * BUF;
    u32x4_t* wb = xb + BM * kBlocks;
    const bool in = s * kBK + 8 * (tid & 7) < K;
#pragma unroll
    for (int q = 0; q < XL; ++q) xb[slot(tid / 8 + q * (NTH / 8), tid & 7)] = in ? r.x[q] : zero4;
#pragma unroll
    for (int q = 0; q < WL; ++q) wb[wdst[q]] = PACKED || in ? r.w[q] : zero4;
  };
  const f32x16_t zero16 = {};
  f32x16_t acc[MT][NT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = zero16;
  auto compute = [&](int s) {
    const u32x4_t* xb = lds + (s & 1) * BUF;
    const u32x4_t* wb = xb + BM * kBlocks;
#pragma unroll
    for (int q = 0; q < kBK / 16; ++q) {
      u32x4_t A[MT], B[NT];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) A[mt] = xb[slot((wm * MT + mt) * 32 + j, 2 * q + h)];
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) B[nt] = wb[slot((wn * NT + nt) * 32 + j, 2 * q + h)];
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[mt][nt] = mfma32<ActBf16>(A[mt], B[nt], acc[mt][nt]);
    }
  };

  // stage s is loaded D + 1 stages before its turn and put into LDS one
  // stage before it
  Regs r[D];
#pragma unroll
  for (int d = 0; d < D; ++d) load(r[d], d);
  put(r[0], 0);
  load(r[0], D);
  __syncthreads();
  for (int s0 = 0; s0 < S; s0 += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const int s = s0 + d;
      if (s < S) compute(s);
      put(r[(d + 1) % D], s + 1);
      load(r[(d + 1) % D], s + 1 + D);
      __syncthreads();
    }
  }
  const int nb = n0 + wn * 32 * NT;
  if (nb >= N) return;
  uint16_t* const ot = reinterpret_cast<uint16_t*>(lds) + wave * 32 * MT * (32 * NT + kOutPad);
  static_assert(static_cast<size_t>(WM * WN) * 32 * MT * (32 * NT + kOutPad) * 2 <=
                    gemm_lds_bytes<BM, BN>(), "fits");
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    uint16_t* const pair = ot + (mt * 32 + 4 * h + (j & 1)) * (32 * NT + kOutPad) + (j & ~1);
#pragma unroll
    for (int r = 0; r < 16; r += 2)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
        put_row_pair(pair + (8 * (r >> 2) + (r & 3)) * (32 * NT + kOutPad) + 32 * nt,
                     f32_to_bf16_rne2(acc[mt][nt][r], acc[mt][nt][r + 1]), j);
  }
  wave_lds_sync();
  const int mb = wm * 32 * MT;
  store_rows<32 * MT, 32 * NT>(Y + static_cast<size_t>(m0 + mb) * N + nb, N, ot,
                               min(32 * MT, mrows - mb), min(32 * NT, N - nb), lane,
                               (N & 7) == 0 && (reinterpret_cast<uintptr_t>(Y) & 15) == 0);
}

template <int MT, int NT, int WM, int WN, int OCC, int D, bool PACKED>
int launch_gemm_t(const uint16_t* W, const uint16_t* X, uint16_t* Y, int N, int K, int M,
                  hipStream_t stream) {
  constexpr int BM = 32 * MT * WM, BN = 32 * NT * WN;
  auto kern = bf16_gemm_kernel<MT, NT, WM, WN, OCC, D, PACKED>;
  const size_t lds = gemm_lds_bytes<BM, BN>();
  if (!allow_lds(kern, lds)) return CUDALM_W4A16_ELAUNCH;
  const int tm = (M + BM - 1) / BM, tn = (N + BN - 1) / BN;
  hipLaunchKernelGGL(kern, dim3(8 * ((tm * tn + 7) / 8)), dim3(WM * WN * 64), lds, stream, W, X, Y,
                     N, K, M, tm, tn);
  return launch_status();
}

}  // namespace

bool bf16_gemm_fits(int N, int M) {
  const int bm = M <= 64 ? 64 : 128;
  return static_cast<long long>((M + bm - 1) / bm) * ((N + 127) / 128) <= kMaxGemmTiles;
}

template <bool PACKED>
int launch_bf16_gemm(const uint16_t* W, const uint16_t* X, uint16_t* Y, int N, int K, int M,
                     hipStream_t stream) {
  if (M <= 64) return launch_gemm_t<2, 1, 1, 4, 3, 2, PACKED>(W, X, Y, N, K, M, stream);
  return launch_gemm_t<2, 2, 2, 2, 2, 2, PACKED>(W, X, Y, N, K, M, stream);
}
template int launch_bf16_gemm<true>(const uint16_t*, const uint16_t*, uint16_t*, int, int, int,
                                    hipStream_t);
template int launch_bf16_gemm<false>(const uint16_t*, const uint16_t*, uint16_t*, int, int, int,
                                     hipStream_t);

}  // namespace cudalm_hip
