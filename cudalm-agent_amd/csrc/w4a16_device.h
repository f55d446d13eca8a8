// W4A16 device helpers shared by the engine's kernel files (gfx950): the
// weight-layout constants, the exact nibble -> bf16 decode, the activation
// pair order and the MFMA offset chain that cancels the decode's 1.5 bias.
#ifndef CUDALM_W4A16_DEVICE_H
#define CUDALM_W4A16_DEVICE_H

#include <type_traits>

#include "hip_common.h"

namespace cudalm_hip {

constexpr int kGroup = 128;     // quantization group (k)
constexpr int kTileRows = 16;   // weight rows per MFMA tile
constexpr int kUnit = 8;        // groups per streamed unit
constexpr uint32_t kNegOffsetPair = 0xBFC0BFC0u;  // bf16 -1.5 in both halves

__host__ __device__ constexpr int packed_scale_pitch(int G) { return 16 * ((G + 7) / 8); }
__host__ __device__ constexpr size_t packed_tile_bytes(int G) {
  return static_cast<size_t>(G) * 1024 + 16 * static_cast<size_t>(packed_scale_pitch(G));
}

// ---------------------------------------------------------------------------
// device helpers
// ---------------------------------------------------------------------------

__device__ __forceinline__ float half_bits_to_f32(uint32_t h) {
  return static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(h)));
}

// 8 nibbles (k = 0..7 of a block, nibble k at bits 4k) -> 4 bf16 pairs
// (k, k+4), each element 1.5 + q/16. ROT: the dword is the prepacked form,
// rotated left by 3 at load time, so pair 0 is already in place (one
// v_bitop3) and pairs 1..3 need one v_alignbit each: 7 VALU ops instead of 8.
__device__ __forceinline__ uint32_t rotr(uint32_t w, int s) {
  return __builtin_amdgcn_alignbit(w, w, s);
}

template <bool ROT = false>
__device__ __forceinline__ u32x4_t decode_nibbles(uint32_t w) {
  u32x4_t a;
  if constexpr (ROT) {
    a[0] = (w & 0x00780078u) ^ 0x3FC03FC0u;
    a[1] = (rotr(w, 4) & 0x00780078u) ^ 0x3FC03FC0u;
    a[2] = (rotr(w, 8) & 0x00780078u) ^ 0x3FC03FC0u;
    a[3] = (rotr(w, 12) & 0x00780078u) ^ 0x3FC03FC0u;
  } else {
    a[0] = ((w << 3) & 0x00780078u) ^ 0x3FC03FC0u;
    a[1] = ((w >> 1) & 0x00780078u) ^ 0x3FC03FC0u;
    a[2] = ((w >> 5) & 0x00780078u) ^ 0x3FC03FC0u;
    a[3] = ((w >> 9) & 0x00780078u) ^ 0x3FC03FC0u;
  }
  return a;
}

// Prepacked form of a file dword of 8 nibbles (see decode_nibbles<true>).
__host__ __device__ __forceinline__ uint32_t prepack_dword(uint32_t w) {
  return (w << 3) | (w >> 29);
}

// Natural bf16 order [x0x1 x2x3 x4x5 x6x7] -> pair order [x0x4 x1x5 x2x6 x3x7].
__device__ __forceinline__ u32x4_t pair_order(u32x4_t v) {
  u32x4_t p;
  // v_perm_b32 byte select over (hi:lo) = (v[2]:v[0]) and (v[3]:v[1]):
  // p0 = lo16(v0) | lo16(v2) << 16, p1 = hi16(v0) | hi16(v2) << 16, ...
  p[0] = __builtin_amdgcn_perm(v[2], v[0], 0x05040100u);
  p[1] = __builtin_amdgcn_perm(v[2], v[0], 0x07060302u);
  p[2] = __builtin_amdgcn_perm(v[3], v[1], 0x05040100u);
  p[3] = __builtin_amdgcn_perm(v[3], v[1], 0x07060302u);
  return p;
}

// -1.5 * (sum over the group of this lane-set's activation rows), as a 16x16
// accumulator tile (all columns equal).
__device__ __forceinline__ f32x4_t group_offset(const u32x4_t (&xa)[4]) {
  const u32x4_t neg = {kNegOffsetPair, kNegOffsetPair, kNegOffsetPair, kNegOffsetPair};
  const f32x4_t zero = {0.0f, 0.0f, 0.0f, 0.0f};
  f32x4_t c = mfma16(xa[0], neg, zero);
  c = mfma16(xa[1], neg, c);
  c = mfma16(xa[2], neg, c);
  c = mfma16(xa[3], neg, c);
  return c;
}

// Activation / output element type of a kernel instance. Both encode a
// weight nibble as an exact value c + q/kUnit in the activation's 16-bit
// format (the nibble in mantissa bits 3..6), cancel c with an MFMA against
// -c, and scale the accumulated sum by kUnit in the epilogue.
struct ActBf16 {
  static constexpr uint32_t kNegOffsetPair = 0xBFC0BFC0u;  // -1.5, -1.5
  static constexpr float kUnit = 16.0f;  // weight element = 1.5 + q / kUnit
  template <bool ROT>
  __device__ static u32x4_t decode(uint32_t w) { return decode_nibbles<ROT>(w); }
  __device__ static f32x4_t mma(u32x4_t a, u32x4_t b, f32x4_t c) { return mfma16(a, b, c); }
  __device__ static uint32_t round(float f) { return f32_to_bf16_rne(f); }
  // two roundings in one dword (lo in bits 0..15)
  __device__ static uint32_t round2(float lo, float hi) { return f32_to_bf16_rne2(lo, hi); }
  __device__ static float widen(uint32_t h) { return bf16_lo(h); }
};

// fp16: 1.0 = 0x3C00 with 10 mantissa bits, so q/16 sits at bit 6 and the
// biased nibble (q + 8 = nibble ^ 8) goes to bits 6..9: 0x3C00 | 0x0200 is
// 1.5, and the element is exactly 1.5 + q/16, the bf16 element's value. One
// shift (one rotation from the prepacked form, which is the file dword
// rotated left by 3) and one v_bitop3 per pair: 8 VALU ops per dword.
// Keeping the bias at 1.5 (not 1.0625 + q/128 with the nibble at bits
// 3..6, one op less) keeps the fp32 cancellation of the offset chain as
// small as in bf16: the reference fixtures then stay within 0.5 fp16 ulp.
struct ActF16 {
  static constexpr uint32_t kNegOffsetPair = 0xBE00BE00u;  // -1.5, -1.5
  static constexpr float kUnit = 16.0f;  // weight element = 1.5 + q / kUnit
  template <bool ROT>
  __device__ static u32x4_t decode(uint32_t w) {
    u32x4_t a;
    if constexpr (ROT) {
      a[0] = (rotr(w, 29) & 0x03C003C0u) ^ 0x3E003E00u;
      a[1] = (rotr(w, 1) & 0x03C003C0u) ^ 0x3E003E00u;
      a[2] = (rotr(w, 5) & 0x03C003C0u) ^ 0x3E003E00u;
      a[3] = (rotr(w, 9) & 0x03C003C0u) ^ 0x3E003E00u;
    } else {
      a[0] = ((w << 6) & 0x03C003C0u) ^ 0x3E003E00u;
      a[1] = ((w << 2) & 0x03C003C0u) ^ 0x3E003E00u;
      a[2] = ((w >> 2) & 0x03C003C0u) ^ 0x3E003E00u;
      a[3] = ((w >> 6) & 0x03C003C0u) ^ 0x3E003E00u;
    }
    return a;
  }
  __device__ static f32x4_t mma(u32x4_t a, u32x4_t b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a),
                                                  __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
  }
  // round to nearest even (v_cvt_f16_f32 under the default rounding mode)
  __device__ static uint32_t round(float f) {
    return __builtin_bit_cast(uint16_t, static_cast<_Float16>(f));
  }
  __device__ static uint32_t round2(float lo, float hi) { return round(lo) | round(hi) << 16; }
  __device__ static float widen(uint32_t h) { return half_bits_to_f32(h & 0xFFFFu); }
};

// An activation trait bound to a weight layout: decode() reads file dwords
// (PACKED false) or prepacked, rotated dwords (PACKED true).
template <class Act, bool PACKED>
struct Layout : Act {
  __device__ static u32x4_t decode(uint32_t w) { return Act::template decode<PACKED>(w); }
};

// -1.5 * (sum over the group of this lane-set's activation rows) in the
// activation type Act.
template <class Act>
__device__ __forceinline__ f32x4_t group_offset_t(const u32x4_t (&xa)[4]) {
  const u32x4_t neg = {Act::kNegOffsetPair, Act::kNegOffsetPair, Act::kNegOffsetPair,
                       Act::kNegOffsetPair};
  const f32x4_t zero = {0.0f, 0.0f, 0.0f, 0.0f};
  f32x4_t c = Act::mma(xa[0], neg, zero);
  c = Act::mma(xa[1], neg, c);
  c = Act::mma(xa[2], neg, c);
  c = Act::mma(xa[3], neg, c);
  return c;
}

// The reference's own loop for one output (tests/cuda/test_int4_gemv_bf16.cpp:
// 54-69; the fp16 twin, tests/cuda/test_int4_gemv.cpp:49-63): fp32, k
// ascending, each term (q * f32(s)) * f32(x). The kernels call it only for
// an output whose fast sum is NaN. That sum cancels the decode's 1.5 bias
// with a second chain over -1.5 * x, so an infinite activation turns into
// Inf - Inf there, where the reference gives +-Inf when every infinite term
// has one sign (and NaN otherwise, or for a NaN activation, or a zero weight
// or scale times an infinity); overflowing finite sums are the same case.
// Recomputing those outputs in the reference's order gives the reference's
// result. W is the projection's weights (file layout [N, K/2], or prepacked:
// tile-major, dwords rotated left by 3), S its fp16 scales (file layout
// only), xrow the activation row (bf16, or fp16 when F16), read with
// device-coherent loads when XCOH (x written by another workgroup of the
// same launch).
template <bool PACKED, bool F16 = false, bool XCOH = false>
__device__ __forceinline__ float w4a16_ref_dot(const uint8_t* W, const uint16_t* S, int K, int n,
                                            const uint16_t* xrow) {
  const int G = K >> 7;
  const uint8_t* tile = W + static_cast<size_t>(n >> 4) * packed_tile_bytes(G);
  const int i = n & 15;
  float acc = 0.0f;
  for (int k = 0; k < K; ++k) {
    const int g = k >> 7;
    int nib;
    float s;
    if constexpr (PACKED) {
      const int kk = k & 127;
      const uint32_t w = *reinterpret_cast<const uint32_t*>(
          tile + static_cast<size_t>(g) * 1024 + 16 * (16 * (kk >> 5) + i) + 4 * ((kk >> 3) & 3));
      nib = static_cast<int>((rotr(w, 3) >> (4 * (kk & 7))) & 15u);
      s = half_bits_to_f32(*reinterpret_cast<const uint16_t*>(
          tile + static_cast<size_t>(G) * 1024 + i * packed_scale_pitch(G) + 2 * g));
    } else {
      const uint8_t b = W[static_cast<size_t>(n) * (K >> 1) + (k >> 1)];
      nib = (k & 1) ? (b >> 4) : (b & 15);
      s = half_bits_to_f32(S[static_cast<size_t>(n) * G + g]);
    }
    const float q = static_cast<float>((nib ^ 8) - 8);
    const uint32_t xb =
        XCOH ? __hip_atomic_load(xrow + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : xrow[k];
    const float x = F16 ? half_bits_to_f32(xb) : bf16_lo(xb);
    acc += (q * s) * x;
  }
  return acc;
}

typedef float f32x16_t __attribute__((ext_vector_type(16)));

// D = A (32 rows x 16 k) * B (16 k x 32 cols) + C in the activation type,
// fp32 accumulate.
template <class Act>
__device__ __forceinline__ f32x16_t mfma32(u32x4_t a, u32x4_t b, f32x16_t c) {
  if constexpr (std::is_same<Act, ActF16>::value)
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a),
                                                  __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                   __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

// LDS layout of staged activations. A row holds K/8 16-byte blocks plus
// kXPad pad blocks, so rows start 2 blocks (mod 16) apart, and inside each
// 128-column group the block of lane quarter a, step d (logical block
// 4a + d, columns 32a + 8d ..) sits at slot 4d + a. One ds_read_b128 step
// of a wave then reads 4 adjacent blocks from each of 16 rows: measured
// conflict-free on gfx950 (4 LDS cycles per instruction), where unswizzled
// rows 1 block (mod 16) apart spend half their cycles in bank conflicts.
constexpr int kXPad = 2;
__host__ __device__ constexpr int x_pitch(int kcl) { return (kcl >> 3) + kXPad; }
__device__ __forceinline__ int x_slot(int c) { return (c & ~15) | ((c & 3) << 2) | ((c >> 2) & 3); }

__device__ __forceinline__ void load_group_x(u32x4_t (&xa)[4], const u32x4_t* xgroup, int a) {
#pragma unroll
  for (int d = 0; d < 4; ++d) xa[d] = xgroup[4 * d + a];
}

// The output of one accumulator: kUnit * total, or, when that is NaN, the
// reference loop's sum for the output (w4a16_ref_dot: infinite and NaN
// activations and overflow keep the reference's semantics).
template <class Act, bool PACKED>
__device__ __forceinline__ float out_value(float total, const uint8_t* w, const uint16_t* s, int K,
                                           int n, const uint16_t* xrow) {
  const float v = Act::kUnit * total;
  if (__builtin_expect(v != v, 0))
    return w4a16_ref_dot<PACKED, std::is_same<Act, ActF16>::value>(w, s, K, n, xrow);
  return v;
}

// y = bf16( f32(bf16(g / (1 + exp(-g)))) * u ) on bf16 inputs g, u: SiLU in
// fp32, rounded to bf16 first, then the product rounded once
// (include/cudalm/kernels/qwen35_kernels.h:146-152).
// silu_mul_bits(g, u) == mul_bits(silu_bits(g), u): the two roundings as
// separate steps, for callers that have g before u.
__device__ __forceinline__ uint32_t silu_bits(uint32_t g_bits) {
  const float g = bf16_lo(g_bits);
  return f32_to_bf16_rne(g / (1.0f + expf(-g)));
}
__device__ __forceinline__ uint32_t mul_bits(uint32_t s_bits, uint32_t u_bits) {
  return f32_to_bf16_rne(bf16_lo(s_bits) * bf16_lo(u_bits));
}
__device__ __forceinline__ uint32_t silu_mul_bits(uint32_t g_bits, uint32_t u_bits) {
  return mul_bits(silu_bits(g_bits), u_bits);
}

// GEMM of many activation rows (w4a16_gemm.hip; M >= 33, and 17 to 32 rows of
// long K), the kernel chosen by shape, for any N, M and K % 128 == 0.
template <class Act, bool PACKED>
int launch_prefill(const uint8_t* W, const uint16_t* S, const uint16_t* X, uint16_t* Y, int N,
                   int K, int M, hipStream_t stream);

// Up to 8 projections sharing the activations x, for one launch of a prefill
// kernel. Its row tiles are numbered over all projections in order; end[j] is
// the first number past projection j's (set by the launch for its tile size).
struct PrefillGroup {
  const uint8_t* w[CUDALM_W4A16_MAX_PROJ];
  const uint16_t* s[CUDALM_W4A16_MAX_PROJ];
  uint16_t* y[CUDALM_W4A16_MAX_PROJ];
  int n[CUDALM_W4A16_MAX_PROJ];
  int end[CUDALM_W4A16_MAX_PROJ];
  const uint16_t* x;
  int count;
};

struct PrefillProj {
  const uint8_t* w;
  const uint16_t* s;
  uint16_t* y;
  int n;
};

// The projection that owns row tile t (uniform), t made relative to it. Every
// field is read at a constant offset and chosen with scalar selects.
__device__ __forceinline__ PrefillProj prefill_proj(const PrefillGroup& P, int& t) {
  PrefillProj v = {P.w[0], P.s[0], P.y[0], P.n[0]};
  int begin = 0;
#pragma unroll
  for (int j = 1; j < CUDALM_W4A16_MAX_PROJ; ++j) {
    const bool past = j < P.count && t >= P.end[j - 1];
    v.w = past ? P.w[j] : v.w;
    v.s = past ? P.s[j] : v.s;
    v.y = past ? P.y[j] : v.y;
    v.n = past ? P.n[j] : v.n;
    begin = past ? P.end[j - 1] : begin;
  }
  t -= begin;
  return v;
}

template <bool PACKED>
int launch_prefill_group(const PrefillGroup& P, int K, int M, hipStream_t stream);
template <bool PACKED>
bool wide_group_serves(const PrefillGroup& P, int K, int M);
template <bool PACKED>
int launch_wide_group(const PrefillGroup& P, int K, int M, hipStream_t stream);

// SwiGLU front half of M > 32 rows on GEMM tiles, and where those beat the
// `chunks` chunks of at most 32 rows that the fused kernels would run.
bool swiglu_gemm_serves(int N, int K, int M, int chunks, bool packed);
template <bool PACKED>
int launch_gemm_swiglu(const uint8_t* Wg, const uint16_t* Sg, const uint8_t* Wu,
                       const uint16_t* Su, const uint16_t* X, uint16_t* Y, int N, int K, int M,
                       hipStream_t stream);

// The 32 x 32 MFMA kernels of launch_prefill alone: 32 activation rows x 256 weight rows per
// 8-wave workgroup (at K = 1024 the split kernel).
template <class Act, bool PACKED>
int launch_prefill32(const uint8_t* W, const uint16_t* S, const uint16_t* X, uint16_t* Y, int N,
                     int K, int M, hipStream_t stream);

// Registers per lane of the split kernel at K = 1024 and of the unit GEMM
// (prepacked instances).
int prefill32_regs();
int prefill_unit_regs();

// GEMM on 64 x 64 wave tiles (w4a16_gemm_wide.hip; 64 x 32 past K = 1024), and
// whether it is the faster one: 64 x 256 tiles for 25/32 of the CUs (prepacked),
// 20/32 (file layout, K <= 1024) or 12/32 (beyond), and few enough rounds of its
// workgroups beside those of the smaller tiles.
template <bool PACKED>
bool wide_serves(int N, int K, int M);
template <class Act, bool PACKED>
int launch_wide(const uint8_t* W, const uint16_t* S, const uint16_t* X, uint16_t* Y, int N, int K,
                int M, hipStream_t stream);

// Its form with four k-slices of one unit each, for more than one round of 64 x
// 32 tiles and at most one of 128 x 32: prepacked 2560 < K <= 4096 (up to 3072 by
// the number of column tiles too), file layout 2048 < K <= 4096 where a unit's
// scales cannot be loaded at once (K / 128 not a multiple of 8, or scales off 16 B).
template <bool PACKED>
bool wide_slices_serve(const uint16_t* S, int N, int K, int M);
template <class Act, bool PACKED>
int launch_wide_slices(const uint8_t* W, const uint16_t* S, const uint16_t* X, uint16_t* Y, int N,
                       int K, int M, hipStream_t stream);

// The same kernel over gate and up, storing silu(gate) * up.
bool wide_swiglu_fits(int N, int K, int M);
template <bool PACKED>
int launch_wide_swiglu(const uint8_t* Wg, const uint16_t* Sg, const uint8_t* Wu,
                       const uint16_t* Su, const uint16_t* X, uint16_t* Y, int N, int K, int M,
                       hipStream_t stream);

}  // namespace cudalm_hip

#endif
