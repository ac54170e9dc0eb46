// fp32 values as sums of two fp16 values, for contractions on the fp16 matrix units at fp32
// precision (included by .hip sources only).
//
// x = hi + lo + e with hi = fp16(x) and lo = fp16(x - hi), both rounded to nearest (x - hi is
// exact in fp32): hi holds 11 significant bits and lo, with its own sign and exponent, the next
// 11 or 12.  e is zero for three values in four and one step of the fp32 value's last bit for the
// others, |e| <= 2^-23 |x|.  A product x y is taken as lo hi' + hi lo' + hi hi', accumulated in
// fp32 with the largest last; lo lo', below 2^-22 |x y| and of either sign, is left out.  The
// matrix units round once per 16 products, so a sum of n of them is off by less than one fp32
// accumulation of them, which makes n roundings: measured against float64, every timed case and
// every test of unlike sizes is closer than on v_mfma_f32 (prefill.hip).
//
// fp16 has five exponent bits, so operands are scaled by powers of two (exact): the largest
// magnitude of a block goes to [2^14, 2^15), below fp16's 65504, and the smallest step of lo,
// 2^-24, is then 2^-38 of that magnitude.  What such steps do to small values beside large ones is
// bounded by the user of this file, which takes results they could show in again on fp32
// instructions; infinities become NaN in lo and so in the sums they enter, which it detects.
//
// Three v_mfma_f32_32x32x16_f16 do the work of eight v_mfma_f32_32x32x2_f32 at half the cycles
// each: 5.3 times the fp32 matrix rate.  (Three bf16 parts hold every bit and need no scale, but
// six products, as linear.hip takes them: the board's power limit then holds the clock to 1.8 GHz,
// and the 12K + 2K prefill chunk at 32 query heads took 2.05 ms however it was scheduled.)
#pragma once

#include <hip/hip_runtime.h>

namespace nva {

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// Eight values in two fp16 parts: one lane's operand of a 32x32x16 (or 16x16x32) product.
struct Split8 {
  f16x8 hi, lo;
};

// The parts of s x, s a power of two.  (x - hi comes from v_fma_mix_f32, which reads the fp16
// half in place.)
__device__ __forceinline__ Split8 split8(f32x8 x, float s) {
  u32x4 hi, lo;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const float a = x[2 * j], b = x[2 * j + 1];
    const f16x2 h = __builtin_convertvector(f32x2{s * a, s * b}, f16x2);
    const f32x2 r{fmaf(s, a, -(float)h[0]), fmaf(s, b, -(float)h[1])};
    hi[j] = __builtin_bit_cast(uint32_t, h);
    lo[j] = __builtin_bit_cast(uint32_t, __builtin_convertvector(r, f16x2));
  }
  return Split8{__builtin_bit_cast(f16x8, hi), __builtin_bit_cast(f16x8, lo)};
}

// Power-of-two scales of a block by the exponent field e of its largest magnitude (clamped to
// [kMinExp, 255], so that every factor is a normal float): split_scale(e) takes that magnitude
// to [2^14, 2^15), split_unscale(e) takes a result back.
constexpr int kMinExp = 22;
__device__ __forceinline__ int split_exp(float largest) {
  return max((int)(__float_as_uint(largest) >> 23) & 255, kMinExp);
}
__device__ __forceinline__ float split_scale(int e) { return __uint_as_float((uint32_t)(268 - e) << 23); }
__device__ __forceinline__ float split_unscale(int e) { return __uint_as_float((uint32_t)(e - 14) << 23); }

// Largest magnitude of eight values.
__device__ __forceinline__ float abs_max(float m, f32x8 x) {
#pragma unroll
  for (int j = 0; j < 8; j++) m = fmaxf(m, fabsf(x[j]));
  return m;
}

// Sum and max over lanes l and l ^ 32; both lanes get the same bits.
__device__ __forceinline__ float sum_halves(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false,
                                                  false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float max_halves(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false,
                                                  false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

template <int CTRL>
__device__ __forceinline__ uint32_t dpp(uint32_t x) {
  return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, CTRL, 0xf, 0xf, true);
}
template <int CTRL>
__device__ __forceinline__ float max_dpp(float x) {
  return fmaxf(x, __uint_as_float(dpp<CTRL>(__float_as_uint(x))));
}

// The wave's maximum of a in lanes 0-31 and of b in lanes 32-63.
__device__ __forceinline__ float max_waves(float a, float b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false,
                                                  false);
  const float x = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
  const auto t = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false,
                                                  false);
  float y = fmaxf(__uint_as_float(t[0]), __uint_as_float(t[1]));
  y = max_dpp<0x128>(y);  // rotations by 8, 4, 2 and 1 within the 16 lanes of a row
  y = max_dpp<0x124>(y);
  y = max_dpp<0x122>(y);
  return max_dpp<0x121>(y);
}

// Scale exponents of a tile pair from its NW (4 or 8) waves' maxima: lanes 0-31 hold the first
// tensor's (lane l that of wave l % NW), lanes 32-63 the second's.
struct TileExps {
  int a, b;
};
template <int NW>
__device__ __forceinline__ TileExps tile_exps(float largest) {
  uint32_t m = __float_as_uint(largest);
  m = max(m, dpp<0xB1>(m));  // lanes ^ 1, ^ 2, then 7 - lane
  m = max(m, dpp<0x4E>(m));
  if constexpr (NW == 8) m = max(m, dpp<0x141>(m));
  const int e = split_exp(__uint_as_float(m));
  return TileExps{__builtin_amdgcn_readlane(e, 0), __builtin_amdgcn_readlane(e, 32)};
}

// Offset (in fp16) of 16-byte chunk c (0..3) of row r of a part whose rows hold 32 values, a
// quarter of LDS's 256-byte bank period: 16 rows at any one column touch every bank once.
__device__ __forceinline__ int part_pos(int r, int c) { return r * 32 + ((c ^ ((r >> 2) & 3)) << 3); }

// c += a b, 32 x 32 x 16: lane l holds row (column) l % 32 of a (b) at k = 8 (l / 32) + 0..7;
// c[r] is row 8 (r / 4) + 4 (l / 32) + r % 4, column l % 32.
__device__ __forceinline__ f32x16 mfma_split(const Split8 &a, const Split8 &b, f32x16 c) {
  c = __builtin_amdgcn_mfma_f32_32x32x16_f16(a.lo, b.hi, c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_32x32x16_f16(a.hi, b.lo, c, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a.hi, b.hi, c, 0, 0, 0);
}

}  // namespace nva
