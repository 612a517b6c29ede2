// Building blocks the matrix-core distance kernels share: float32 products on the bfloat16
// matrix pipe, integer argmin keys, the norm of a staged row.
#pragma once
#include <hip/hip_runtime.h>

#include "mfma_traits.h"

namespace kmhip {

// Squared norm of one centroid row, j ascending, multiply and add rounded separately:
// the value row_norms would store (kmeans_labels.h:187-199). The fused
// kernels call it when they are given no norm buffer, which spares the Lloyd loop a launch.
template <typename T>
__device__ __forceinline__ T row_sqnorm(const T *__restrict__ x, int d) {
#pragma clang fp contract(off)
  T acc = 0;
  int j = 0;
  for (; j + 8 <= d; j += 8) {  // (eight loads under way at a time)
    T v[8];
#pragma unroll
    for (int e = 0; e < 8; e++) v[e] = x[j + e];
#pragma unroll
    for (int e = 0; e < 8; e++) acc = acc + v[e] * v[e];
  }
  for (; j < d; j++) {
    const T v = x[j];
    acc = acc + v * v;
  }
  return acc;
}

// Three-input unsigned minimum as ONE instruction. Written as inline assembly
// because the optimiser otherwise re-associates a chain of them into pairs of
// two-input minima and spends 12 instead of 8 instructions on 16 keys.
__device__ __forceinline__ unsigned umin3(unsigned a, unsigned b, unsigned c) {
  unsigned r;
  asm("v_min3_u32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}
// The middle one of three, likewise.
__device__ __forceinline__ unsigned umed3(unsigned a, unsigned b, unsigned c) {
  unsigned r;
  asm("v_med3_u32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}
// The smallest of the 16 keys of a tile; `second` becomes the second smallest of them, the running
// minimum `best` and the running second minimum. Triples give their two smallest with two
// instructions, so the second minimum costs 12 instructions on top of the 8 of the minimum alone.
__device__ __forceinline__ unsigned two_smallest_keys(const unsigned (&key)[16], unsigned best, unsigned &second) {
  unsigned lo[5], mid[5];
#pragma unroll
  for (int i = 0; i < 5; i++) {
    lo[i] = umin3(key[3 * i], key[3 * i + 1], key[3 * i + 2]);
    mid[i] = umed3(key[3 * i], key[3 * i + 1], key[3 * i + 2]);
  }
  const unsigned a = umin3(lo[0], lo[1], lo[2]), b = umin3(lo[3], lo[4], key[15]);
  const unsigned am = umed3(lo[0], lo[1], lo[2]), bm = umed3(lo[3], lo[4], key[15]);
  second = umin3(umin3(mid[0], mid[1], mid[2]), umin3(mid[3], mid[4], am), umin3(bm, umed3(a, b, best), second));
  return min(a, b);
}
// Whether two distances of a row, compared at 16 ulp, lie so close that the bfloat16 products and the
// float32 instructions may order them differently. settle_margin() bounds the rounding of both forms
// relative to xx + cc, and a centroid at a distance `second` has a norm of at most 2 xx + 2 second; two
// buckets of 16 ulp come on top. (A row whose norm is infinite is said to be tied as well, a NaN never is.)
struct TieBound {
  float of_norm, of_second;  // tied when of_second * second - best <= of_norm * xx; of_norm -infinity: never
};
__device__ __forceinline__ bool near_tie(float best, float second, float xx, TieBound b) {
  return fmaf(b.of_second, second, -best) <= b.of_norm * xx;
}
// Each form's d roundings are 0.3 ulp of a partial sum of at most xx + cc, so the difference of two
// distances in two forms has an rms of about 0.3 sqrt(d) eps (xx + cc) (measured without the norms' own
// error, which both share: 0.4 to 1.3 eps a distance at 3 to 64 features). Five times that and more: the
// bound on cc makes xx + cc half again as large as it is, and a constant is there for the roundings that
// do not depend on d.
static inline TieBound settle_margin(int d, bool settle) {
  const float m = (3.0f + sqrtf((float)d)) * 1.1920929e-7f;
  return settle ? TieBound{3.0f * m, 1.0f - 2.0f * m - 3.9e-6f} : TieBound{-__builtin_huge_valf(), 1.0f};
}
// the floats whose upper halves are the low and the high half of a packed pair
__device__ __forceinline__ float bf16_low(unsigned p) { return __uint_as_float(p << 16); }
__device__ __forceinline__ float bf16_high(unsigned p) { return __uint_as_float(p & 0xFFFF0000u); }
// centroid row of accumulator v (runtime v) of the 32x32 float tile
__device__ __forceinline__ int key_row(unsigned v, int g) {
  return (int)((v >> 2) * 8 + (unsigned)g * 4 + (v & 3));
}

// float32 products on the bfloat16 matrix pipe. A float is the exact sum of three
// bfloat16 values (8 significant bits each: the float rounded to bfloat16, the remainder
// rounded to bfloat16, and what is left of it, which has at most 8 significant bits; every
// subtraction is exact), so x * c is the exact sum of the nine products of their parts, each
// of which a float holds exactly (16 bits). v_mfma_f32_32x32x16_bf16 adds such products
// into float accumulators: the result carries float rounding of the running sum only, as
// the float32 instruction's does. (It adds the eight products of lane group 0 to the accumulator, then
// the eight of group 1; either time all nine terms are aligned to the largest, with a few bits beyond a
// float's, and the sum is rounded. Checked on hardware.) On gfx950 the instruction runs at 16 times the float32
// rate (nine of them per 16 features take 288 cycles where eight v_mfma_f32_32x32x2_f32
// take 512). The parts are rounded to nearest (v_cvt_pk_bf16_f32), not cut off: the
// remainders then carry either sign, and the products the 6-product form leaves out cancel
// on average instead of adding up to a bias of the distances (cut-off parts all have the
// sign of the float they come from; measured on 6000 x 200 blobs far from the origin, the
// sum of the minimum distances came out 1.6e-5 too large).
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef unsigned uintx4 __attribute__((ext_vector_type(4)));
// two floats rounded to bfloat16 in one register: a in bits 0-15, b in bits 16-31
__device__ __forceinline__ unsigned cvt_pk_bf16(float a, float b) {
  const floatx2 f = {a, b};
  return __builtin_bit_cast(unsigned, __builtin_convertvector(f, bf16x2));
}
// The three parts of two floats, each pair packed like cvt_pk_bf16 packs it: 11 vector
// instructions (three conversions, four unpackings, four subtractions).
struct Bf16x3Pair {
  unsigned h, m, l;
};
__device__ __forceinline__ Bf16x3Pair split_pair_bf16x3(float a, float b) {
  Bf16x3Pair p;
  p.h = cvt_pk_bf16(a, b);
  const float ra = a - __uint_as_float(p.h << 16), rb = b - __uint_as_float(p.h & 0xFFFF0000u);
  p.m = cvt_pk_bf16(ra, rb);
  p.l = cvt_pk_bf16(ra - __uint_as_float(p.m << 16), rb - __uint_as_float(p.m & 0xFFFF0000u));
  return p;
}
// A squared norm as an exact sum of three bfloat16 values with their bits in the low halves of
// h, m and l. Cut off instead of rounded: the largest floats would round to an infinity, and all
// parts have the norm's sign here anyway. Infinities and NaN stay whole in the first part.
struct Bf16x3 {
  unsigned h, m, l;
};
__device__ __forceinline__ Bf16x3 split_norm_bf16x3(float v) {
  Bf16x3 p;
  const unsigned u = __float_as_uint(v);
  p.h = u >> 16;
  const float r = v - __uint_as_float(u & 0xFFFF0000u);
  const unsigned ur = __float_as_uint(r);
  p.m = ur >> 16;
  p.l = __float_as_uint(r - __uint_as_float(ur & 0xFFFF0000u)) >> 16;
  if ((u & 0x7F800000u) == 0x7F800000u) {
    if ((u & 0xFFFFu) != 0) p.h |= 0x40u;  // (a NaN whose payload lies in the low half)
    p.m = p.l = 0;
  }
  return p;
}
__device__ __forceinline__ floatx16 mma_bf16(uintx4 a, uintx4 b, floatx16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

}  // namespace kmhip
