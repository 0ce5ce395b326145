// Device helpers of the split kernels: fp32 products as three fp16 products
// (conv_split.hip describes the split and its range).
#pragma once

#include "internal.h"

namespace rvc {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 halfx2 __attribute__((ext_vector_type(2)));
typedef _Float16 halfx8 __attribute__((ext_vector_type(8)));

constexpr float kScaleX = 64.f;                 // the inputs' usual scale
constexpr float kXMin = 0x1p-6f, kXMax = 960.f;  // the magnitudes it serves
// whether a largest magnitude m, scaled, lies where the two parts hold what the
// sums need: 0, or from where fp16's subnormals cost less than 2^-24 of it up to
// where fp16 ends.  Infinities and NaN do not.
__device__ __forceinline__ bool split_holds(float m) {
  return m == 0.f || (m >= kXMin * kScaleX && m <= kXMax * kScaleX);
}

// the OR over the waves of a workgroup of its threads' low two bits; one barrier,
// slot: NW words that no wave still reads from an earlier call
template <int NW>
__device__ __forceinline__ unsigned block_or(unsigned bits, unsigned* slot) {
  const unsigned v = (__any(bits & 1u) ? 1u : 0u) | (__any(bits & 2u) ? 2u : 0u);
  if ((threadIdx.x & 63) == 0) slot[threadIdx.x >> 6] = v;
  __syncthreads();
  unsigned f = 0;
#pragma unroll
  for (int w = 0; w < NW; ++w) f |= slot[w];
  return (unsigned)__builtin_amdgcn_readfirstlane((int)f);
}
// the largest m over a workgroup; two barriers
template <int NW>
__device__ __forceinline__ float block_max(float m, float* slot) {
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) m = fmaxf(m, __shfl_xor(m, d));
  if ((threadIdx.x & 63) == 0) slot[threadIdx.x >> 6] = m;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < NW; ++w) m = fmaxf(m, slot[w]);
  __syncthreads();
  return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, m)));
}
// largest magnitudes m[i]: bit 0 where one does not lie in the split's range,
// bit 1 where one does and is not 0; top: the largest finite one
template <int N>
__device__ __forceinline__ unsigned range_bits(const float (&m)[N], float scale, float& top) {
  unsigned f = 0;
  top = 0.f;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const float v = m[i] * scale;
    f |= split_holds(v) ? (v > 0.f ? 2u : 0u) : 1u;
    top = m[i] < __builtin_inff() ? fmaxf(top, m[i]) : top;
  }
  return f;
}

// one product of two operands: 8 channels of a row and of a column per lane
template <bool BF>
__device__ __forceinline__ floatx16 mma16(uint4 w, uint4 x, floatx16 c) {
  if constexpr (BF)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, w), __builtin_bit_cast(bf16x8, x), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(halfx8, w), __builtin_bit_cast(halfx8, x), c, 0, 0, 0);
}
__device__ __forceinline__ uint4 buf_load16(__amdgpu_buffer_rsrc_t r, unsigned voff, unsigned soff) {
  return __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
}
__device__ __forceinline__ float buf_load4(__amdgpu_buffer_rsrc_t r, unsigned voff, unsigned soff) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0));
}
// leaky ReLU for slopes in [0, 1]: max(v, v slope), as one instruction each
// (fmaxf quiets its operands first).  Never straight into or out of an MFMA: the
// compiler does not see the asm as the VALU instruction it is, and leaves out the
// wait states between the two.
__device__ __forceinline__ float leaky(float v, float slope) {
  float r;
  asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(v), "v"(v * slope));
  return r;
}
// the same for operands of an MFMA
__device__ __forceinline__ float leaky_mma(float v, float slope) { return v < 0.f ? v * slope : v; }
// max(m, |a|, |b|)
__device__ __forceinline__ float max3_abs(float m, float a, float b) {
  asm("v_max3_f32 %0, %0, abs(%1), abs(%2)" : "+v"(m) : "v"(a), "v"(b));
  return m;
}
// two floats -> two bf16 (round to nearest even), lo in the low half
__device__ __forceinline__ unsigned pk_bf16(float lo, float hi) {
  return __builtin_bit_cast(unsigned, __builtin_convertvector(floatx2{lo, hi}, bf16x2));
}
// the two parts of a pair of floats
__device__ __forceinline__ void split2(float a, float b, unsigned& h, unsigned& l) {
  const halfx2 hv = __builtin_convertvector(floatx2{a, b}, halfx2);
  const floatx2 r = {a - (float)hv.x, b - (float)hv.y};
  h = __builtin_bit_cast(unsigned, hv);
  l = __builtin_bit_cast(unsigned, __builtin_convertvector(r, halfx2));
}
// the power of two that moves m (finite, above 0) into [2^14, 2^15), within the
// normal floats on both sides of 1: what lies up to 2^14 below it is held too
__device__ __forceinline__ float pow2_scale(float m) {
  const int e = (int)(__builtin_bit_cast(unsigned, m) >> 23) - 127;
  return __builtin_bit_cast(float, (unsigned)(min(max(14 - e, -126), 126) + 127) << 23);
}
// eight channels of one column to LDS: their fp16 parts of v * sx at dst and
// dst + part, largest magnitude to vmax; or (BF) their bf16 at dst
template <bool BF>
__device__ __forceinline__ void stage_unit(float (&v)[8], float sx, float& vmax, uint4* dst, int part) {
  uint4 h, l;
  if constexpr (BF) {
    *dst = make_uint4(pk_bf16(v[0], v[1]), pk_bf16(v[2], v[3]), pk_bf16(v[4], v[5]), pk_bf16(v[6], v[7]));
  } else {
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] *= sx;
#pragma unroll
    for (int j = 0; j < 8; j += 2) vmax = max3_abs(vmax, v[j], v[j + 1]);
    split2(v[0], v[1], h.x, l.x);
    split2(v[2], v[3], h.y, l.y);
    split2(v[4], v[5], h.z, l.z);
    split2(v[6], v[7], h.w, l.w);
    dst[0] = h;
    dst[part] = l;
  }
}
// A wave's 32 TM x 32 TN sums on the fp32 matrix cores, from where the operands
// lie in fp32, C channels (a multiple of 8) by K taps: the sums that a split
// cannot form.  w(A, k, c) fills A[m] with row 32 m + lane % 32's weight of
// channel c + lane / 32 and tap k, x(B, k, c) B[n] with column 32 n + lane % 32's
// input.
template <int TM, int TN, class W, class X>
__device__ __forceinline__ void fp32_sums(floatx16 (&acc)[TM][TN], int C, int K, W w, X x) {
#pragma unroll
  for (int m = 0; m < TM; ++m)
#pragma unroll
    for (int n = 0; n < TN; ++n)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[m][n][r] = 0.f;
#pragma unroll 1
  for (int k = 0; k < K; ++k)
#pragma unroll 1
    for (int c = 0; c < C; c += 8) {
      float A[4][TM], B[4][TN];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        w(A[u], k, c + 2 * u);
        x(B[u], k, c + 2 * u);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int m = 0; m < TM; ++m)
#pragma unroll
          for (int n = 0; n < TN; ++n)
            acc[m][n] = __builtin_amdgcn_mfma_f32_32x32x2f32(A[u][m], B[u][n], acc[m][n], 0, 0, 0);
    }
}
template <int TM>
__device__ __forceinline__ void swap_sets(uint4 (&a)[2][TM], uint4 (&b)[2][TM]) {
#pragma unroll
  for (int m = 0; m < TM; ++m) {
    uint4 t = a[0][m];
    a[0][m] = a[1][m];
    a[1][m] = t;
    t = b[0][m];
    b[0][m] = b[1][m];
    b[1][m] = t;
  }
}
// The order of one tap: products, then the loads whose registers they have
// freed, so that a load has the rest of the tap to land (C = 256, 10 000
// columns: six launches 0.73 -> 0.65 ms).  The weights run two taps ahead in two
// register sets: with few workgroups a CU nothing else hides their way from L2
// (C = 256 at 1000 columns 0.385 -> 0.24 ms, at 10 000 0.605 -> 0.51).
template <bool BF, int TM, int TN>
__device__ __forceinline__ void sched_tap() {
  if constexpr (BF) {
    __builtin_amdgcn_sched_group_barrier(0x008, TM * TN, 0);
    __builtin_amdgcn_sched_group_barrier(0x020, TM, 0);
    __builtin_amdgcn_sched_group_barrier(0x100, TN, 0);
    __builtin_amdgcn_sched_group_barrier(0x008, TM * TN, 0);
    __builtin_amdgcn_sched_group_barrier(0x020, TM, 0);
    __builtin_amdgcn_sched_group_barrier(0x100, TN, 0);
  } else {
    __builtin_amdgcn_sched_group_barrier(0x008, TM * TN, 0);
    __builtin_amdgcn_sched_group_barrier(0x020, TM, 0);
    __builtin_amdgcn_sched_group_barrier(0x008, TM * TN, 0);
    __builtin_amdgcn_sched_group_barrier(0x100, TN, 0);
    __builtin_amdgcn_sched_group_barrier(0x008, TM * TN, 0);
    __builtin_amdgcn_sched_group_barrier(0x020, TM, 0);
    __builtin_amdgcn_sched_group_barrier(0x100, TN, 0);
  }
}

}  // namespace rvc
