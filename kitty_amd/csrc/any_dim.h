// Device helpers of the attention kernels for head dimensions 64 and 256 (any_dim.hip: chunks, any_decode.hip: decode).
#pragma once
#include "decode_common.h"

namespace kitty {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef uint32_t uint4v __attribute__((ext_vector_type(4)));
typedef short short4v __attribute__((ext_vector_type(4)));

constexpr float kLog2e = 1.44269504088896340736f;
constexpr uint32_t kCodeMagic = 0x64006400u;   // fp16 1024 in both halves: 1024 + n is exact for n < 1024
constexpr float kProbScale = 32768.f;          // probabilities as matrix operands: see below
constexpr int kProbParts = 3;

__device__ __forceinline__ float4v mfma16(const uint32_t (&a)[4], const uint32_t (&b)[4], float4v c) {
  const uint4v av = {a[0], a[1], a[2], a[3]}, bv = {b[0], b[1], b[2], b[3]};
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, av), __builtin_bit_cast(half8, bv), c, 0, 0, 0);
}
// Transposing LDS read: lane i of a 16-lane block receives 16-bit piece i of the four 32-byte rows whose
// 8-byte quarters lanes 4r .. 4r+3 address; r0 = (row 0, row 1), r1 = (row 2, row 3).
__device__ __forceinline__ void lds_tr(const uint8_t* p, uint32_t& r0, uint32_t& r1) {
  const short4v v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((short4v __attribute__((address_space(3)))*)p);
  const uint2 u = __builtin_bit_cast(uint2, v);
  r0 = u.x;
  r1 = u.y;
}
__device__ __forceinline__ float4v mfma16(const uint32_t (&a)[4], const uint4& b, float4v c) {
  const uint32_t bb[4] = {b.x, b.y, b.z, b.w};
  return mfma16(a, bb, c);
}
__device__ __forceinline__ uint32_t low_halves(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x05040100u); }
__device__ __forceinline__ uint32_t high_halves(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x07060302u); }
// fp16(code) * scale + zero with BOTH operations rounded to fp16 (kitty_attention.py:162-165, 317-320 as
// eager torch and the Triton interpreter evaluate them), for two codes.  `c` holds 1024 + code * 2^SHIFT in each
// half (a code may stay at the bit where it lies): (1024 + code * 2^SHIFT) * 2^-SHIFT - 1024 * 2^-SHIFT is exact.
template <int SHIFT>
__device__ __forceinline__ uint32_t dequant_word(uint32_t c, uint32_t scale, uint32_t zero) {
#pragma clang fp contract(off)
  constexpr _Float16 k = (_Float16)(1.0f / (1 << SHIFT)), o = (_Float16)(1024.0f / (1 << SHIFT));
  const half2v x = __builtin_bit_cast(half2v, c);
  const half2v f = SHIFT == 0 ? x - half2v{o, o} : __builtin_elementwise_fma(x, half2v{k, k}, half2v{-o, -o});
  const half2v m = f * __builtin_bit_cast(half2v, scale);
  const half2v r = m + __builtin_bit_cast(half2v, zero);
  return __builtin_bit_cast(uint32_t, r);
}
// the value codes of d-tile u of a word: codes 0 .. 4 where they lie, the others after one shift for the three.  `magic`:
// kCodeMagic, in a register if masking and merging are to be one instruction
template <int U>
__device__ __forceinline__ uint32_t dequant_v(uint32_t x, uint32_t x10, uint32_t magic, uint32_t scale, uint32_t zero) {
  constexpr int k = 2 * (U < 5 ? U : U - 5);
  return dequant_word<k>(((U < 5 ? x : x10) & (0x00030003u << k)) | magic, scale, zero);
}
// infinities as the largest finite number: operands of the second and third part of a probability, which may be 0 or negative
// (the first part, times the infinity itself, has already made the sum infinite).  Costs the fp16 rows two instructions a
// word and packed tiles a look at their scales: 3 % at D = 64 and D = 256
__device__ __forceinline__ uint32_t finite_word(uint32_t x) {
  const half2v top = {(_Float16)65504.f, (_Float16)65504.f};
  const half2v v = __builtin_elementwise_min(__builtin_elementwise_max(__builtin_bit_cast(half2v, x), -top), top);
  return __builtin_bit_cast(uint32_t, v);
}
// maximum over lanes l, l^16, l^32, l^48
__device__ __forceinline__ float max_over_lane_groups(float v) {
  const unsigned b = __builtin_bit_cast(unsigned, v);
  const auto r = __builtin_amdgcn_permlane16_swap(b, b, false, false);
  const unsigned r0 = r[0], r1 = r[1];   // as scalars first: a bit_cast of r[1] itself reads element 0
  const float m = fmaxf(__builtin_bit_cast(float, r0), __builtin_bit_cast(float, r1));
  const unsigned c = __builtin_bit_cast(unsigned, m);
  const auto q = __builtin_amdgcn_permlane32_swap(c, c, false, false);
  const unsigned q0 = q[0], q1 = q[1];
  return fmaxf(__builtin_bit_cast(float, q0), __builtin_bit_cast(float, q1));
}

}  // namespace
}  // namespace kitty
