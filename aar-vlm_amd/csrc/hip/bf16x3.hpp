// fp32 products on the bf16 matrix cores, without giving up fp32 precision.
//
// x = hi + mid + lo exactly, each a bf16: hi = bf16(x) rounded to nearest
// leaves a remainder of at most 16 significant bits, mid = bf16 of it leaves
// at most 8, which lo holds.  A product a b then is the sum of nine bf16
// products, each exact in fp32; the three smallest (mid lo, lo mid, lo lo,
// together at most about 2^-25 |a b| and of either sign) are left out, and the
// other six run on v_mfma_f32_32x32x16_bf16, the hi hi products into one fp32
// accumulator and the five smaller ones into another, added at the end.  The
// matrix unit sums 16 products per instruction before it rounds, so a chain
// over K rounds K / 16 times where v_mfma_f32_32x32x2f32 rounds K times.
//
// Measured on MI355X against fp64 sums (32 x 32 outputs x 16 blocks; relative
// 2-norm error, fp32 instruction -> six products): standard normal operands,
// K = 16 7.4e-8 -> 3.2e-8, 64 1.45e-7 -> 5.0e-8, 384 3.5e-7 -> 1.1e-7, 1024
// 5.8e-7 -> 1.9e-7, 4096 1.15e-6 -> 3.9e-7, 16384 2.3e-6 -> 8.1e-7; uniform
// [0, 1) 4096 8.4e-7 -> 3.0e-7; magnitudes spread over 2^+-10 4096 9.2e-7 ->
// 4.1e-7; mean error (256 blocks) below 1e-9 of the outputs' scale.
// (Truncating instead of rounding the parts biases the sums: 1.05e-5 on the
// uniform ones.)  The bf16 unit reaches 1976 TFLOP/s where the fp32 one
// reaches 139: 329 TFLOP/s of fp32 products.
//
// The matrix op takes subnormal bf16 operands and sums subnormal results as
// they are (measured), so the split is exact wherever an element's last bit
// is at least 2^-133, bf16's smallest step: for all elements from 2^-110 up.
// What the split does not cover is handed to the fp32 instruction by the
// callers: sums that the part a smaller element leaves over reaches
// (split_loss_floor), infinities, and magnitudes that round to infinity or whose
// products' sums might (split_overflows).  NaN operands give NaN in the same
// outputs either way.
//
// Operands in several bf16 parts are a published method (G. Henry, P. Tang, A.
// Heinecke, "Leveraging the bfloat16 Artificial Intelligence Datatype For
// Higher-Precision Computations", ARITH 2019).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "common.hpp"

namespace aar {

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kSplitProducts = 6;
// Product p multiplies part kSplitA[p] of the left operand with part
// kSplitB[p] of the right one (0 hi, 1 mid, 2 lo), smallest first.
__device__ constexpr int kSplitA[kSplitProducts] = {2, 0, 1, 1, 0, 0};
__device__ constexpr int kSplitB[kSplitProducts] = {0, 2, 1, 0, 1, 0};

// Two floats to a pair of bf16 (v_cvt_pk_bf16_f32, round to nearest even).
__device__ __forceinline__ uint32_t bf16_pair(float a, float b) {
  const f32x2 v = {a, b};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}

// The three bf16 parts of (a, b) as pairs: a in the low halves.  `rem` collects
// the bits of what the lowest parts are rounded from: every element is held
// exactly as long as none of its low 16 bits is set.  (An opaque three-way or,
// v_bitop3_b32: plain ors are reassociated over the whole tile, which kept 12
// more registers alive in the 256x128 GEMM tile.)
__device__ __forceinline__ void bf16_split_pair(float a, float b, uint32_t (&p)[3], uint32_t& rem) {
  p[0] = bf16_pair(a, b);
  a -= __uint_as_float(p[0] << 16);
  b -= __uint_as_float(p[0] & 0xffff0000u);
  p[1] = bf16_pair(a, b);
  a -= __uint_as_float(p[1] << 16);
  b -= __uint_as_float(p[1] & 0xffff0000u);
#if defined(__HIP_DEVICE_COMPILE__)
  rem = __builtin_amdgcn_bitop3_b32(rem, __float_as_uint(a), __float_as_uint(b), 0xfe);
#endif
  p[2] = bf16_pair(a, b);
}
constexpr uint32_t kSplitRemBits = 0xffffu;

// D = A B + C for 32x32 tiles over 16 k: lane (r = lane % 32, h = lane / 32)
// holds A[r][8h .. 8h+7] and B[8h .. 8h+7][r]; C/D as the fp32 32x32
// instructions (register i: row 8 (i / 4) + 4 h + i % 4, column r).
__device__ __forceinline__ f32x16 mfma_bf16(const u32x4& a, const u32x4& b, const f32x16& c) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0,
                                                 0);
#else
  return c;
#endif
}

// Keeps the compiler's scheduler from moving instructions across this point.
__device__ __forceinline__ void sched_fence() {
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_sched_barrier(0);
#endif
}

// This wave's LDS accesses are complete and every wave is here; global loads
// in flight stay in flight (a workgroup fence would wait for them).
__device__ __forceinline__ void lds_barrier() {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
#endif
}

// Sums of fewer than 2^26 products of magnitudes up to this stay finite.
constexpr float kSplitPlain = 1.1258999068426240e15f;  // 2^50
// Whether a sum of n products of magnitudes up to ma and mb might leave fp32's
// range where the exact one does not (2^126 leaves room for the parts' rounding).
__device__ __forceinline__ bool split_overflows(float ma, float mb, float n) {
  const float top = 8.5070591730234616e37f;  // 2^126
  return !(ma <= top && mb <= top && ma * mb * n <= top);
}
// The magnitude from which on such a sum does not feel what elements below 2^-110
// leave over: at most 2^-134 each, so n 2^-134 (ma + mb) in all,
// which is less than 2^-24 of it.
__device__ __forceinline__ float split_loss_floor(float ma, float mb, float n) {
  return n * 7.7037197775489434e-34f * (ma + mb);  // 2^-110
}

}  // namespace aar
