// mc_ops.h -- matrix-core building blocks shared by the chunked scan kernels
// (naju_scan_mc.hip, naju_scan_map.hip). Internal to the library.
#ifndef NAJU_MC_OPS_H
#define NAJU_MC_OPS_H

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "scan_internal.h"

namespace naju_detail {
namespace {

typedef float f4_t __attribute__((ext_vector_type(4)));

// D += A B for one 16x16x4 float32 tile: lane l supplies A[l%16][l/16] and
// B[l/16][l%16] and holds D[4(l/16) + r][l%16] in value r.
__device__ __forceinline__ f4_t mma(float a, float b, f4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Four values that are exact in the 2-byte stream type TT (B and C as
// staged: converted from TT, zero rows included) packed as TT pairs.
template <typename TT>
__device__ __forceinline__ void pack4(const float (&x)[4], uint32_t (&w)[2]) {
  if constexpr (__is_same(TT, bf16_t)) {
    // the upper halves of the float bits (exact: the low halves are zero)
#pragma unroll
    for (int k = 0; k < 2; ++k)
      w[k] = __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, x[2 * k + 1]), __builtin_bit_cast(uint32_t, x[2 * k]),
                                   0x07060302u);
  } else {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      typedef _Float16 h2 __attribute__((ext_vector_type(2)));
      const h2 h = {(_Float16)x[2 * k], (_Float16)x[2 * k + 1]};
      w[k] = __builtin_bit_cast(uint32_t, h);
    }
  }
}

// D += A B with K = 32 on the 16-bit matrix-core path, for operands exact in
// TT (bf16 or f16): lane l supplies A[l%16][k] and B[k][l%16] for its eight
// k of the product, a0 and b0 (then a1 and b1) packed by pack4 from the same
// four k each, so that any assignment of the lane's values to k pairs A and
// B alike. The products are exact in float32 and only the accumulation
// rounds, as on the float32 path, at one instruction in place of eight.
template <typename TT>
__device__ __forceinline__ f4_t mma_k32(const uint32_t (&a0)[2], const uint32_t (&a1)[2], const uint32_t (&b0)[2],
                                        const uint32_t (&b1)[2], f4_t c) {
  typedef uint32_t u4 __attribute__((ext_vector_type(4)));
  const u4 av = {a0[0], a0[1], a1[0], a1[1]}, bv = {b0[0], b0[1], b1[0], b1[1]};
  if constexpr (__is_same(TT, bf16_t)) {
    typedef __bf16 v8 __attribute__((ext_vector_type(8)));
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8, av), __builtin_bit_cast(v8, bv), c, 0, 0,
                                                   0);
  } else {
    typedef _Float16 v8 __attribute__((ext_vector_type(8)));
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8, av), __builtin_bit_cast(v8, bv), c, 0, 0, 0);
  }
}

// x[k] = hi + mid + lo exactly, in three bf16 parts packed in pairs like
// pack4: hi keeps the top 8 significant bits of x (truncated), mid the next
// 8 of the remainder and lo the at most 8 left, so each part is exact in
// bf16 and each difference exact in float32. (x = +-inf or nan gives nan
// parts; the states and adjoints split here are finite for finite inputs.)
__device__ __forceinline__ void split4_bf16(const float (&x)[4], uint32_t (&h)[2], uint32_t (&md)[2],
                                            uint32_t (&lo)[2]) {
  uint32_t hb[4], mb[4], lb[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    // x as rounded: the subtraction below must not be fused with the
    // product that formed x (the parts would then sum to the unrounded
    // product, differently wherever the compiler chose to fuse)
    float xk = x[k];
    asm volatile("" : "+v"(xk));
    hb[k] = __builtin_bit_cast(uint32_t, xk) & 0xffff0000u;
    const float r = xk - __builtin_bit_cast(float, hb[k]);
    mb[k] = __builtin_bit_cast(uint32_t, r) & 0xffff0000u;
    lb[k] = __builtin_bit_cast(uint32_t, r - __builtin_bit_cast(float, mb[k]));
  }
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    h[k] = __builtin_amdgcn_perm(hb[2 * k + 1], hb[2 * k], 0x07060302u);
    md[k] = __builtin_amdgcn_perm(mb[2 * k + 1], mb[2 * k], 0x07060302u);
    lo[k] = __builtin_amdgcn_perm(lb[2 * k + 1], lb[2 * k], 0x07060302u);
  }
}

// D += A B over the lane's four k (the k-steps of four 16x16x4 float32
// products) with A exact in bf16 (a: packed by pack4) and B float32 given by
// its split4_bf16 parts: hi and mid in one K = 32 product, lo (with zeros)
// in a second. Each product is exact; the result matches the float32 path
// up to the accumulation's rounding, at two instructions in place of four.
// (The K = 16 form, v_mfma_f32_16x16x16_bf16, took the lo part at first and
// gave run-to-run different results in this position on gfx950 with the
// compiler's default scheduling; the K = 32 form is used throughout.)
__device__ __forceinline__ f4_t mma_x3(const uint32_t (&a)[2], const uint32_t (&h)[2], const uint32_t (&md)[2],
                                       const uint32_t (&lo)[2], f4_t c) {
  c = mma_k32<bf16_t>(a, a, h, md, c);
  const uint32_t z[2] = {0u, 0u};
  return mma_k32<bf16_t>(a, z, lo, z, c);
}

}  // namespace
}  // namespace naju_detail

#endif  // NAJU_MC_OPS_H
