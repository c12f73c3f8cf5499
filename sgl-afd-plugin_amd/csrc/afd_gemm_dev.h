// Device pieces that the grouped GEMMs share, large tiles (afd_gemm_mx.hip, afd_gemm_fp8.hip,
// afd_gemm_a16.hip) and few rows (afd_gemm_rows.hip): a token's result is the same bits from either,
// so what computes it stands here once.
#pragma once

#include "afd_common.h"

namespace afd {

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

// The scaled MFMA with a 4-dword (e2m1) first operand. The clang builtin takes 8 dwords for every
// operand format; the intrinsic's operand type follows the format, and e2m1 needs only 4.
// The kernels pass the e2m1 weights as the first operand and the e4m3 activations as the
// second (D = W X^T), so a lane's accumulators belong to one activation row.
extern "C" __device__ v16f mfma_scale_f4_f8(v4i a, v8i b, v16f c, int cbsz, int blgp,
                                            int opsel_a, int scale_a, int opsel_b, int scale_b)
    __asm("llvm.amdgcn.mfma.scale.f32.32x32x64.f8f6f4.v4i32.v8i32");

// the 8 e2m1 codes of dword d (element 2i in the low nibble of byte i) times 2^(code - 127),
// as the 8 bf16 of an MFMA operand (element i in half i % 2 of dword i / 2). The instruction
// takes the scale's exponent field as the UE8M0 code, so `scale` is the code shifted into it.
__device__ __forceinline__ v8bf expand_fp4(uint32_t d, float scale) {
  v4i r;
  r[0] = __builtin_bit_cast(int, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(d, scale, 0));
  r[1] = __builtin_bit_cast(int, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(d, scale, 1));
  r[2] = __builtin_bit_cast(int, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(d, scale, 2));
  r[3] = __builtin_bit_cast(int, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(d, scale, 3));
  return __builtin_bit_cast(v8bf, r);
}

// the 8 e4m3 codes of dwords d0, d1 (element i in byte i % 4 of dword i / 4) as the 8 bf16 of
// an MFMA operand, exactly (scale 2^0)
__device__ __forceinline__ v8bf expand_fp8(uint32_t d0, uint32_t d1) {
  v4i r;
  r[0] = __builtin_bit_cast(int, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(d0, 1.0f, false));
  r[1] = __builtin_bit_cast(int, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(d0, 1.0f, true));
  r[2] = __builtin_bit_cast(int, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(d1, 1.0f, false));
  r[3] = __builtin_bit_cast(int, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(d1, 1.0f, true));
  return __builtin_bit_cast(v8bf, r);
}

// A uniform read of data the kernel never writes (the FP8 block scales), through the scalar
// cache: read through a generic pointer the compiler has to assume a store of the kernel may
// alias it and issues a vector load, whose wait then drains the copies in flight.
__device__ __forceinline__ float load_uniform(const float* p) {
  return *(const __attribute__((address_space(4))) float*)p;
}

// Epilogues: a lane holds, of one activation row's 32-column tile, columns 8 q4 + 4 lk .. + 3
// (q4 = 0..3, accumulators 4 q4 .. 4 q4 + 3; lk = lane / 32).
// e4m3 codes d[q4] of those columns -> the 16 of columns 16 lk .. 16 lk + 15: lane half 0 takes
// columns 0-15 (its d0, d1 and the partner's), half 1 columns 16-31 (the partner's d2, d3 and its own).
__device__ __forceinline__ v4i e4m3_chunk(const uint32_t (&d)[4], int lk) {
  const uint32_t p0 = swap_halves(d[2], d[0], lk);
  const uint32_t p1 = swap_halves(d[3], d[1], lk);
  v4i chunk;
  chunk[0] = static_cast<int>(lk ? p0 : d[0]);
  chunk[1] = static_cast<int>(lk ? d[2] : p0);
  chunk[2] = static_cast<int>(lk ? p1 : d[1]);
  chunk[3] = static_cast<int>(lk ? d[3] : p1);
  return chunk;
}
// the 16 values h -> bf16, as whole 16-byte chunks 2 pr + lk (pr = 0, 1) in column order.
// v_permlane32_swap trades the first operand of lanes 32-63 for the second operand of lanes 0-31:
// afterwards lane half 0 holds its own columns of chunk 2 pr and its partner's, lane half 1 its
// partner's columns of chunk 2 pr + 1 and its own, with no select.
template <typename H>
__device__ __forceinline__ void bf16_chunks(const H& h, v4i (&chunk)[2]) {
  uint32_t hb[4][2];
#pragma unroll
  for (int q4 = 0; q4 < 4; ++q4) {
    hb[q4][0] = pk_bf16(h[4 * q4], h[4 * q4 + 1]);
    hb[q4][1] = pk_bf16(h[4 * q4 + 2], h[4 * q4 + 3]);
  }
#pragma unroll
  for (int pr = 0; pr < 2; ++pr) {
    const auto d0 = __builtin_amdgcn_permlane32_swap(hb[2 * pr][0], hb[2 * pr + 1][0], false, false);
    const auto d1 = __builtin_amdgcn_permlane32_swap(hb[2 * pr][1], hb[2 * pr + 1][1], false, false);
    chunk[pr] = v4i{static_cast<int>(d0[0]), static_cast<int>(d1[0]), static_cast<int>(d0[1]),
                    static_cast<int>(d1[1])};
  }
}

}  // namespace afd
