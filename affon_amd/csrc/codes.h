// Packed codes as bf16 MFMA operands, shared by the kernels that keep the
// codes exact in the matrix cores.
#pragma once

#include "lds_pipeline.h"

namespace affon {
namespace pipeline {

typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

// Bytes 0,1 (HIGH false) or 2,3 (HIGH true) of `bytes` read as FP8 E4M3 and
// times SCALE, converted to a bf16 pair. A byte holding n < 16 reads as
// n * 2^-9, exactly.
template <bool HIGH, int SCALE>
__device__ __forceinline__ uint32_t bf16_pair_fp8(uint32_t bytes) {
  return __builtin_bit_cast(uint32_t,
                            __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(bytes, static_cast<float>(SCALE), HIGH));
}

// Operands t = 0, 1 from 16 codes in k order (`words`: BITS / 2 words): codes
// 8t .. 8t+7 into operand t as bf16. 2/4-bit codes go through the FP8
// conversion and come out times SCALE * 2^-9 (SCALE 512: the integers); 8-bit
// codes through v_cvt_f32_ubyteN (exact in bf16 up to 255).
template <int BITS, int SCALE = 1>
__device__ __forceinline__ void codes_bf16(const uint32_t* words, u32x4_t* op) {
  if constexpr (BITS == 4) {  // word t = codes 8t .. 8t+7, code i in nibble i
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const uint32_t w = words[t];
      const uint32_t even = w & 0x0f0f0f0fu;         // byte j = code 2j
      const uint32_t odd = (w >> 4) & 0x0f0f0f0fu;   // byte j = code 2j+1
      const uint32_t lo = __builtin_amdgcn_perm(odd, even, 0x05010400u);  // codes 0,1,2,3
      const uint32_t hi = __builtin_amdgcn_perm(odd, even, 0x07030602u);  // codes 4,5,6,7
      op[t] = u32x4_t{bf16_pair_fp8<false, SCALE>(lo), bf16_pair_fp8<true, SCALE>(lo),
                      bf16_pair_fp8<false, SCALE>(hi), bf16_pair_fp8<true, SCALE>(hi)};
    }
  } else if constexpr (BITS == 2) {  // one word, code i at bits 2i
    const uint32_t w = words[0];
    uint32_t m[4];  // byte j of m[u] = code 4j + u
#pragma unroll
    for (int u = 0; u < 4; ++u) m[u] = (w >> (2 * u)) & 0x03030303u;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      // bytes 2t, 2t+1 of m[u] hold codes 8t+u and 8t+4+u.
      const uint32_t sel = (2 * t) | ((4 + 2 * t) << 8) | ((2 * t + 1) << 16) | ((5 + 2 * t) << 24);
      const uint32_t q01 = __builtin_amdgcn_perm(m[1], m[0], sel);  // codes 8t, 8t+1, 8t+4, 8t+5
      const uint32_t q23 = __builtin_amdgcn_perm(m[3], m[2], sel);  // codes 8t+2, 8t+3, 8t+6, 8t+7
      const uint32_t lo = __builtin_amdgcn_perm(q23, q01, 0x05040100u);  // codes 8t .. 8t+3
      const uint32_t hi = __builtin_amdgcn_perm(q23, q01, 0x07060302u);  // codes 8t+4 .. 8t+7
      op[t] = u32x4_t{bf16_pair_fp8<false, SCALE>(lo), bf16_pair_fp8<true, SCALE>(lo),
                      bf16_pair_fp8<false, SCALE>(hi), bf16_pair_fp8<true, SCALE>(hi)};
    }
  } else {  // words 2t, 2t+1 = codes 8t .. 8t+7, one byte each
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      uint32_t pairs[4];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const uint32_t v = opaque(words[2 * t + i]);
        pairs[2 * i] = pack_bf16(static_cast<float>(v & 0xffu), static_cast<float>((v >> 8) & 0xffu));
        pairs[2 * i + 1] = pack_bf16(static_cast<float>((v >> 16) & 0xffu), static_cast<float>(v >> 24));
      }
      op[t] = u32x4_t{pairs[0], pairs[1], pairs[2], pairs[3]};
    }
  }
}

}  // namespace pipeline
}  // namespace affon
