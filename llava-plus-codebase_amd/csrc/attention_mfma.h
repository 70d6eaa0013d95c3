// MFMA / LDS-layout helpers shared by the flash forward kernels (attention.hip) and the flash backward kernels (attn_bwd.hip).
#pragma once
#include "common.h"

namespace lmx {

template <typename T> struct Mfma32;
template <> struct Mfma32<bf16_t> {
    static __device__ __forceinline__ f32x16 run(const uint4& a, const uint4& b, const f32x16& c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_v, a), __builtin_bit_cast(bf16x8_v, b), c, 0, 0, 0);
    }
};
template <> struct Mfma32<f16_t> {
    static __device__ __forceinline__ f32x16 run(const uint4& a, const uint4& b, const f32x16& c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_v, a), __builtin_bit_cast(f16x8_v, b), c, 0, 0, 0);
    }
};

constexpr int FA_KT = 64;      // keys per tile (flash_body with 64 rows of 128: 32)
// log2 units: skip the O rescale until a row max grows by more.  The probability that stands at the maximum is 1, which 16 bits hold exactly, others are rounded: a larger threshold leaves
// the maximum behind in more rows.  1087 causal rows in bf16, relative error against 64 bits at 8 | 4 | 2 | 1 | 0: 2.039e-3 | 2.038e-3 | 2.003e-3 | 1.975e-3 | 1.968e-3, time 22.0 | 22.4 | 22.9 | 23.6 | 23.7 us
constexpr float FA_DEFER = 2.f;

// K tile in LDS: [keys][D] 16-bit; 16-byte chunks XOR-swizzled so a ds_read_b128 lane group (16 distinct rows,
// same logical chunk) touches 16 distinct 16-byte slots of the 256-byte bank row.
template <int D> __device__ __forceinline__ int k_lds_off(int row, int chunk) {
    if constexpr (D == 128) return row * 256 + (((chunk ^ row) & 15) << 4);
    else return row * 128 + (((chunk ^ (row >> 1)) & 7) << 4);
}
// Key order inside a 32-key block.  The 32x32 accumulator of Sᵀ = K Qᵀ holds tile row (r & 3) + 8 (r >> 2) + 4 hi in register r of lane half hi, and the
// P·V step (kb, s2) takes registers 8 s2 .. + 7 as its 8 k-values: with K fed in natural order those are keys {4 hi .. + 3} and {8 + 4 hi .. + 3} (+ 16 s2),
// i.e. the Vᵀ operand needs TWO 8-byte LDS reads, 2-way bank-conflicted (1.46 M conflict cycles per launch in the counters).  Feeding K row pi(l31) =
// l31 with bits 2 and 3 swapped as tile row l31 makes them the 8 CONSECUTIVE keys 16 s2 + 8 hi .. + 7: one conflict-free 16-byte read.  (pi maps each
// 16-lane service group of ds_read_b128 onto itself, so the K fragment reads stay conflict-free.)
__device__ __forceinline__ int fa_key_perm(int l31) { return (l31 & 0x13) | ((l31 & 4) << 1) | ((l31 & 8) >> 1); }

}  // namespace lmx
