// Operand types of the 16-bit matrix-core projections and the FP8 weight
// conversions, shared by mfma.hip and mfma_small.hip.
#pragma once

#include "lh_device.h"

namespace lh {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Activation plane formats of the GEMM: three exact BF16 planes (hi + mid + lo),
// or two FP16 planes of a row scaled by 2^e (h + l, about 22 significant bits).
enum { PLANES_BF16 = 3, PLANES_F16 = 2 };

// FP8 -> BF16 (or FP16) weight fragments, exact either way: the 16 codes of
// u (row bytes 16g .. 16g+15 of the step) give the two 8-column k-slices
// h = 0 (bytes 0..7) and h = 1.
__device__ __forceinline__ void fp8x16_to_bf16x8x2(u32x4 u, bf16x8& lo, bf16x8& hi)
{
    u32x4 a, b;
    a.x = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(u.x, 1.0f, false));
    a.y = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(u.x, 1.0f, true));
    a.z = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(u.y, 1.0f, false));
    a.w = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(u.y, 1.0f, true));
    b.x = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(u.z, 1.0f, false));
    b.y = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(u.z, 1.0f, true));
    b.z = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(u.w, 1.0f, false));
    b.w = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(u.w, 1.0f, true));
    lo = __builtin_bit_cast(bf16x8, a);
    hi = __builtin_bit_cast(bf16x8, b);
}

__device__ __forceinline__ void fp8x16_to_f16x8x2(u32x4 u, f16x8& lo, f16x8& hi)
{
    u32x4 a, b;
    a.x = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(u.x, 1.0f, false));
    a.y = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(u.x, 1.0f, true));
    a.z = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(u.y, 1.0f, false));
    a.w = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(u.y, 1.0f, true));
    b.x = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(u.z, 1.0f, false));
    b.y = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(u.z, 1.0f, true));
    b.z = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(u.w, 1.0f, false));
    b.w = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(u.w, 1.0f, true));
    lo = __builtin_bit_cast(f16x8, a);
    hi = __builtin_bit_cast(f16x8, b);
}

}  // namespace lh
