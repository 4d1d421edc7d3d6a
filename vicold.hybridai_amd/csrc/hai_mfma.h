// hai_mfma.h -- matrix-core primitives shared by the batched and prompt GEMMs:
// the bf16 MFMA forms and the exact E4M3 -> bf16 decode.
#pragma once

#include "hai_device.h"

namespace hai {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ f32x4 mfma16(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                   0, 0, 0);
}
// 32 x 32 x 16: lane l holds A row l % 32 (B column l % 32), k 8 (l / 32) .. +7;
// result element r of lane l is row 8 (r / 4) + 4 (l / 32) + r % 4, column
// l % 32.  On MI355X this form issues at 2.1-2.2 PFLOP/s against 0.8-1.3
// for the 16 x 16 x 32 one (register-operand probe, 1-4 blocks per CU).
__device__ __forceinline__ f32x16 mfma32(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                   0, 0, 0);
}

// E4M3 codes (4 per word) -> 4 bf16 of the same values (exact: every E4M3
// value, the reference's +-480 included, has at most 4 significant bits);
// CHECK handles 0x7F / 0xFF, which the hardware conversion maps to NaN.
template <bool CHECK>
__device__ __forceinline__ void e4m3x4_to_bf16(uint32_t w, uint32_t& lo, uint32_t& hi) {
    typedef float f2v __attribute__((ext_vector_type(2)));
    f2v a = __builtin_amdgcn_cvt_pk_f32_fp8(static_cast<int>(w), false);
    f2v b = __builtin_amdgcn_cvt_pk_f32_fp8(static_cast<int>(w), true);
    if (CHECK && ((((w & 0x7f7f7f7fu) + 0x01010101u) & 0x80808080u) != 0u)) {
        // exact decode of fp8_dequant.cc:12-26 for the word holding a special code
        float f[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t c = (w >> (8 * j)) & 0xffu;
            const uint32_t t = c & 0x7fu;
            float v = t >= 8u ? __uint_as_float((t << 20) + 0x3c000000u)
                              : __uint_as_float((t << 20) + 0x3c800000u) - 0x1p-6f;
            f[j] = (c & 0x80u) ? -v : v;
        }
        a = f2v{f[0], f[1]};
        b = f2v{f[2], f[3]};
    }
    lo = (__float_as_uint(a.x) >> 16) | (__float_as_uint(a.y) & 0xffff0000u);
    hi = (__float_as_uint(b.x) >> 16) | (__float_as_uint(b.y) & 0xffff0000u);
}

// The same without the 0x7F / 0xFF check, by gfx950's scaled conversion (scale
// 1): two codes to two bf16 in one instruction, exact.
__device__ __forceinline__ uint32_t e4m3x2_to_bf16(uint32_t w, bool high) {
    typedef __bf16 b2v __attribute__((ext_vector_type(2)));
    const b2v v = high ? __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.0f, true)
                       : __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.0f, false);
    return __builtin_bit_cast(uint32_t, v);
}

}  // namespace hai
