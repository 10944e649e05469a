// The element conversions of copyto! (src/arch/copy/copy.jl:38-43), shared by the copy kernels.
#pragma once

#include "moye_common.hpp"

namespace moye {

__device__ __forceinline__ float bf16_to_f32(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

// round to nearest even, a NaN made quiet: v_cvt_pk_bf16_f32 (the same bits as the integer form for all 2^32 inputs)
__device__ __forceinline__ uint16_t f32_to_bf16(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }

// OCP e4m3fn <-> fp32 through v_cvt_f32_fp8 / v_cvt_pk_fp8_f32.  Narrowing rounds to nearest even and turns NaN, infinities
// and everything beyond the last tie (|x| > 464) into NaN, as the integer form these replaced did: a one-off kernel compared
// the two over all 2^32 inputs (and all 256 the other way) on the hardware.  They differ in one thing only, the sign of a NaN:
// the instructions make every NaN negative, here a NaN keeps the sign it came with.
__device__ __forceinline__ float f8e4m3_to_f32(uint8_t b) {
    return b == 0x7f ? __uint_as_float(0x7fc00000u) : __builtin_amdgcn_cvt_f32_fp8((int)b, 0);
}
__device__ __forceinline__ uint8_t f32_to_f8e4m3(float f) {
    const uint8_t h = (uint8_t)(__builtin_amdgcn_cvt_pk_fp8_f32(f, f, 0, false) & 0xff);
    return f != f ? (uint8_t)(((__float_as_uint(f) >> 24) & 0x80) | 0x7f) : h;
}

template <int kDt>
__device__ __forceinline__ double load_as_f64(const char* p) {
    if constexpr (kDt == MOYE_F32) return (double)*reinterpret_cast<const float*>(p);
    else if constexpr (kDt == MOYE_F16) return (double)(float)*reinterpret_cast<const _Float16*>(p);
    else if constexpr (kDt == MOYE_BF16) return (double)bf16_to_f32(*reinterpret_cast<const uint16_t*>(p));
    else if constexpr (kDt == MOYE_F8E4M3) return (double)f8e4m3_to_f32(*reinterpret_cast<const uint8_t*>(p));
    else return *reinterpret_cast<const double*>(p);
}

// Every narrower float format here embeds exactly in fp32 and fp32 in fp64, so one rounding
// step per conversion happens below (f64 -> f16/bf16/f8 goes through f32 only when the source
// was at most f32, which is then exact).
template <int kDt>
__device__ __forceinline__ void store_from(char* p, double v, bool src_is_f64) {
    if constexpr (kDt == MOYE_F64) *reinterpret_cast<double*>(p) = v;
    else if constexpr (kDt == MOYE_F32) *reinterpret_cast<float*>(p) = (float)v;
    else if constexpr (kDt == MOYE_F16)
        *reinterpret_cast<_Float16*>(p) = src_is_f64 ? (_Float16)v : (_Float16)(float)v;
    else if constexpr (kDt == MOYE_BF16) *reinterpret_cast<uint16_t*>(p) = f32_to_bf16((float)v);
    else *reinterpret_cast<uint8_t*>(p) = f32_to_f8e4m3((float)v);
}

}  // namespace moye
