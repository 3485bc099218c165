// Device helpers shared by the MFMA GEMM files (gemm.hip, gemm_ring.hip): vector types, exact f16
// integers from quants, loads that name an LDS destination.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/ferrum_hip.h"

namespace fh {

// Kinds kept as GGUF rows, and their bytes per 32 elements
template <int KIND>
constexpr bool kGguf = KIND != FH_Q8_0 && KIND != FH_Q4_0;
template <int KIND>
constexpr bool kFp8 = KIND == FH_FP8_E4M3 || KIND == FH_FP8_E5M2;
template <int KIND>
constexpr uint32_t kGgufBlock = kFp8<KIND> ? 34 : KIND == FH_MXFP4 ? 17 : 64;

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ float half_to_float(uint32_t h) {
    return (float)__builtin_bit_cast(_Float16, (uint16_t)h);
}

__device__ __forceinline__ float e8m0_half_scale(uint32_t e) {  // mxfp4.rs:26-33
    return e < 2 ? __uint_as_float(0x00200000u << e) : __uint_as_float((e - 1) << 23);
}

__device__ __forceinline__ uint32_t f16x2_add(uint32_t w, _Float16 bias) {
    const f16x2 v = __builtin_bit_cast(f16x2, w) + f16x2{bias, bias};
    return __builtin_bit_cast(uint32_t, v);
}

typedef __attribute__((address_space(3))) void lds_void_t;
typedef int32_t i32x4 __attribute__((ext_vector_type(4)));

// A raw buffer descriptor in scalar registers over [base, base + bytes) (the make_rsrc layout).
__device__ __forceinline__ i32x4 sgpr_rsrc(const void *base, uint32_t bytes) {
    const uint64_t a = (uint64_t)base;
    return i32x4{__builtin_amdgcn_readfirstlane((int32_t)(uint32_t)a),
                 __builtin_amdgcn_readfirstlane((int32_t)((uint32_t)(a >> 32) & 0xffffu)),
                 __builtin_amdgcn_readfirstlane((int32_t)bytes), 0x00020000};
}
// 16 (4) bytes per lane from r at voff into LDS at lds + 16 (4) * lane; lds wave-uniform. An M0
// write needs one wait state before a load that reads it.
__device__ __forceinline__ void asm_load_lds16(i32x4 r, uint32_t lds, uint32_t voff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(lds), "v"(voff),
                 "s"(r)
                 : "m0");
}
__device__ __forceinline__ void asm_load_lds4(i32x4 r, uint32_t lds, uint32_t voff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, 0 offen lds" ::"s"(lds), "v"(voff), "s"(r)
                 : "m0");
}

}  // namespace fh
