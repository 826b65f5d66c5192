// Device helpers that the tail's kernels (neck.hip, neck_fused.hip) share.
#pragma once
#include "common.hpp"

namespace ppocr {

// z * sigmoid(z) by the hardware exp2 and reciprocal (a few ulp from the correctly rounded one).
__device__ __forceinline__ float swish_fast(float z) { return z * __builtin_amdgcn_rcpf(1.0f + __expf(-z)); }

// The largest of two or three values, one instruction each (fmaxf on values the compiler cannot
// prove canonical, MFMA results and shuffles, costs a v_max_f32 x, x, x per operand first).
// Operands are scores, never NaN unless the inputs are; then the query's outputs are NaN with
// either form.  The hardware needs wait states between an MFMA and a read of its result, and the
// compiler counts them only for instructions it knows.  max_f32 and max3_f32 are such ones
// (v_maximum3_f32).  The settled forms are inline assembly, for scores that went through
// a settle: in the attention of neck.hip the compiler holds 114 registers with them and 139
// with the others (256 lines 145 us, 147 with the others).
__device__ __forceinline__ float max_f32(float a, float b) { return __builtin_elementwise_maximum(a, b); }
__device__ __forceinline__ float max3_f32(float a, float b, float c) { return max_f32(max_f32(a, b), c); }
__device__ __forceinline__ float max_settled(float a, float b) {
    float r;
    asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ float max3_settled(float a, float b, float c) {
    float r;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
// Waits until the results of MFMAs may be read; no read of them moves before it.  As many wait
// states as the compiler puts before a vector instruction that reads them: 8 after
// v_mfma_f32_16x16x16_f16, 10 after v_mfma_f32_16x16x4_f32.
__device__ __forceinline__ void settle_f16(f32x4& a, f32x4& b, f32x4& c, f32x4& d) {
    asm("s_nop 7" : "+v"(a), "+v"(b), "+v"(c), "+v"(d));
}
__device__ __forceinline__ void settle_f32(f32x4& a, f32x4& b, f32x4& c, f32x4& d) {
    asm("s_nop 7\n\ts_nop 1" : "+v"(a), "+v"(b), "+v"(c), "+v"(d));
}

}  // namespace ppocr
