// Image output: the sRGB tonemap of src/kernel/tonemap.cu:7-39 (ToneMapping /
// ToneMappingKernel / LinearToSrgb / ApplySrgbGamma).
//
// Per channel: c < 0.0031308 ? 12.92 c : 1.055 c^(1/2.4) - 0.055, selected as glm::lerp does
// (x (1 - t) + y t, so a NaN in the branch not taken still propagates), clamped to [0, 1] with
// glm's (x < y ? y : x) / (y < x ? y : x), scaled by 255 and truncated to a byte; NaN gives 0.
// The power is evaluated in double and rounded once to float, so the CPU restatement gets the
// same bits from its own double pow.
#include "cx_internal.h"

namespace cx {

__device__ __forceinline__ uint32_t srgb_byte(float c) {
    const bool cond = c < 0.0031308f;
    const float ifTrue = 12.92f * c;
    const float p = (float)pow((double)c, (double)(1.0f / 2.4f));
    const float ifFalse = 1.055f * p - 0.055f;
    const float t = cond ? 1.0f : 0.0f;
    float v = ifFalse * (1.0f - t) + ifTrue * t;
    v = (v < 0.0f) ? 0.0f : v;
    v = (1.0f < v) ? 1.0f : v;
    v = v * 255.0f;
    return isnan(v) ? 0u : (uint32_t)(uint8_t)v;
}

// srgb_byte without the double power, or near = true: the byte then needs srgb_byte.
//
// Below 0.0031308 the branch taken is 12.92 c (a negative c gives NaN through the power, so 0);
// from 1.001 on the clamp gives 255, except where 12.92 c overflows and the branch not taken gives
// NaN, so 0.  Between them v_log_f32 and v_exp_f32 (one unit in the last place each) give the value
// on the scale of 255.  Errors there, with p the power and L = log2 c: 269 p (ln 2 (ulp(L) / 2.4 +
// ulp(L / 2.4) / 2) + 2^-23), at most 5e-5; the product, the difference and the two constants, 4e-5;
// srgb_byte's own roundings, 6e-5; together below 1.5e-4.  A value within SRGB_NEAR of a whole
// number is left to srgb_byte (one value in 2000; at twice the distance 4K took 33.8 us).
static constexpr float SRGB_NEAR = 0.25f / 1024.0f;

__device__ __forceinline__ uint32_t srgb_byte_fast(float c, bool& near) {
    const float lin = 12.92f * c;
    const float e = 269.025f * __builtin_amdgcn_exp2f(__builtin_amdgcn_logf(c) * (1.0f / 2.4f)) - 14.025f;
    const float part = e - floorf(e);
    const bool curve = c >= 0.0031308f && c < 1.001f;
    near = curve && !(part >= SRGB_NEAR && part <= 1.0f - SRGB_NEAR);
    if (curve) return (uint32_t)(int)e;
    if (c >= 1.001f) return lin < INFINITY ? 255u : 0u;
    return c > 0.0f ? (uint32_t)(int)(lin * 255.0f) : 0u;   // false for NaN
}

typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));   // the caller's floats: no wider alignment

// Memory bound: 5 bytes per value.  A thread encodes the four values of one aligned 4-byte word of
// the output (16-byte load, 4-byte store); the words at the ends, where the output does not begin
// or end on a word, go value by value.  The double power on every value was the cost before: a call
// on 24.9 M values (4K RGB) took 144 us, 33 to 35 us now (3.7 TB/s, the launch included).
__global__ __launch_bounds__(256) void k_tonemap(const float* __restrict__ hdr, uint8_t* __restrict__ ldr, uint32_t n,
                                                 uint32_t shift, uint32_t words) {
    const uint32_t g = blockIdx.x * 256u + threadIdx.x;
    if (g >= words) return;
    const int64_t first = 4 * (int64_t)g - shift;   // of the word's values
    if (first >= 0 && first + 4 <= (int64_t)n) {
        const f32x4u c = *(const f32x4u*)(hdr + first);
        uint32_t word = 0;
        bool near[4];
#pragma unroll
        for (int j = 0; j < 4; j++) word |= srgb_byte_fast(c[j], near[j]) << (8 * j);
        if (near[0] | near[1] | near[2] | near[3]) {
            // one value after the other, each thread its next: the power is rarely needed twice
            uint32_t todo = (near[0] ? 1u : 0u) | (near[1] ? 2u : 0u) | (near[2] ? 4u : 0u) | (near[3] ? 8u : 0u);
            while (todo) {
                const uint32_t j = (uint32_t)__builtin_ctz(todo);
                todo &= todo - 1u;
                const float x = j == 0 ? c[0] : j == 1 ? c[1] : j == 2 ? c[2] : c[3];
                // 1, which clamped images hold over whole regions, is next to a step, but its power is 1:
                // 1.055f - 0.055f is 1 - 2^-24 (a white 4K image 44 us, 174 by the double power)
                const uint32_t byte = x == 1.0f ? 254u : srgb_byte(x);
                word = (word & ~(0xffu << (8u * j))) | (byte << (8u * j));
            }
        }
        *(uint32_t*)(ldr + first) = word;
        return;
    }
    for (int j = 0; j < 4; j++)
        if (first + j >= 0 && first + j < (int64_t)n) ldr[first + j] = (uint8_t)srgb_byte(hdr[first + j]);
}

hipError_t launch_tonemap(const float* hdr, uint8_t* ldr, uint32_t n, hipStream_t s) {
    if (n == 0) return hipSuccess;
    const uint32_t shift = (uint32_t)((uintptr_t)ldr & 3u);
    const uint32_t words = (uint32_t)(((uint64_t)n + shift + 3) / 4);
    hipLaunchKernelGGL(k_tonemap, dim3((words + 255) / 256), dim3(256), 0, s, hdr, ldr, n, shift, words);
    return hipGetLastError();
}

}  // namespace cx
