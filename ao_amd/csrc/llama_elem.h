// The 16-bit element types of the Llama harness kernels (llama_decode.hip, llama_prefill.hip).
#pragma once
#include "common.h"

namespace ao {

// The 16-bit element type of the activations, weights and caches: bf16 (the int4 / int8 models) or fp16 (the FP6 model,
// whose linear takes fp16 activations).  Conversions of single values and of the two halves of a packed dword, and the
// rounding an op writing that dtype applies.
struct ElemBf16 {
    static __device__ __forceinline__ float lo(uint32_t u) { return __uint_as_float(u << 16); }
    static __device__ __forceinline__ float hi(uint32_t u) { return __uint_as_float(u & 0xffff0000u); }
    static __device__ __forceinline__ float from_bits(uint16_t b) { return bf16_bits_to_f32(b); }
    static __device__ __forceinline__ uint16_t to_bits(float f) { return f32_to_bf16_bits(f); }
    static __device__ __forceinline__ float rne(float f) { return rne_bf16(f); }
    static constexpr uint32_t kNegInf2 = 0xff80ff80u;  // two -inf
};
struct ElemF16 {
    static __device__ __forceinline__ float lo(uint32_t u) { return f16_bits_to_f32((uint16_t)(u & 0xffffu)); }
    static __device__ __forceinline__ float hi(uint32_t u) { return f16_bits_to_f32((uint16_t)(u >> 16)); }
    static __device__ __forceinline__ float from_bits(uint16_t b) { return f16_bits_to_f32(b); }
    static __device__ __forceinline__ uint16_t to_bits(float f) { return f32_to_f16_bits(f); }
    static __device__ __forceinline__ float rne(float f) { return f16_bits_to_f32(f32_to_f16_bits(f)); }
    static constexpr uint32_t kNegInf2 = 0xfc00fc00u;  // two -inf
};

}  // namespace ao
