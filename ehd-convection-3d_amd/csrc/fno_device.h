// fno_device.h -- device helpers shared by the surrogate's kernels.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace ehd {
namespace {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// rounded to nearest even, two to a conversion instruction
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi)
{
    const bf16x2 v = {(__bf16)lo, (__bf16)hi};
    uint32_t u;
    __builtin_memcpy(&u, &v, 4);
    return u;
}

__device__ __forceinline__ uint32_t to_bf16(float f) { return pack_bf16(f, 0.f) & 0xFFFFu; }

// GELU with the exact (erf) form, and its derivative
__device__ __forceinline__ float gelu(float v) { return 0.5f * v * (1.0f + erff(v * 0.70710678118654752f)); }

__device__ __forceinline__ float gelu_grad(float x)
{
    return 0.5f * (1.0f + erff(x * 0.70710678118654752f)) + x * expf(-0.5f * x * x) * 0.3989422804014327f;
}

// eight floats rounded to one lane's eight k-values of an MFMA operand
__device__ __forceinline__ bf16x8 to_bf16x8(const float* v)
{
    uint32_t w[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = pack_bf16(v[2 * i], v[2 * i + 1]);
    bf16x8 r;
    __builtin_memcpy(&r, w, 16);
    return r;
}

__device__ __forceinline__ f32x4 mfma(bf16x8 a, bf16x8 b, f32x4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

}  // namespace
}  // namespace ehd
