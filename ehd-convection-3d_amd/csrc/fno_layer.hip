// fno_layer.hip -- the last step of a Fourier layer and of its adjoint in one
// pass: the transform along z out of the truncated spectrum, the pointwise
// channel mixing, their sum, the bias and the activation (or the product with
// its derivative).
//
// As two GEMMs the transform wrote the full activation and the pointwise
// product read it back: two of the six passes over it per layer.  What
// bounds the fused form is memory: it reads the input and the spectrum, writes the result and, in
// training, moves the pre-activation once.
//
// The transform contracts over kz for each channel, the pointwise product
// over the channels for each z: both leave a point's results in one column of
// lanes, four z of one channel or four channels of one z to a register
// group, so that a 4x4 exchange between the four rows of 16 lanes (two lane
// swaps of two registers each) brings the transform into the other's order;
// no value goes through LDS.  The spectrum of 32 points is staged once for
// all z as bf16 in LDS, in operand order.
//
// Bit-identical to those GEMMs: one 16x16x32 step per product, real and
// imaginary parts apart, then (product + (real - imaginary)) + bias in FP32.
// At 8 samples of 64x64x64 points, width 32, 12 modes along z: 181 us, with the
// GELU 235, with its derivative 267, where the transform took 90 and the product
// 181 to 220.
#include <hip/hip_runtime.h>

#include "fno_device.h"
#include "fno_internal.h"

namespace ehd {
namespace {

constexpr int PT = 32;   // points of a workgroup: column lj of product pt is point 2 lj + pt
constexpr int KM = 16;   // modes along z staged per point, zeros beyond

// the same value, of which the compiler makes no addresses ahead of its use: kept for each of the
// loop's bases they would fill the registers
__device__ __forceinline__ unsigned here(unsigned v)
{
    asm("" : "+v"(v));
    return v;
}

// a uniform base and a lane's offset of below 2^32 bytes: one scalar address, one vector register
__device__ __forceinline__ float2 load2(const float* base, unsigned bytes)
{
    return *(const float2*)((const char*)base + bytes);
}
__device__ __forceinline__ void store2(float* base, unsigned bytes, float2 v) { *(float2*)((char*)base + bytes) = v; }

__device__ __forceinline__ void swap16(float& a, float& b)   // odd rows of a with even rows of b
{
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    a = __uint_as_float(r[0]);
    b = __uint_as_float(r[1]);
}

__device__ __forceinline__ void swap32(float& a, float& b)   // upper half of a with lower half of b
{
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    a = __uint_as_float(r[0]);
    b = __uint_as_float(r[1]);
}

// x[b][c][z][p] -> out[b][m][z][p], W[m][c] at m*sm + c*sk, spectrum
// [b][m][kz][p], transform [kz][z] (imaginary part times sa).
// A wave has 16 of the channels m and 16 z at a time; the spectrum lies in
// dynamic LDS, [part][m][pt][lj][kz].
template <int WT, int MODE>
__global__ void __launch_bounds__(256, 2)
layer_out_kernel(const float* __restrict__ x, const float* __restrict__ W, int sm, int sk,
                 const float* __restrict__ Ar, const float* __restrict__ Ai, float sa, const float* __restrict__ Sr,
                 const float* __restrict__ Si, const float* __restrict__ bias, const float* __restrict__ dact,
                 float* __restrict__ pre, float* __restrict__ out, int KZ, int Z, int P)
{
    constexpr int w = WT * 16;
    extern __shared__ __align__(16) unsigned short Sp[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, lj = lane & 15, lg = lane >> 4;
    const int tiles = (P + PT - 1) / PT;
    const int b = blockIdx.x / tiles, p0 = (blockIdx.x - b * tiles) * PT;
    const long long S = (long long)Z * P;
    // stage: 4 points of two kz a thread
    for (int i = threadIdx.x; i < 2 * w * KM / 2 * (PT / 4); i += 256) {
        const int q = i % (PT / 4), k = 2 * (i / (PT / 4) % (KM / 2)), r = i / (PT / 4 * KM / 2);   // r: part*w + m
        const int m = r % w, p = p0 + 4 * q;
        const float* src = (r < w ? Sr : Si) + (((long long)b * w + m) * KZ + k) * P + p;
        float4 u = make_float4(0.f, 0.f, 0.f, 0.f), v = u;
        if (p < P && k < KZ) u = *(const float4*)src;
        if (p < P && k + 1 < KZ) v = *(const float4*)(src + P);
        // points 4q .. 4q + 3: columns 2q and 2q + 1 of both products
        unsigned short* d = Sp + (r * PT + 2 * q) * KM + k;
        *(uint32_t*)d = pack_bf16(u.x, v.x);
        *(uint32_t*)(d + 16 * KM) = pack_bf16(u.y, v.y);
        *(uint32_t*)(d + KM) = pack_bf16(u.z, v.z);
        *(uint32_t*)(d + 17 * KM) = pack_bf16(u.w, v.w);
    }
    __syncthreads();
    const int m0 = (wave % WT) * 16;
    bf16x8 aw;
    float bv[4];
    {
        float f[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] = 8 * lg + e < w ? W[(m0 + lj) * sm + (8 * lg + e) * sk] : 0.f;
        aw = to_bf16x8(f);
#pragma unroll
        for (int e = 0; e < 4; ++e) bv[e] = MODE <= kLayerGelu ? bias[m0 + 4 * lg + e] : 0.f;
    }
    const int p = p0 + 2 * lj;
    const bool on = p < P;
    // bytes to the input's channels 8 lg .. and the output's m0 + 4 lg ..: 32 bits as S < 2^25
    const unsigned xo = 4u * ((unsigned)(8 * lg < w ? 8 * lg : 0) * (unsigned)S + (on ? p : 0));
    const unsigned oo = 4u * ((unsigned)(4 * lg) * (unsigned)S + (on ? p : 0));
    const float* xb = x + (long long)b * w * S;
    const long long ob = ((long long)b * w + m0) * S;
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    for (int z0 = (wave / WT) * 16; z0 < Z; z0 += 4 / WT * 16) {
        float2 xr[8];
        auto load = [&](int z) {
            const unsigned o = here(xo);
#pragma unroll
            for (int e = 0; e < 8; ++e) xr[e] = load2(xb + e * S + (long long)z * P, o);
        };
        load(z0);
        bf16x8 ar, ai;
        {
            float f[8], g[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const bool in = 8 * lg + e < KZ && z0 + lj < Z;
                const int at = in ? (8 * lg + e) * Z + z0 + lj : 0;
                f[e] = in ? Ar[at] : 0.f;
                g[e] = in ? sa * Ai[at] : 0.f;
            }
            ar = to_bf16x8(f);
            ai = to_bf16x8(g);
        }
        // sp[pt][4 g + c][e]: channel m0 + 4 lg + c, z0 + 4 g + e, from the products of the
        // channels m0 + 4 g + c, which hold z0 + 4 lg + e
        float sp[2][16][4];
#pragma unroll
        for (int pt = 0; pt < 2; ++pt)
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                f32x4 r[4];
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const unsigned short* s = Sp + (((m0 + 4 * g + c) * 2 + pt) * 16 + lj) * KM + 8 * (lg & 1);
                    bf16x8 br, bi;
                    __builtin_memcpy(&br, s, 16);
                    __builtin_memcpy(&bi, s + w * PT * KM, 16);
                    if (lg >= 2) br = bi = bf16x8{};
                    r[g] = mfma(ar, br, zero) - mfma(ai, bi, zero);
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    float q0 = r[0][e], q1 = r[1][e], q2 = r[2][e], q3 = r[3][e];
                    swap16(q0, q1);
                    swap16(q2, q3);
                    swap32(q0, q2);
                    swap32(q1, q3);
                    sp[pt][c][e] = q0;
                    sp[pt][4 + c][e] = q1;
                    sp[pt][8 + c][e] = q2;
                    sp[pt][12 + c][e] = q3;
                }
                __builtin_amdgcn_sched_barrier(0);   // no reads ahead: the registers are full
            }
#pragma unroll 1
        for (int g = 0; g < 4 && z0 + 4 * g < Z; ++g) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int z = z0 + 4 * g + e;
                if (z >= Z) break;
                float f0[8], f1[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    f0[i] = 8 * lg < w ? xr[i].x : 0.f;
                    f1[i] = 8 * lg < w ? xr[i].y : 0.f;
                }
                const bf16x8 b0 = to_bf16x8(f0), b1 = to_bf16x8(f1);
                if (z + 1 < Z) load(z + 1);
                const long long at = ob + (long long)z * P;
                const unsigned o = here(oo);
                float2 u[4];
                if (MODE == kLayerGrad)
#pragma unroll
                    for (int c = 0; c < 4; ++c) u[c] = load2(dact + at + c * S, o);
                const f32x4 y0 = mfma(aw, b0, zero), y1 = mfma(aw, b1, zero);
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    float2 y = make_float2(y0[c] + sp[0][c][e], y1[c] + sp[1][c][e]);
                    if (MODE <= kLayerGelu) y = make_float2(y.x + bv[c], y.y + bv[c]);
                    if (MODE == kLayerGelu) {
                        if (pre && on) store2(pre + at + c * S, o, y);
                        y = make_float2(gelu(y.x), gelu(y.y));
                    }
                    if (MODE == kLayerGrad) y = make_float2(y.x * gelu_grad(u[c].x), y.y * gelu_grad(u[c].y));
                    if (on) store2(out + at + c * S, o, y);
                }
            }
            // the next four z to the front: a rolled loop keeps the code of 16 z within the instruction cache
#pragma unroll
            for (int pt = 0; pt < 2; ++pt)
#pragma unroll
                for (int m = 0; m < 12; ++m)
#pragma unroll
                    for (int e = 0; e < 4; ++e) sp[pt][m][e] = sp[pt][m + 4][e];
        }
    }
}

template <int WT>
hipError_t launch(const LayerOut& a, hipStream_t st)
{
    const int lds = 2 * WT * 16 * PT * KM * 2;
    const auto kernel = a.mode == kLayerBias   ? layer_out_kernel<WT, kLayerBias>
                        : a.mode == kLayerGelu ? layer_out_kernel<WT, kLayerGelu>
                        : a.mode == kLayerNone ? layer_out_kernel<WT, kLayerNone>
                                               : layer_out_kernel<WT, kLayerGrad>;
    const long long blocks = (long long)((a.P + PT - 1) / PT) * a.B;
    if (blocks > 2147483647LL) return hipErrorInvalidValue;
    kernel<<<(unsigned)blocks, 256, lds, st>>>(a.x, a.W, a.sm, a.sk, a.Ar, a.Ai, a.sa, a.Sr, a.Si, a.bias, a.dact,
                                               a.pre, a.out, a.KZ, a.Z, a.P);
    return hipGetLastError();
}

}  // namespace

// 512 workgroups, two on every compute unit, run at a time; where the last such
// round is less than seven eighths full the GEMMs, which spread the same work
// wider, are the faster ones.  Training steps at width 32, kernel against
// GEMMs: 64x64x64 with 2, 3, 4 samples (256, 384, 512 workgroups) 2.42/2.32,
// 2.97/2.87, 3.20/3.40 ms; 48x48x64 with 6, 8 (432, 576) 3.24/3.23, 4.20/4.01 ms.
bool layer_fits(int w, int B, int KZ, int Z, long long P)
{
    const long long blocks = (P + PT - 1) / PT * B, rounds = (blocks + 511) / 512;
    return (w == 16 || w == 32) && KZ <= KM && P % 4 == 0 && Z * P < (1 << 25) && 8 * blocks >= 7 * 512 * rounds;
}

hipError_t layer_out(const LayerOut& a, hipStream_t st)
{
    if (a.B < 1 || a.P < 1 || a.Z < 1 || a.KZ < 1 || !layer_fits(a.w, a.B, a.KZ, a.Z, a.P) ||
        (a.mode <= kLayerGelu && !a.bias) || (a.mode == kLayerGrad && !a.dact))
        return hipErrorInvalidValue;
    return a.w == 32 ? launch<2>(a, st) : launch<1>(a, st);
}

}  // namespace ehd
