// fno_mix.hip -- the per-mode channel mixing of the surrogate's spectral
// layers: for every retained mode md a complex product of the batch's channel
// vectors with the mode's own weight matrix, and its two adjoints.
//
// The spectra are [b][c][md] (md innermost), the weights [md][c][o].  As
// batched GEMMs (one 64 x 64 tile a mode, 8 x 32 of it used, every spectrum
// element fetched by its own 4-byte load) these took 75 us each at batch 8,
// width 32, 12 modes per axis, for 85 MB: 1.1 TB/s.  Here a workgroup takes 16
// consecutive modes: it turns their spectrum rows (64-byte pieces) into LDS
// operands once, and each of its waves then streams one mode's weights from
// memory straight into MFMA operands.  Bound by the
// weights' traffic: 22 us forward (3.9 TB/s), 37 us for the two adjoints together
// (4.2 TB/s), which were 75 us each.
//
// The products are those of the GEMMs bit for bit: operands rounded to bf16
// once, one 16x16x32 step over k (channels or batch, at most 32), the real
// part as the difference of two accumulators, the imaginary part Ar Bi before
// Ai Br.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "fno_device.h"
#include "fno_internal.h"

namespace ehd {
namespace {

constexpr int MD = 16;        // modes of a workgroup
constexpr int KP = 40;        // pitch of operand rows of up to 32 channels (bf16 elements)

// Spectrum rows of MD modes from md0 into T[part][md][b][c] (pitch KP), and
// into U[part][md][c][b] (pitch BP) if U is given
template <int W, int BP>
__device__ __forceinline__ void load_spectrum(const float* __restrict__ Xr, const float* __restrict__ Xi, int B, int NM,
                                              int md0, unsigned short* T, unsigned short* U)
{
    // units: (part, b, pair of channels, quad of modes)
    const int units = 2 * B * (W / 2) * (MD / 4);
    for (int u = threadIdx.x; u < units; u += blockDim.x) {
        const int q = u & 3, cp = (u >> 2) % (W / 2), pb = (u >> 2) / (W / 2), part = pb >= B, b = part ? pb - B : pb;
        const int md = md0 + 4 * q;
        if (md >= NM) continue;   // NM is a multiple of 4
        const float* p = (part ? Xi : Xr) + ((long long)b * W + 2 * cp) * NM + md;
        const float4 v0 = *(const float4*)p, v1 = *(const float4*)(p + NM);
        const float x0[4] = {v0.x, v0.y, v0.z, v0.w}, x1[4] = {v1.x, v1.y, v1.z, v1.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int row = part * MD + 4 * q + i;
            const uint32_t w = pack_bf16(x0[i], x1[i]);
            if (T) *(uint32_t*)&T[(row * BP + b) * KP + 2 * cp] = w;
            if (U) {
                U[(row * W + 2 * cp) * BP + b] = (unsigned short)w;
                U[(row * W + 2 * cp + 1) * BP + b] = (unsigned short)(w >> 16);
            }
        }
    }
}

__device__ __forceinline__ bf16x8 operand(const unsigned short* p)
{
    bf16x8 r;
    __builtin_memcpy(&r, p, 16);
    return r;
}

__device__ __forceinline__ bf16x8 negated(bf16x8 v)
{
    uint32_t w[4];
    __builtin_memcpy(w, &v, 16);
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] ^= 0x80008000u;
    __builtin_memcpy(&v, w, 16);
    return v;
}

// The results of MD modes on their way out, Out[part][b][c][md]: the waves put
// one mode's values down, the block then writes rows of 16 modes (64 bytes;
// stored straight from the MFMA lanes every value is a memory access of its
// own, 4 bytes at a stride of NM: 52 us a forward call).  The modes of a row
// are rotated by its channel, so that a wave's 16 channels hit distinct banks.
__device__ __forceinline__ int out_at(int row, int i) { return row * MD + ((i + row) & (MD - 1)); }

template <int W, int BP>
__device__ __forceinline__ void store_spectrum(const float* Out, float* __restrict__ Xr, float* __restrict__ Xi, int B,
                                               int NM, int md0)
{
    for (int u = threadIdx.x; u < 2 * B * W * (MD / 4); u += blockDim.x) {
        const int q = u & 3, pr = u >> 2, part = pr >= B * W, r = part ? pr - B * W : pr, md = md0 + 4 * q;
        if (md >= NM) continue;
        const int row = part * BP * W + r;
        *(float4*)((part ? Xi : Xr) + (long long)r * NM + md) =
            make_float4(Out[out_at(row, 4 * q)], Out[out_at(row, 4 * q + 1)], Out[out_at(row, 4 * q + 2)],
                        Out[out_at(row, 4 * q + 3)]);
    }
}

// Y[b][o] = sum_c S[b][c] R[c][o] for every mode
template <int W, int BP>
__global__ void __launch_bounds__(256) mix_fwd_kernel(const float* __restrict__ Sr, const float* __restrict__ Si,
                                                      const float* __restrict__ Rr, const float* __restrict__ Ri,
                                                      float* __restrict__ Yr, float* __restrict__ Yi, int B, int NM)
{
    __shared__ __align__(16) unsigned short T[2 * MD * BP * KP];
    __shared__ __align__(16) float Out[2 * BP * W * MD];
    const int md0 = blockIdx.x * MD;
    load_spectrum<W, BP>(Sr, Si, B, NM, md0, T, nullptr);
    __syncthreads();
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, lj = lane & 15, lg = lane >> 4;
    const bool k_in = 8 * lg < W;
    for (int i = wave; i < MD && md0 + i < NM; i += 4) {
        const int md = md0 + i;
        float br[W / 16][8] = {}, bi[W / 16][8] = {};
        if (k_in) {
#pragma unroll
            for (int t = 0; t < W / 16; ++t)
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const long long o = ((long long)md * W + 8 * lg + e) * W + t * 16 + lj;
                    br[t][e] = Rr[o];
                    bi[t][e] = Ri[o];
                }
        }
        bf16x8 ar = {}, ai = {};
        if (k_in) {   // rows beyond the batch repeat one of it and are not stored
            ar = operand(&T[(i * BP + (lj < B ? lj : 0)) * KP + 8 * lg]);
            ai = operand(&T[((MD + i) * BP + (lj < B ? lj : 0)) * KP + 8 * lg]);
        }
#pragma unroll
        for (int t = 0; t < W / 16; ++t) {
            const bf16x8 xr = to_bf16x8(br[t]), xi = to_bf16x8(bi[t]);
            const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
            f32x4 rr = mfma(ar, xr, zero), ii = mfma(ai, xi, zero), ri = mfma(ar, xi, zero);
            ri = mfma(ai, xr, ri);
            rr -= ii;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int b = 4 * lg + e;
                if (b < B) {
                    Out[out_at(b * W + t * 16 + lj, i)] = rr[e];
                    Out[out_at((BP + b) * W + t * 16 + lj, i)] = ri[e];
                }
            }
        }
    }
    __syncthreads();
    store_spectrum<W, BP>(Out, Yr, Yi, B, NM, md0);
}

// From G[b][o] (the gradient of Y): dR[c][o] = sum_b conj(S[b][c]) G[b][o], and
// the gradient of S, sum_o G[b][o] conj(R[c][o]), in the place of S
template <int W, int BP>
__global__ void __launch_bounds__(256) mix_bwd_kernel(float* __restrict__ Sr, float* __restrict__ Si,
                                                      const float* __restrict__ Gr, const float* __restrict__ Gi,
                                                      const float* __restrict__ Rr, const float* __restrict__ Ri,
                                                      float* __restrict__ dRr, float* __restrict__ dRi, int B, int NM)
{
    __shared__ __align__(16) unsigned short Gt[2 * MD * BP * KP];   // [part][md][b][o]
    __shared__ __align__(16) unsigned short K[2 * 2 * MD * W * BP];  // [G, S][part][md][channel][b], then Out
    unsigned short *Gk = K, *Sk = K + 2 * MD * W * BP;
    float* Out = (float*)K;                                         // 2 BP W MD floats, the same bytes
    const int md0 = blockIdx.x * MD;
    for (int k = threadIdx.x; k < 2 * MD * W * BP; k += blockDim.x) ((uint32_t*)K)[k] = 0;   // samples beyond the batch
    __syncthreads();
    load_spectrum<W, BP>(Gr, Gi, B, NM, md0, Gt, Gk);
    load_spectrum<W, BP>(Sr, Si, B, NM, md0, nullptr, Sk);
    __syncthreads();
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, lj = lane & 15, lg = lane >> 4;
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    // dR: k runs over the batch
    for (int i = wave; i < MD && md0 + i < NM; i += 4) {
        bf16x8 gr[W / 16] = {}, gi[W / 16] = {}, sr[W / 16] = {}, si[W / 16] = {};
        if (8 * lg < BP) {
#pragma unroll
            for (int t = 0; t < W / 16; ++t) {
                gr[t] = operand(&Gk[(i * W + t * 16 + lj) * BP + 8 * lg]);
                gi[t] = operand(&Gk[((MD + i) * W + t * 16 + lj) * BP + 8 * lg]);
                sr[t] = operand(&Sk[(i * W + t * 16 + lj) * BP + 8 * lg]);
                si[t] = operand(&Sk[((MD + i) * W + t * 16 + lj) * BP + 8 * lg]);
            }
        }
#pragma unroll
        for (int t = 0; t < W / 16; ++t) si[t] = negated(si[t]);
#pragma unroll
        for (int tc = 0; tc < W / 16; ++tc)
#pragma unroll
            for (int to = 0; to < W / 16; ++to) {
                f32x4 rr = mfma(sr[tc], gr[to], zero), ii = mfma(si[tc], gi[to], zero), ri = mfma(sr[tc], gi[to], zero);
                ri = mfma(si[tc], gr[to], ri);
                rr -= ii;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const long long o = ((long long)(md0 + i) * W + tc * 16 + 4 * lg + e) * W + to * 16 + lj;
                    dRr[o] = rr[e];
                    dRi[o] = ri[e];
                }
            }
    }
    __syncthreads();   // Gk and Sk are done with
    // gradient of S: k runs over the output channels
    const bool k_in = 8 * lg < W;
    for (int i = wave; i < MD && md0 + i < NM; i += 4) {
        float br[W / 16][8] = {}, bi[W / 16][8] = {};
        bf16x8 ar = {}, ai = {};
        if (k_in) {
#pragma unroll
            for (int t = 0; t < W / 16; ++t) {
                const long long o = ((long long)(md0 + i) * W + t * 16 + lj) * W + 8 * lg;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    *(float4*)&br[t][4 * h] = *(const float4*)(Rr + o + 4 * h);
                    *(float4*)&bi[t][4 * h] = *(const float4*)(Ri + o + 4 * h);
                }
            }
            ar = operand(&Gt[(i * BP + (lj < B ? lj : 0)) * KP + 8 * lg]);
            ai = operand(&Gt[((MD + i) * BP + (lj < B ? lj : 0)) * KP + 8 * lg]);
        }
#pragma unroll
        for (int t = 0; t < W / 16; ++t) {
            const bf16x8 xr = to_bf16x8(br[t]), xi = negated(to_bf16x8(bi[t]));
            f32x4 rr = mfma(ar, xr, zero), ii = mfma(ai, xi, zero), ri = mfma(ar, xi, zero);
            ri = mfma(ai, xr, ri);
            rr -= ii;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int b = 4 * lg + e;
                if (b < B) {
                    Out[out_at(b * W + t * 16 + lj, i)] = rr[e];
                    Out[out_at((BP + b) * W + t * 16 + lj, i)] = ri[e];
                }
            }
        }
    }
    __syncthreads();
    store_spectrum<W, BP>(Out, Sr, Si, B, NM, md0);
}

// f(W, BP): widths 16 and 32, at most 16 samples (BP = 8 or 16)
template <class F>
void with_sizes(int w, int B, const F& f)
{
    if (w == 16 && B <= 8) f(std::integral_constant<int, 16>{}, std::integral_constant<int, 8>{});
    else if (w == 16) f(std::integral_constant<int, 16>{}, std::integral_constant<int, 16>{});
    else if (B <= 8) f(std::integral_constant<int, 32>{}, std::integral_constant<int, 8>{});
    else f(std::integral_constant<int, 32>{}, std::integral_constant<int, 16>{});
}

}  // namespace

// Widths that fill the 16-wide tiles and batches of one row tile; any other
// shape stays with the batched GEMM.
bool mix_fits(int w, int B) { return (w == 16 || w == 32) && B >= 1 && B <= 16; }

hipError_t mix_forward(int w, int B, int NM, const float* Sr, const float* Si, const float* Rr, const float* Ri,
                       float* Yr, float* Yi, hipStream_t st)
{
    if (!mix_fits(w, B) || NM <= 0 || NM % 4) return hipErrorInvalidValue;
    with_sizes(w, B, [&](auto W, auto BP) {
        mix_fwd_kernel<W.value, BP.value><<<(NM + MD - 1) / MD, 256, 0, st>>>(Sr, Si, Rr, Ri, Yr, Yi, B, NM);
    });
    return hipGetLastError();
}

hipError_t mix_backward(int w, int B, int NM, float* Sr, float* Si, const float* Gr, const float* Gi, const float* Rr,
                        const float* Ri, float* dRr, float* dRi, hipStream_t st)
{
    if (!mix_fits(w, B) || NM <= 0 || NM % 4) return hipErrorInvalidValue;
    with_sizes(w, B, [&](auto W, auto BP) {
        mix_bwd_kernel<W.value, BP.value><<<(NM + MD - 1) / MD, 256, 0, st>>>(Sr, Si, Gr, Gi, Rr, Ri, dRr, dRi, B, NM);
    });
    return hipGetLastError();
}

}  // namespace ehd
