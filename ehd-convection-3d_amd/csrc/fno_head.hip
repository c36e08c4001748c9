// fno_head.hip -- the surrogate's projection width -> 128 -> d_out at every
// point (bias, GELU between the two layers) and its backward pass, one kernel
// each way.
//
// As separate GEMMs the hidden layer went through memory at every step: 128
// channels of pre-activations and of activations written and read forward,
// read again and their gradient written once and read three times backward:
// ten passes over four times the bytes of the input.  Here the hidden channels of a tile
// of points live in registers and LDS; the pre-activation is kept for the
// backward pass (a prediction keeps nothing), which forms the activation, the
// hidden gradient, the input gradient, both weight gradients and the bias sums
// from it in one go.  What bounds it is the error function of every hidden
// value, computed once each way, no longer memory.
//
// Bit-identical to those GEMMs: the same 16x16x32 steps over the same k (the
// input channels; 128 hidden in four steps; d_out; 32 consecutive points of a
// slice of 2048), operands rounded to bf16 where the GEMMs staged them, FP32
// epilogues.  At 8 samples of 64x64x64 points, width 32, 2.0 ms of GEMMs and
// sums became 0.37 ms forward and 1.07 backward (0.08 for a prediction of 4).
#include <hip/hip_runtime.h>

#include "fno_device.h"
#include "fno_internal.h"

namespace ehd {
namespace {

constexpr int H = 128, HT = H / 16;   // hidden channels and their 16-channel tiles
constexpr int PT = 32;                // points of a tile, two 16-point halves
constexpr int HP = H + 8;             // pitch of a point's hidden channels (bf16)
constexpr int QP = PT + 8;            // pitch of a hidden channel's points (bf16)
constexpr int SLICE = 2048;           // points of one partial weight gradient

// LDS written by some lanes of a wave is read by others of the same wave
__device__ __forceinline__ void wave_exchange()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ bf16x8 operand(const unsigned short* p)
{
    bf16x8 r;
    __builtin_memcpy(&r, p, 16);
    return r;
}

// the sum of a quad as a sum over stored values forms it: no product of its
// terms is fused into the additions
__device__ __forceinline__ float quad_total(float4 d)
{
#pragma clang fp contract(off)
    return (d.x + d.y) + (d.z + d.w);
}

// operand of row (column) m of M[m][k] at m*sm + k*sk, k = k0 .. k0 + 7: zero beyond rows x cols
__device__ __forceinline__ bf16x8 weights(const float* __restrict__ M, int m, int rows, int sm, int k0, int cols, int sk)
{
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = (m < rows && k0 + e < cols) ? M[m * sm + (k0 + e) * sk] : 0.f;
    return to_bf16x8(v);
}

// out[o][p] = b2[o] + sum_h W2[h][o] gelu(z1[h][p]), z1[h][p] = b1[h] + sum_c W1[c][h] v[c][p].
// A wave takes tiles of PT points in turn, points as rows and channels as
// columns of the products, so that a lane holds four consecutive points of a
// channel; the hidden channels turn around in the wave's piece of LDS.
// KEEP: z1 is stored.
template <int WT, bool KEEP>
__global__ void __launch_bounds__(256) head_fwd_kernel(const float* __restrict__ v, const float* __restrict__ W1,
                                                       const float* __restrict__ b1, const float* __restrict__ W2,
                                                       const float* __restrict__ b2, float* __restrict__ z1,
                                                       float* __restrict__ out, int B, int O, long long S)
{
    constexpr int w = WT * 16;
    __shared__ __align__(16) unsigned short Hs[4][PT * HP];   // [wave][point][hidden]
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, lj = lane & 15, lg = lane >> 4;
    unsigned short* Hw = Hs[wave];
    bf16x8 a1[HT], a2[H / 32];
    float bias[HT];
#pragma unroll
    for (int t = 0; t < HT; ++t) {
        a1[t] = weights(W1, t * 16 + lj, H, 1, 8 * lg, w, H);
        bias[t] = b1[t * 16 + lj];
    }
#pragma unroll
    for (int s = 0; s < H / 32; ++s) a2[s] = weights(W2, lj, O, 1, 32 * s + 8 * lg, H, O);
    const float bias2 = lj < O ? b2[lj] : 0.f;
    const long long per = (S + PT - 1) / PT, tiles = per * B;
    for (long long tile = (long long)blockIdx.x * 4 + wave; tile < tiles; tile += (long long)gridDim.x * 4) {
        const int b = (int)(tile / per);
        const long long p0 = (tile - b * per) * PT;
        bf16x8 x[2];
#pragma unroll
        for (int ct = 0; ct < 2; ++ct) {
            // a row beyond the last point repeats it and is not stored
            const long long p = p0 + ct * 16 + lj < S ? p0 + ct * 16 + lj : S - 1;
            const float* row = v + ((long long)b * w + (8 * lg < w ? 8 * lg : 0)) * S + p;
            float f[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                f[e] = row[e * S];
                if (8 * lg >= w) f[e] = 0.f;
            }
            x[ct] = to_bf16x8(f);
        }
        wave_exchange();   // the last tile's reads of Hw are done
#pragma unroll
        for (int t = 0; t < HT; ++t)
#pragma unroll
            for (int ct = 0; ct < 2; ++ct) {
                const f32x4 acc = mfma(x[ct], a1[t], f32x4{0.f, 0.f, 0.f, 0.f});
                const long long p = p0 + ct * 16 + 4 * lg;
                float4 z;
                z.x = acc[0] + bias[t];
                z.y = acc[1] + bias[t];
                z.z = acc[2] + bias[t];
                z.w = acc[3] + bias[t];
                if (KEEP && p < S) *(float4*)(z1 + ((long long)b * H + t * 16 + lj) * S + p) = z;
                unsigned short* q = Hw + (ct * 16 + 4 * lg) * HP + t * 16 + lj;
                q[0] = (unsigned short)to_bf16(gelu(z.x));
                q[HP] = (unsigned short)to_bf16(gelu(z.y));
                q[2 * HP] = (unsigned short)to_bf16(gelu(z.z));
                q[3 * HP] = (unsigned short)to_bf16(gelu(z.w));
            }
        wave_exchange();
#pragma unroll
        for (int ct = 0; ct < 2; ++ct) {
            f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < H / 32; ++s) acc = mfma(operand(&Hw[(ct * 16 + lj) * HP + 32 * s + 8 * lg]), a2[s], acc);
            const long long p = p0 + ct * 16 + 4 * lg;
            if (lj < O && p < S)
                *(float4*)(out + ((long long)b * O + lj) * S + p) =
                    make_float4(acc[0] + bias2, acc[1] + bias2, acc[2] + bias2, acc[3] + bias2);
        }
    }
}

// The backward pass of one slice of a sample's points, a workgroup's, PT
// points at a time in order (the order of the weight gradients' sums):
//   dh[h][p] = (sum_o W2[h][o] dout[o][p]) gelu'(z1[h][p]),
//   dv[c][p] = sum_h W1[c][h] dh[h][p],
//   dW1[c][h] = sum_p v[c][p] dh[h][p], dW2[h][o] = sum_p gelu(z1[h][p]) dout[o][p] over the slice,
//   quads[h][p/4] = the sums of four consecutive dh, for the bias gradient.
// A wave has 32 hidden channels, their weights and gradients in registers,
// and one of the tile's 16x16 pieces of dv, for which the waves exchange dh
// (two buffers, one barrier a tile).
template <int WT>
__global__ void __launch_bounds__(256, 4)
head_bwd_kernel(const float* __restrict__ v, const float* __restrict__ z1, const float* __restrict__ dout,
                const float* __restrict__ W1, const float* __restrict__ W2, float* __restrict__ dv,
                float* __restrict__ dW1, float* __restrict__ dW2, float* __restrict__ quads, int O, int S,
                int nsplit)
{
    constexpr int w = WT * 16;
    __shared__ __align__(16) unsigned short Ds[2][PT * HP];   // dh [point][hidden]
    __shared__ __align__(16) unsigned short Ks[4][2 * 32 * QP];   // [wave][dh, activation][its hidden channel][point]
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, lj = lane & 15, lg = lane >> 4;
    const int h0 = wave * 32, dp = wave & 1, dc = wave >> 1;   // this wave's channels; its half and channel tile of dv
    unsigned short* Kw = Ks[wave];
    const int b = blockIdx.x / nsplit;
    const int q0 = (blockIdx.x - b * nsplit) * SLICE;
    const int q1 = q0 + SLICE < S ? q0 + SLICE : S;   // a multiple of 4
    const float* vb = v + (long long)b * w * S;
    const float* ob = dout + (long long)b * O * S;
    const float* zb = z1 + ((long long)b * H + h0) * S;
    float* qb = quads + ((long long)b * H + h0) * (S / 4);
    float* db = dv + ((long long)b * w + dc * 16) * S;
    const unsigned row = (unsigned)lj * S;   // this lane's channel, in a tile of 16: 32 bits as S < 2^26
    bf16x8 a2[2], a1[H / 32];
#pragma unroll
    for (int t = 0; t < 2; ++t) a2[t] = weights(W2, h0 + t * 16 + lj, H, O, 8 * lg, O, 1);
    if (dc < WT)
#pragma unroll
        for (int s = 0; s < H / 32; ++s) a1[s] = weights(W1, dc * 16 + lj, w, H, 32 * s + 8 * lg, H, 1);
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    f32x4 g1[WT][2], g2[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        g2[t] = zero;
#pragma unroll
        for (int c = 0; c < WT; ++c) g1[c][t] = zero;
    }
    int buf = 0;
    for (int p0 = q0; p0 < q1; p0 += PT, buf ^= 1) {
        // rows of points: dout's channels of a point
        bf16x8 xo[2];
#pragma unroll
        for (int ct = 0; ct < 2; ++ct) {
            const int p = p0 + ct * 16 + lj;
            const unsigned at = p < q1 ? p : q0;
            float f[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                f[e] = 0.f;
                if (e < O) f[e] = (ob + (long long)e * S)[at];
                if (lg != 0 || p >= q1) f[e] = 0.f;
            }
            xo[ct] = to_bf16x8(f);
        }
        // eight consecutive points of a channel
        auto points = [&](const float* x0, unsigned r, bool on) {
            float f[8];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int p = p0 + 8 * lg + 4 * h;
                const float4 x = (on && p < q1) ? *(const float4*)(x0 + (r + p)) : make_float4(0.f, 0.f, 0.f, 0.f);
                f[4 * h] = x.x;
                f[4 * h + 1] = x.y;
                f[4 * h + 2] = x.z;
                f[4 * h + 3] = x.w;
            }
            return to_bf16x8(f);
        };
        bf16x8 xv[WT];
#pragma unroll
        for (int c = 0; c < WT; ++c) xv[c] = points(vb + (long long)c * 16 * S, row, true);
        const bf16x8 xk = points(ob, lj < O ? row : 0, lj < O);
        unsigned short* D = Ds[buf];
        wave_exchange();   // the last tile's reads of Kw are done
        // piece s: channel tile s/2, half s%2 of the points; rolled, so that
        // one piece's error functions at a time take registers
        auto zload = [&](int s) {
            const int p = p0 + (s & 1) * 16 + 4 * lg;
            return p < q1 ? *(const float4*)(zb + (long long)(s >> 1) * 16 * S + (row + p)) : make_float4(0.f, 0.f, 0.f, 0.f);
        };
        float4 zn = zload(0);
#pragma unroll 1
        for (int s = 0; s < 4; ++s) {
            const float4 z = zn;
            if (s < 3) zn = zload(s + 1);
            const f32x4 acc = mfma((s & 1) ? xo[1] : xo[0], (s >> 1) ? a2[1] : a2[0], zero);
            const int p = p0 + (s & 1) * 16 + 4 * lg;
            float4 d;
            d.x = acc[0] * gelu_grad(z.x);
            d.y = acc[1] * gelu_grad(z.y);
            d.z = acc[2] * gelu_grad(z.z);
            d.w = acc[3] * gelu_grad(z.w);
            if (p < q1) (qb + (long long)(s >> 1) * 16 * (S / 4))[(row + p) / 4] = quad_total(d);
            else d = make_float4(0.f, 0.f, 0.f, 0.f);
            const uint2 k = make_uint2(pack_bf16(d.x, d.y), pack_bf16(d.z, d.w));
            const int ko = ((s >> 1) * 16 + lj) * QP + (s & 1) * 16 + 4 * lg;
            *(uint2*)&Kw[ko] = k;
            // beyond the slice z = 0 and so is gelu(z)
            *(uint2*)&Kw[32 * QP + ko] = make_uint2(pack_bf16(gelu(z.x), gelu(z.y)), pack_bf16(gelu(z.z), gelu(z.w)));
            unsigned short* q = D + ((s & 1) * 16 + 4 * lg) * HP + h0 + (s >> 1) * 16 + lj;
            q[0] = (unsigned short)k.x;
            q[HP] = (unsigned short)(k.x >> 16);
            q[2 * HP] = (unsigned short)k.y;
            q[3 * HP] = (unsigned short)(k.y >> 16);
        }
        __syncthreads();
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const bf16x8 x = operand(&Kw[(t * 16 + lj) * QP + 8 * lg]);
#pragma unroll
            for (int c = 0; c < WT; ++c) g1[c][t] = mfma(xv[c], x, g1[c][t]);
            g2[t] = mfma(operand(&Kw[(32 + t * 16 + lj) * QP + 8 * lg]), xk, g2[t]);
        }
        if (dc < WT) {
            f32x4 acc = zero;
#pragma unroll
            for (int s = 0; s < H / 32; ++s) acc = mfma(operand(&D[(dp * 16 + lj) * HP + 32 * s + 8 * lg]), a1[s], acc);
            const int p = p0 + dp * 16 + 4 * lg;
            if (p < q1) *(float4*)(db + (row + p)) = make_float4(acc[0], acc[1], acc[2], acc[3]);
        }
    }
    float* G1 = dW1 + (long long)blockIdx.x * w * H;
    float* G2 = dW2 + (long long)blockIdx.x * H * O;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
#pragma unroll
            for (int c = 0; c < WT; ++c) G1[(c * 16 + 4 * lg + e) * H + h0 + t * 16 + lj] = g1[c][t][e];
            if (lj < O) G2[(h0 + t * 16 + 4 * lg + e) * O + lj] = g2[t][e];
        }
}

}  // namespace

bool head_fits(int w, int hidden, int O, long long S)
{
    return (w == 16 || w == 32) && hidden == H && O <= 8 && S % 4 == 0 && S < (1 << 26);
}

hipError_t head_forward(int w, int B, int O, long long S, const float* v, const float* W1, const float* b1,
                        const float* W2, const float* b2, float* z1, float* out, hipStream_t st)
{
    if (!head_fits(w, H, O, S) || B < 1 || S < 1) return hipErrorInvalidValue;
    const long long blocks = ((S + PT - 1) / PT * B + 3) / 4;
    // at most 2048 workgroups: the weights' operands are loaded once for several tiles
    const unsigned grid = (unsigned)(blocks < 2048 ? blocks : 2048);
    const auto kernel = w == 32 ? (z1 ? head_fwd_kernel<2, true> : head_fwd_kernel<2, false>)
                                : (z1 ? head_fwd_kernel<1, true> : head_fwd_kernel<1, false>);
    kernel<<<grid, 256, 0, st>>>(v, W1, b1, W2, b2, z1, out, B, O, S);
    return hipGetLastError();
}

int head_slices(long long S) { return (int)((S + SLICE - 1) / SLICE); }

hipError_t head_backward(int w, int B, int O, long long S, const float* v, const float* z1, const float* dout,
                         const float* W1, const float* W2, float* dv, float* dW1, float* dW2, float* quads,
                         hipStream_t st)
{
    if (!head_fits(w, H, O, S) || B < 1 || S < 1) return hipErrorInvalidValue;
    const int nsplit = head_slices(S);
    const unsigned grid = (unsigned)((long long)B * nsplit);
    const auto kernel = w == 32 ? head_bwd_kernel<2> : head_bwd_kernel<1>;
    kernel<<<grid, 256, 0, st>>>(v, z1, dout, W1, W2, dv, dW1, dW2, quads, O, (int)S, nsplit);
    return hipGetLastError();
}

}  // namespace ehd
