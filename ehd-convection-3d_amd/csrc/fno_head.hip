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
// sums became 0.28 ms forward and 0.51 backward (0.08 for a prediction of 4).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "fno_device.h"
#include "fno_internal.h"

namespace ehd {
namespace {

constexpr int H = 128, HT = H / 16;   // hidden channels and their 16-channel tiles
constexpr int PT = 32;                // points of a tile, two 16-point halves
constexpr int HP = H + 8;             // pitch of a point's hidden channels (bf16)
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
__device__ __forceinline__ float quad_total(const float* d)
{
#pragma clang fp contract(off)
    return (d[0] + d[1]) + (d[2] + d[3]);
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
// Row i of half ct of a tile is point 8 (i/4) + 4 ct + i%4: the four rows of a
// lane in both halves are eight consecutive points.  KEEP: z1 is stored, tile
// by tile in the order in which the lanes hold it, [tile][t][ct][lane][4].
// (By channel, z1 was a page per channel for every 128 bytes: 0.35 against
// 0.28 ms here and 1.04 against 0.87 in the backward kernel at 8 samples of
// 64x64x64, width 32.)
template <int WT, bool KEEP>
__global__ void __launch_bounds__(256) head_fwd_kernel(const float* __restrict__ v, const float* __restrict__ W1,
                                                       const float* __restrict__ b1, const float* __restrict__ W2,
                                                       const float* __restrict__ b2, float* __restrict__ z1,
                                                       float* __restrict__ out, int B, int O, long long S)
{
    constexpr int w = WT * 16;
    __shared__ __align__(16) unsigned short Hs[4][PT * HP];   // [wave][point][hidden]
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, lj = lane & 15, lg = lane >> 4;
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
            // a row beyond the last point repeats it; its output is not stored
            const long long pr = p0 + 8 * (lj >> 2) + 4 * ct + (lj & 3), p = pr < S ? pr : S - 1;
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
                float4 z;
                z.x = acc[0] + bias[t];
                z.y = acc[1] + bias[t];
                z.z = acc[2] + bias[t];
                z.w = acc[3] + bias[t];
                if (KEEP) *(float4*)(z1 + tile * (H * PT) + ((t * 2 + ct) * 64 + lane) * 4) = z;
                unsigned short* q = Hw + (8 * lg + 4 * ct) * HP + t * 16 + lj;
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
//   quads[tile][h][PT/4] = the sums of four consecutive dh, for the bias gradient.
// A wave has 32 hidden channels, their weights and gradients in registers,
// and one of the tile's 16x16 pieces of dv, for which the waves exchange dh
// (two buffers, one barrier a tile).  With the forward kernel's order of the
// points, dh and the activation lie in the lanes as the weight gradients'
// products take them.
template <int WT>
__global__ void __launch_bounds__(256, 4)
head_bwd_kernel(const float* __restrict__ v, const float* __restrict__ z1, const float* __restrict__ dout,
                const float* __restrict__ W1, const float* __restrict__ W2, float* __restrict__ dv,
                float* __restrict__ dW1, float* __restrict__ dW2, float* __restrict__ quads, int O, int S,
                int nsplit)
{
    constexpr int w = WT * 16;
    __shared__ __align__(16) unsigned short Ds[2][PT * HP];   // dh [point][hidden]
    __shared__ __align__(16) unsigned short Ws[w * HP];       // W1 [c][hidden]
    __shared__ __align__(16) unsigned short Xs[4][PT * 8];    // dout [wave][row of the products][channel]
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, lj = lane & 15, lg = lane >> 4;
    const int h0 = wave * 32, dp = wave & 1, dc = wave >> 1;   // this wave's channels; its half and channel tile of dv
    unsigned short* Xw = Xs[wave];
    const int b = blockIdx.x / nsplit;
    const int q0 = (blockIdx.x - b * nsplit) * SLICE;
    const int q1 = q0 + SLICE < S ? q0 + SLICE : S;   // a multiple of 4
    const float* vb = v + (long long)b * w * S;
    const float* ob = dout + (long long)b * O * S;
    float* db = dv + ((long long)b * w + dc * 16) * S;
    const unsigned row = (unsigned)lj * S;   // this lane's channel, in a tile of 16: 32 bits as S < 2^26
    const unsigned rowo = lj < O ? row : 0;
    for (int i = threadIdx.x; i < w * H / 2; i += 256) {
        const float2 x = *(const float2*)(W1 + 2 * i);
        *(uint32_t*)&Ws[(i / (H / 2)) * HP + 2 * (i % (H / 2))] = pack_bf16(x.x, x.y);
    }
    bf16x8 a2[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) a2[t] = weights(W2, h0 + t * 16 + lj, H, O, 8 * lg, O, 1);
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    f32x4 g1[WT][2], g2[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        g2[t] = zero;
#pragma unroll
        for (int c = 0; c < WT; ++c) g1[c][t] = zero;
    }
    float4 z[2][2], xr[WT + 1][2];
    const float* zt = z1 + ((long long)b * ((S + PT - 1) / PT) + q0 / PT) * (H * PT) + h0 * PT + lane * 4;
    float* qt = quads + ((long long)b * ((S + PT - 1) / PT) + q0 / PT) * (H * PT / 4) + h0 * (PT / 4) +
                lj * (PT / 4) + 2 * lg;
    auto load_z = [&](int t) {
        z[t][0] = *(const float4*)(zt + t * 512);
        z[t][1] = *(const float4*)(zt + t * 512 + 256);
    };
    auto load_x = [&](int p0) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int q = p0 + 8 * lg + 4 * k, p = q < q1 ? q : q1 - 4;
#pragma unroll
            for (int c = 0; c < WT; ++c) xr[c][k] = *(const float4*)(vb + (long long)c * 16 * S + (row + p));
            xr[WT][k] = *(const float4*)(ob + (rowo + p));
        }
    };
    int buf = 0;
    for (int p0 = q0; p0 < q1; p0 += PT, buf ^= 1) {
        load_x(p0);
        load_z(0);
        load_z(1);
        unsigned short* D = Ds[buf];
        if (p0 + PT > q1)   // points beyond the slice count as zeros
#pragma unroll
            for (int c = 0; c <= WT; ++c)
#pragma unroll
                for (int k = 0; k < 2; ++k)
                    if (p0 + 8 * lg + 4 * k >= q1) xr[c][k] = make_float4(0.f, 0.f, 0.f, 0.f);
        bf16x8 x[WT + 1];
#pragma unroll
        for (int c = 0; c <= WT; ++c) {
            const float f[8] = {xr[c][0].x, xr[c][0].y, xr[c][0].z, xr[c][0].w,
                                xr[c][1].x, xr[c][1].y, xr[c][1].z, xr[c][1].w};
            x[c] = to_bf16x8(f);
        }
        if (lj >= O) x[WT] = bf16x8{};
        // dout turns from points to channels through LDS (loaded a second time by
        // channel, 16 loads of a quarter of a wave: 0.87 against 0.57 ms): point 8 lg + 4 ct + i is row 16 ct + 4 lg + i of the products
        wave_exchange();
        if (lj < 8) {
            unsigned short q[8];
            __builtin_memcpy(q, &x[WT], 16);
#pragma unroll
            for (int e = 0; e < 8; ++e) Xw[(16 * (e >> 2) + 4 * lg + (e & 3)) * 8 + lj] = q[e];
        }
        wave_exchange();
        bf16x8 xo[2] = {};
        if (lg == 0) {
            xo[0] = operand(&Xw[lj * 8]);
            xo[1] = operand(&Xw[(16 + lj) * 8]);
        }
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            float d[8], h[8];
#pragma unroll
            for (int ct = 0; ct < 2; ++ct) {
                const f32x4 acc = mfma(xo[ct], a2[t], zero);
                const float zs[4] = {z[t][ct].x, z[t][ct].y, z[t][ct].z, z[t][ct].w};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    d[4 * ct + e] = acc[e] * gelu_grad(zs[e]);
                    h[4 * ct + e] = gelu(zs[e]);
                }
            }
            if (p0 + PT > q1)
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if (p0 + 8 * lg + (e & 4) >= q1) d[e] = h[e] = 0.f;
            *(float2*)(qt + t * (16 * PT / 4)) = make_float2(quad_total(d), quad_total(d + 4));
            const bf16x8 xd = to_bf16x8(d);
            unsigned short q[8];
            __builtin_memcpy(q, &xd, 16);
#pragma unroll
            for (int e = 0; e < 8; ++e) D[(8 * lg + e) * HP + h0 + t * 16 + lj] = q[e];
#pragma unroll
            for (int c = 0; c < WT; ++c) g1[c][t] = mfma(x[c], xd, g1[c][t]);
            g2[t] = mfma(to_bf16x8(h), x[WT], g2[t]);
        }
        zt += H * PT;
        qt += H * PT / 4;
        __syncthreads();
        if (dc < WT) {
            f32x4 acc = zero;
#pragma unroll
            for (int s = 0; s < H / 32; ++s)
                acc = mfma(operand(&D[(dp * 16 + lj) * HP + 32 * s + 8 * lg]),
                           operand(&Ws[(dc * 16 + lj) * HP + 32 * s + 8 * lg]), acc);
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

// A workgroup walks a slice of 2048 points; with fewer than 128 of them the
// GEMMs, which spread a slice over several workgroups, are faster.  Training steps,
// kernel against GEMMs: width 32, 32x32x24 with 1, 4 samples (12, 48 slices) 0.98/0.84,
// 1.27/1.19 ms, 64x64x64 with 1 (128) 1.80/1.81, with 2 2.32/2.56; width 16, 48x48x64 with 1
// (72) 1.06/1.04, 32x32x48 with 8 (192) 1.52/1.60.
int head_batch(long long S) { return (int)((128 + head_slices(S) - 1) / head_slices(S)); }

long long head_points(long long S) { return (S + PT - 1) / PT * PT; }

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
