// fno_internal.h -- kernels of the Fourier-neural-operator surrogate.
#pragma once

#include <hip/hip_runtime.h>

namespace ehd {

// C(i1,i2)[m][n] = alpha * sum_k A(i1,i2)[m][k] * B(i1,i2)[k][n] + beta * C(i1,i2)[m][n]
// with A[m][k] at A + i1*a1 + i2*a2 + m*am + k*ak (likewise B, C): FP32 in
// memory, bf16 matrix-core products, FP32 accumulation.
struct GemmArgs {
    int M, N, K;
    const float* A;
    long long am, ak;
    const float* B;
    long long bk, bn;
    float* C;
    long long cm, cn;
    int nb1, nb2;
    long long a1, a2, b1, b2, c1, c2;
    float alpha, beta;
    int ksplit;        // > 0: batch index i2 takes k in [i2*ksplit, (i2+1)*ksplit) (split-K partial sums)
    // epilogue after alpha/beta: + bias[m] (null: none), then act:
    //   kActGelu: pre (C's offsets) = the value, C = gelu(value);
    //   kActGeluGrad: C = value * gelu'(dact) (dact at C's offsets)
    const float* bias = nullptr;
    int act = 0;
    float* pre = nullptr;
    const float* dact = nullptr;
};
constexpr int kActNone = 0, kActGelu = 1, kActGeluGrad = 2;

hipError_t gemm_bf16(const GemmArgs& g, hipStream_t st);
// Complex product on the matrix cores: with Ar = g.A, Br = g.B, Cr = g.C,
//   Cr = alpha * Re[(Ar + i sa Ai)(Br + i sb Bi)] + beta * Cr,
//   Ci = alpha * Im[(Ar + i sa Ai)(Br + i sb Bi)] + beta * Ci,
// each imaginary plane at the same strides as its real plane; Ai or Bi null:
// that operand is real; Ci null: only Cr is written.  sa, sb = +1 or -1
// (-1 conjugates).  No split-K.
struct CGemmArgs {
    GemmArgs g;
    const float* Ai;
    const float* Bi;
    float* Ci;
    float sa, sb;
};
hipError_t cgemm_bf16(const CGemmArgs& x, hipStream_t st);
// The per-mode mixing of a spectral layer (fno_mix.hip), bit-identical to the
// batched complex GEMMs: spectra [b][c][md], weights [md][c][o], md < NM
// (a multiple of 4); shapes for which mix_fits holds.
//   forward:  Y[b][o] = sum_c S[b][c] R[c][o]
//   backward: dR[c][o] = sum_b conj(S[b][c]) G[b][o], then S[b][c] = sum_o G[b][o] conj(R[c][o])
bool mix_fits(int w, int B);
hipError_t mix_forward(int w, int B, int NM, const float* Sr, const float* Si, const float* Rr, const float* Ri,
                       float* Yr, float* Yi, hipStream_t st);
hipError_t mix_backward(int w, int B, int NM, float* Sr, float* Si, const float* Gr, const float* Gi, const float* Rr,
                        const float* Ri, float* dRr, float* dRi, hipStream_t st);
// The transforms along z and y of real v[bc][z][y][x] (fno_dft.hip), bit-identical to two complex GEMMs:
// shapes for which dft_fits holds,
//   out[bc][kz][ky][x] = sum_y (Br + i s Bi)[ky][y] sum_z (Ar + i s Ai)[kz][z] v
bool dft_fits(int BC, int KZ, int KY, int X, int Y, int Z);
hipError_t dft_zy(const float* v, const float* Ar, const float* Ai, const float* Br, const float* Bi, float s,
                  float* outr, float* outi, int BC, int KZ, int KY, int X, int Y, int Z, hipStream_t st);
// The end of a Fourier layer or of its adjoint (fno_layer.hip), bit-identical
// to a complex and a pointwise GEMM: shapes for which layer_fits holds,
//   out[b][m][z][p] = sum_c W[m][c] x[b][c][z][p] + Re sum_kz (Ar + i sa Ai)[kz][z] (Sr + i Si)[b][m][kz][p]
// with W[m][c] at m*sm + c*sk, then by mode
//   kLayerBias: + bias[m]; kLayerGelu: + bias[m], stored to pre unless that is null, gelu;
//   kLayerNone: as it is;  kLayerGrad: times gelu'(dact).
constexpr int kLayerBias = 0, kLayerGelu = 1, kLayerNone = 2, kLayerGrad = 3;
struct LayerOut {
    int mode, w, B, KZ, Z, P;
    const float* x;
    const float* W;
    int sm, sk;
    const float *Ar, *Ai;
    float sa;
    const float *Sr, *Si;
    float* out;
    const float* bias = nullptr;
    const float* dact = nullptr;
    float* pre = nullptr;
};
bool layer_fits(int w, int B, int KZ, int Z, long long P);
hipError_t layer_out(const LayerOut& a, hipStream_t st);
// The projection width -> hidden -> d_out of a prediction and its backward
// pass (fno_head.hip), bit-identical to the pointwise GEMMs: shapes for which
// head_fits holds, S points a sample, weights [c][h] and [h][o], biases b1, b2.
//   forward:  z1 = b1 + W1 v (B hidden head_points(S) floats in an order of its own,
//             stored unless z1 is null), out = b2 + W2 gelu(z1)
//   backward: dv[b][c], the partial sums dW1[slice][c][h] and dW2[slice][h][o] of
//             B head_slices(S) slices, and the sums of four consecutive points of
//             the hidden layer's gradient, quads[b][tile of 32 points][h][8]
bool head_fits(int w, int hidden, int O, long long S);
int head_batch(long long S);   // from this batch on the backward kernel is the faster one
long long head_points(long long S);   // in whole tiles
int head_slices(long long S);
hipError_t head_forward(int w, int B, int O, long long S, const float* v, const float* W1, const float* b1,
                        const float* W2, const float* b2, float* z1, float* out, hipStream_t st);
hipError_t head_backward(int w, int B, int O, long long S, const float* v, const float* z1, const float* dout,
                         const float* W1, const float* W2, float* dv, float* dW1, float* dW2, float* quads,
                         hipStream_t st);
// staging layout gemm_bf16 picks for A and B: 0 k unit-stride, 1 m (n) unit-stride
// (16-byte loads), 2 element loads
int gemm_layout_a(const GemmArgs& g);
int gemm_layout_b(const GemmArgs& g);
// result layout: 0 element stores, 1 n unit-stride, 2 m unit-stride (16-byte
// stores through LDS)
int gemm_layout_c(const GemmArgs& g);
// dst[i] = beta*dst[i] + sum_j src[j*n + i], j < nslices; part holds
// sum_slices_part_floats(n) floats of workspace
long long sum_slices_part_floats(long long n);
hipError_t sum_slices(const float* src, float* dst, long long n, int nslices, float beta, float* part, hipStream_t st);
// db[c] (+)= sum_{b,s} g[b][c][s]; part holds channel_sum_part_floats(B, C, S) floats of workspace
long long channel_sum_part_floats(int B, int C, long long S);
hipError_t channel_sum(const float* g, float* db, int B, int C, long long S, bool accumulate, float* part,
                       hipStream_t st);
// the same sums of g, to the last bit, from the sums of its quads, quads[b][tile of 32 points][c][8]
// (S a multiple of 4, C of 8)
hipError_t channel_sum_quads(const float* quads, float* db, int B, int C, long long S, float* part, hipStream_t st);
// grad = 2 (out - tgt) / n, part[mse_blocks()] = partial sums of (out - tgt)^2; n a multiple of 4
int mse_blocks();
hipError_t mse(const float* out, const float* tgt, float* grad, double* part, long long n, hipStream_t st);
// in[b], tgt[b] = samples idx[b] (on the host) of ds_in and ds_tgt, nin and ntgt floats each
// (multiples of 4)
hipError_t gather(const float* ds_in, const float* ds_tgt, const int* idx, int B, long long nin, long long ntgt,
                  float* in, float* tgt, hipStream_t st);
// Adam (Kingma & Ba 2015), t counts from 1
hipError_t adam(float* p, const float* g, float* m, float* v, long long n, float lr, float b1, float b2, float eps,
                int t, hipStream_t st);

}  // namespace ehd
