// fno_dft.hip -- the truncated transforms along z and y of a Fourier layer's
// input (and of its output gradient in the adjoint) in one pass.
//
// As two complex GEMMs the result along z, 2 KZ/Z of the input's size, was
// written and read back, and 12 modes filled a fifth of the 64-row tiles of
// both.  Here a workgroup transforms 32 columns x (whole cache lines) of one
// channel, 32 y at a time: along z, rounded to bf16 into LDS as the second
// transform's operands, then one step along y for every kz, whose sums stay in
// registers.  What bounds it is the one read of the input.  (16 columns and
// all y at once, half lines: 159 us against 91 here and 128 as two GEMMs, at 8
// samples of 64x64x64, width 32, 12 modes along z and 24 along y.)
//
// Bit-identical to those GEMMs: 16x16x32 steps over the same z and y in the
// same order, the same rounding between them.
#include <hip/hip_runtime.h>

#include "fno_device.h"
#include "fno_internal.h"

namespace ehd {
namespace {

constexpr int XT = 32;         // columns of a workgroup: column lj of product pt is x0 + 2 lj + pt
constexpr int kThreads = 512, kWaves = kThreads / 64;
constexpr int YP = 32 + 8;     // pitch of a column's 32 y in LDS
constexpr int kLdsMost = 80 * 1024;   // two workgroups share a compute unit

__host__ __device__ constexpr int steps(int n) { return (n + 31) / 32; }
__host__ __device__ constexpr int pitch(int n) { return 32 * steps(n) + 8; }

// LDS in bf16: tables along z [part][16][pitch(Z)] and y [part][KYp][pitch(Y)] (KYp: whole tiles of 16), then
// 32 y of the result along z [part][KZ][x][YP]
int lds_bytes(int KZ, int KY, int Y, int Z)
{
    return 4 * (16 * pitch(Z) + (KY + 15) / 16 * 16 * pitch(Y) + KZ * XT * YP);
}

// the second transform's pieces of 16 ky x 16 columns, kz of each, and a wave's share of them
int units(int KZ, int KY) { return (KZ * ((KY + 15) / 16) * 2 + kWaves - 1) / kWaves; }

// the same value, of which the compiler makes no addresses ahead of its use
__device__ __forceinline__ unsigned here(unsigned v)
{
    asm("" : "+v"(v));
    return v;
}

__device__ __forceinline__ float2 load2(const float* base, unsigned bytes)
{
    return *(const float2*)((const char*)base + bytes);
}

__device__ __forceinline__ bf16x8 operand(const unsigned short* p)
{
    bf16x8 r;
    __builtin_memcpy(&r, p, 16);
    return r;
}

// both parts of a table T[row][n] as rows of pitch(n), zeros beyond rows x n; the imaginary part times s
__device__ __forceinline__ void stage(const float* __restrict__ Tr, const float* __restrict__ Ti, float s, int rows,
                                      int n, int rows_lds, unsigned short* d)
{
    const int pn = pitch(n), all = rows_lds * pn;
#pragma unroll 4
    for (int i = threadIdx.x; i < all; i += kThreads) {
        const int r = i / pn, k = i - r * pn;
        const bool in = r < rows && k < n;
        const int at = in ? r * n + k : 0;
        const float x = Tr[at], y = Ti[at];
        d[i] = (unsigned short)to_bf16(in ? x : 0.f);
        d[all + i] = (unsigned short)to_bf16(in ? s * y : 0.f);
    }
}

// v[bc][z][y][x] -> out[bc][kz][ky][x] = sum_y B[ky][y] sum_z A[kz][z] v, A = Ar + i s Ai, B = Br + i s Bi;
// U: most pieces of a wave
template <int U>
__global__ void __launch_bounds__(kThreads, U <= 6 ? 4 : 2)
dft_zy_kernel(const float* __restrict__ v, const float* __restrict__ Ar, const float* __restrict__ Ai,
              const float* __restrict__ Br, const float* __restrict__ Bi, float s, float* __restrict__ outr,
              float* __restrict__ outi, int KZ, int KY, int X, int Y, int Z)
{
    extern __shared__ __align__(16) unsigned short lds[];
    const int xt = (X + XT - 1) / XT, bc = blockIdx.x / xt, x0 = (blockIdx.x - bc * xt) * XT;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, lj = lane & 15,
              lg = lane >> 4;
    const int pz = pitch(Z), py = pitch(Y), KYp = (KY + 15) / 16 * 16;
    unsigned short* Ta = lds;
    unsigned short* Tb = Ta + 2 * 16 * pz;
    unsigned short* Vz = Tb + 2 * KYp * py;
    const int part = KZ * XT * YP;
    const int P = X * Y, nz = steps(Z);
    const int x = x0 + 2 * lj < X ? x0 + 2 * lj : X - 2;   // columns beyond the last repeat it and are not stored
    const float* vb = v + (long long)bc * Z * P;
    const unsigned at = 4u * (unsigned)(8 * lg * P + x);   // bytes: 32 bits as 32 P < 2^30
    // the loads of a step, 8 z of a y a lane, run one step ahead
    float2 f[8];
    auto fetch = [&](int y, int k) {
        const float* base = vb + (long long)32 * k * P + y * X;
        if (32 * k + 32 <= Z) {
            const unsigned o = here(at);
#pragma unroll
            for (int e = 0; e < 8; ++e) f[e] = load2(base + e * P, o);
        } else {
            const int last = Z - 1 - 32 * k;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int z = 8 * here(lg) + e;
                f[e] = load2(base, 4u * (unsigned)((z < last ? z : last) * P + x));
                if (z > last) f[e] = make_float2(0.f, 0.f);
            }
        }
    };
    const int ny = 32 * steps(Y);
    if (wave < Y) fetch(wave, 0);
    stage(Ar, Ai, s, KZ, Z, 16, Ta);
    stage(Br, Bi, s, KY, Y, KYp, Tb);
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    f32x4 rr[U], ii[U], ri[U];
#pragma unroll
    for (int u = 0; u < U; ++u) rr[u] = ii[u] = ri[u] = zero;
    const int pieces = KZ * (KYp / 16) * 2;
    for (int y0 = 0; y0 < ny; y0 += 32) {
        __syncthreads();   // the tables are there; the last step's reads of Vz are done
        for (int y = y0 + wave; y < y0 + 32; y += kWaves) {
            f32x4 r[2] = {zero, zero}, i[2] = {zero, zero};
            if (y < Y)
                for (int k = 0; k < nz; ++k) {
                    float g[2][8];
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        g[0][e] = f[e].x;
                        g[1][e] = f[e].y;
                    }
                    const bf16x8 b[2] = {to_bf16x8(g[0]), to_bf16x8(g[1])};
                    if (k + 1 < nz) fetch(y, k + 1);
                    else if (y + kWaves < Y) fetch(y + kWaves, 0);
                    const bf16x8 ar = operand(Ta + lj * pz + 32 * k + 8 * lg);
                    const bf16x8 ai = operand(Ta + (16 + lj) * pz + 32 * k + 8 * lg);
#pragma unroll
                    for (int pt = 0; pt < 2; ++pt) {
                        r[pt] = mfma(ar, b[pt], r[pt]);
                        i[pt] = mfma(ai, b[pt], i[pt]);
                    }
                }
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (4 * lg + e < KZ)
#pragma unroll
                    for (int pt = 0; pt < 2; ++pt) {
                        unsigned short* d = Vz + ((4 * lg + e) * XT + pt * 16 + lj) * YP + (y - y0);
                        d[0] = (unsigned short)to_bf16(r[pt][e]);
                        d[part] = (unsigned short)to_bf16(i[pt][e]);
                    }
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int n = wave + u * kWaves;   // [ky tile][kz][pt]
            if (n < pieces) {
                const unsigned short* a = Tb + (n / (2 * KZ) * 16 + lj) * py + y0 + 8 * lg;
                const unsigned short* b = Vz + (n % (2 * KZ) * 16 + lj) * YP + 8 * lg;
                const bf16x8 ar = operand(a), ai = operand(a + KYp * py), br = operand(b), bi = operand(b + part);
                rr[u] = mfma(ar, br, rr[u]);
                ii[u] = mfma(ai, bi, ii[u]);
                ri[u] = mfma(ar, bi, ri[u]);
                ri[u] = mfma(ai, br, ri[u]);
            }
        }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int n = wave + u * kWaves, k0 = n / (2 * KZ) * 16, kz = n % (2 * KZ) / 2, xo = x0 + 2 * lj + n % 2;
        if (n < pieces && xo < X)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (k0 + 4 * lg + e < KY) {
                    const long long o = (((long long)bc * KZ + kz) * KY + k0 + 4 * lg + e) * X + xo;
                    outr[o] = rr[u][e] - ii[u][e];
                    outi[o] = ri[u][e];
                }
    }
}

}  // namespace

// Two workgroups must share a compute unit's LDS for the loads of one to cover
// the other's second transform.  That, not the 16 rows of the first product,
// bounds the modes along z: a mode takes 5 KB beside the tables, so at most 15
// of them fit (Y, Z <= 32, KY <= 16), at Y = Z = 64 at most 14 with KY <= 16 and
// 13 with KY <= 32; at Y = 128 11 with KY = 24.  And the workgroups must fill the chip: one takes
// a whole column, where the GEMMs split the planes further.  Training steps,
// kernel against GEMMs: width 32, 64x64x64 with 1, 4 samples (64, 256
// workgroups) 2.07/2.05, 3.20/3.31 ms, 48x48x64 with 6 (384) 3.24/3.24; width
// 16, 48x48x48 with 4 (128) 1.68/1.57.
bool dft_fits(int BC, int KZ, int KY, int X, int Y, int Z)
{
    return KZ <= 16 && X % 2 == 0 && units(KZ, KY) <= 8 && lds_bytes(KZ, KY, Y, Z) <= kLdsMost &&
           32LL * X * Y < (1 << 30) && (long long)BC * ((X + XT - 1) / XT) >= 256;
}

hipError_t dft_zy(const float* v, const float* Ar, const float* Ai, const float* Br, const float* Bi, float s,
                  float* outr, float* outi, int BC, int KZ, int KY, int X, int Y, int Z, hipStream_t st)
{
    if (BC < 1 || KZ < 1 || KY < 1 || X < 1 || Y < 1 || Z < 1 || !dft_fits(BC, KZ, KY, X, Y, Z))
        return hipErrorInvalidValue;
    const long long blocks = (long long)BC * ((X + XT - 1) / XT);
    if (blocks > 2147483647LL) return hipErrorInvalidValue;
    const int bytes = lds_bytes(KZ, KY, Y, Z), u = units(KZ, KY);
    const auto kernel = u <= 3 ? dft_zy_kernel<3> : u <= 6 ? dft_zy_kernel<6> : dft_zy_kernel<8>;
    if (bytes > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
        if (e != hipSuccess) return e;
    }
    kernel<<<(unsigned)blocks, kThreads, bytes, st>>>(v, Ar, Ai, Br, Bi, s, outr, outi, KZ, KY, X, Y, Z);
    return hipGetLastError();
}

}  // namespace ehd
