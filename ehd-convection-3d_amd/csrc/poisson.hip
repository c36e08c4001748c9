// poisson.hip -- spectral Poisson solve for the potential.
//
// The reference (poisson.cu:78-167, main.cu:191-203) odd-extends the charge
// to nz' = 2(nz-1) planes, runs a 3-D complex DFT, divides by
//   mu = 4/dz^2 sin^2(kz dz/2) + kx^2 + ky^2
// and transforms back.  Along z that is the eigen-decomposition (a DST) of the
// second-difference operator with Dirichlet walls, so the same potential
// follows from
//   (1) a real-to-complex DFT along x and a complex DFT along y of
//       s = -q/eps on each interior plane z = 1..nz-2,
//   (2) per (kx,ky) mode, the tridiagonal solve
//       phi[z-1] - (2 + k^2 dz^2) phi[z] + phi[z+1] = dz^2 s[z],
//       phi = 0 on both walls, in FP64,
//   (3) the inverse DFTs,
// with the wall potential carried by phi_L(z) = V (1 - z/(nz-1)), which the
// second-difference operator annihilates (the lifting terms V/dz^2 of
// poisson.cu:99,119 only ever reach mode (0,0)).  The DFTs are Stockham
// mixed-radix FFTs in LDS with register butterflies of up to 16 points
// (radices 2 to 5, 7 to 9, 11, 13, 16); a larger prime factor is a stage of
// half the products of the direct DFT.
//
// Spectral layout: [z-1][kx][ky], kx in [0, nx/2], ky fastest.
// FP32S path: the spectra are float; mode (0,0) is solved in FP64 and kept
// as the per-plane mean phibar[z] (FP64), and phi holds phi - phibar in
// float, so that E = -grad(phi) loses no digits to the large wall potential.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "ehd_internal.h"
#include "fft_plan.h"

namespace ehd {
namespace {

template <typename T>
struct cplx {
    T x, y;
};

// Buffer pointers of a solve come from its job table in memory, so the
// compiler cannot see that they are global: without the address space it
// emits flat loads and stores.  Kernels access them through gptr().
#define EHD_GLOBAL __attribute__((address_space(1)))
template <typename X>
__device__ __forceinline__ EHD_GLOBAL X* gptr(X* p)
{
    return (EHD_GLOBAL X*)p;
}
template <typename T>
__device__ __forceinline__ cplx<T> ldc(EHD_GLOBAL const cplx<T>* p)
{
    return cplx<T>{p->x, p->y};
}
template <typename T>
__device__ __forceinline__ void stc(EHD_GLOBAL cplx<T>* p, cplx<T> v)
{
    p->x = v.x;
    p->y = v.y;
}

template <typename T>
__device__ __forceinline__ cplx<T> cmul(cplx<T> a, cplx<T> b)
{
    return {a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x};
}
template <typename T>
__device__ __forceinline__ cplx<T> cadd(cplx<T> a, cplx<T> b) { return {a.x + b.x, a.y + b.y}; }
template <typename T>
__device__ __forceinline__ cplx<T> csub(cplx<T> a, cplx<T> b) { return {a.x - b.x, a.y - b.y}; }
// i*s*a for s = +-1
template <typename T>
__device__ __forceinline__ cplx<T> cis(cplx<T> a, T s) { return {-s * a.y, s * a.x}; }

// root W_n^(sign*m) from the forward table tw[m] = exp(-2 pi i m/n)
template <typename T>
__device__ __forceinline__ cplx<T> root(const cplx<T>* tw, int m, int sign)
{
    cplx<T> w = tw[m];
    if (sign > 0) w.y = -w.y;
    return w;
}

// ---------------------------------------------------------------------------
// Compile-time planned FFT (the grid sizes the configurations use).  Radix 16
// and 8 butterflies run in registers (as 4x4 and 4x2 with constant inner
// twiddles), so a 256-point line takes two stages and one LDS exchange.  The
// radix schedule, the strides and every index division are constants.
// Radix of stage st: the power-of-two part 2^p is split into ceil(p/4)
// balanced stages (each 2..16, larger first: 512 = 8*8*8, 256 = 16*16,
// 128 = 16*8, 64 = 8*8), then the factors 3 and 5.  Balanced stages keep the
// butterflies per line (N / radix) small in every stage.
constexpr int ct_radix(int n, int st)
{
    if (n <= 0) return 0;
    int p = 0, r = n;
    while (r % 2 == 0) {
        r /= 2;
        ++p;
    }
    const int s2 = (p + 3) / 4;
    if (st < s2) {
        const int bits = p / s2 + (st < p % s2 ? 1 : 0);
        return 1 << bits;
    }
    int s = s2;
    const int odd[2] = {3, 5};
    for (int i = 0; i < 2; ++i)
        while (r % odd[i] == 0) {
            if (s == st) return odd[i];
            r /= odd[i];
            ++s;
        }
    return 0;
}
constexpr int ct_nst(int n)
{
    int s = 0;
    while (ct_radix(n, s) != 0) ++s;
    return s;
}
// largest number of butterflies of one line over the stages (N / smallest radix)
constexpr int ct_max_nb(int n)
{
    int m = 0;
    for (int s = 0; s < ct_nst(n); ++s) m = (n / ct_radix(n, s) > m) ? n / ct_radix(n, s) : m;
    return m;
}
// the plan covers n completely (no factor left for a runtime stage)
constexpr bool ct_complete(int n)
{
    int r = n;
    for (int s = 0; s < ct_nst(n); ++s) r /= ct_radix(n, s);
    return r == 1;
}

// a * (c + i s)
template <typename T>
__device__ __forceinline__ cplx<T> crot(cplx<T> a, T c, T s)
{
    return {a.x * c - a.y * s, a.x * s + a.y * c};
}

template <typename T>
__device__ __forceinline__ void dft4(cplx<T>& a, cplx<T>& b, cplx<T>& c, cplx<T>& d, T sg)
{
    const cplx<T> t0 = cadd(a, c), t1 = csub(a, c), t2 = cadd(b, d), t3 = csub(b, d);
    const cplx<T> it3 = cis(t3, sg);
    a = cadd(t0, t2);
    b = cadd(t1, it3);
    c = csub(t0, t2);
    d = csub(t1, it3);
}

// cos and sin of 2 pi m / R, m = 1 .. R/2, of the odd radices done by pairs
template <int R>
struct Roots;
template <>
struct Roots<7> {
    static constexpr double c[3] = {0.6234898018587335305250, -0.2225209339563144042889, -0.9009688679024191262361};
    static constexpr double s[3] = {0.7818314824680298087084, 0.9749279121818236070181, 0.4338837391175581204758};
};
template <>
struct Roots<9> {
    static constexpr double c[4] = {0.7660444431189780352024, 0.1736481776669303488517, -0.5, -0.9396926207859083840541};
    static constexpr double s[4] = {0.6427876096865393263226, 0.9848077530122080593667, 0.8660254037844386467637,
                                    0.3420201433256687330441};
};
template <>
struct Roots<11> {
    static constexpr double c[5] = {0.8412535328311811688618, 0.4154150130018864255293, -0.1423148382732851404438,
                                    -0.6548607339452850640569, -0.9594929736144973898904};
    static constexpr double s[5] = {0.5406408174555975821076, 0.9096319953545183714117, 0.9898214418809327323761,
                                    0.7557495743542582837740, 0.2817325568414296977114};
};
template <>
struct Roots<13> {
    static constexpr double c[6] = {0.8854560256532098959004, 0.5680647467311558025118, 0.1205366802553230533491,
                                    -0.3546048870425356259696, -0.7485107481711010986346, -0.9709418174260520271570};
    static constexpr double s[6] = {0.4647231720437685456560, 0.8229838658936563945796, 0.9927088740980539928008,
                                    0.9350162426854148234398, 0.6631226582407952023768, 0.2393156642875577671488};
};

// DFT of odd length R from the sums and differences of the pairs (r, R - r):
// X_q, X_{R-q} = (x_0 + sum_r cos(2 pi r q/R) s_r) +- i sg sum_r sin(2 pi r q/R) d_r,
// half the products of the direct sum
template <typename T, int R>
__device__ __forceinline__ void bfly_pairs(cplx<T>* v, T sg)
{
    constexpr int H = R / 2;
    cplx<T> s[H], d[H], x0 = v[0];
#pragma unroll
    for (int r = 1; r <= H; ++r) {
        s[r - 1] = cadd(v[r], v[R - r]);
        d[r - 1] = csub(v[r], v[R - r]);
        v[0] = cadd(v[0], s[r - 1]);
    }
#pragma unroll
    for (int q = 1; q <= H; ++q) {
        cplx<T> a = x0, b = {(T)0, (T)0};
#pragma unroll
        for (int r = 1; r <= H; ++r) {
            const int m = (r * q) % R, n = m <= H ? m : R - m;   // n = 0 only for R = 9
            const T c = n > 0 ? (T)Roots<R>::c[n > 0 ? n - 1 : 0] : (T)1;
            const T sn = n > 0 ? (T)(m <= H ? Roots<R>::s[n > 0 ? n - 1 : 0] : -Roots<R>::s[n > 0 ? n - 1 : 0]) : (T)0;
            a.x += c * s[r - 1].x;
            a.y += c * s[r - 1].y;
            b.x += sn * d[r - 1].x;
            b.y += sn * d[r - 1].y;
        }
        const cplx<T> ib = cis(b, sg);
        v[q] = cadd(a, ib);
        v[R - q] = csub(a, ib);
    }
}

template <typename T, int R>
__device__ __forceinline__ void bfly(cplx<T>* v, T sg)
{
    if constexpr (R == 2) {
        const cplx<T> a = v[0], b = v[1];
        v[0] = cadd(a, b);
        v[1] = csub(a, b);
    } else if constexpr (R == 4) {
        dft4(v[0], v[1], v[2], v[3], sg);
    } else if constexpr (R == 8) {
        // n = 2 n1 + n2, k = k1 + 4 k2: DFT4 over n1, inner twiddle W8^(n2 k1), DFT2 over n2
        const T h = (T)0.70710678118654752440;
        cplx<T> a0 = v[0], a1 = v[2], a2 = v[4], a3 = v[6];
        cplx<T> b0 = v[1], b1 = v[3], b2 = v[5], b3 = v[7];
        dft4(a0, a1, a2, a3, sg);
        dft4(b0, b1, b2, b3, sg);
        b1 = crot(b1, h, sg * h);      // W8^1
        b2 = cis(b2, sg);              // W8^2 = i sg
        b3 = crot(b3, -h, sg * h);     // W8^3
        v[0] = cadd(a0, b0); v[4] = csub(a0, b0);
        v[1] = cadd(a1, b1); v[5] = csub(a1, b1);
        v[2] = cadd(a2, b2); v[6] = csub(a2, b2);
        v[3] = cadd(a3, b3); v[7] = csub(a3, b3);
    } else if constexpr (R == 16) {
        // n = 4 n1 + n2, k = k1 + 4 k2: DFT4 over n1, inner twiddle W16^(n2 k1), DFT4 over n2
        const T c1 = (T)0.92387953251128675613, s1 = (T)0.38268343236508977173, h = (T)0.70710678118654752440;
        cplx<T> a[4][4];
#pragma unroll
        for (int n2 = 0; n2 < 4; ++n2) {
            a[n2][0] = v[n2]; a[n2][1] = v[4 + n2]; a[n2][2] = v[8 + n2]; a[n2][3] = v[12 + n2];
            dft4(a[n2][0], a[n2][1], a[n2][2], a[n2][3], sg);
        }
        a[1][1] = crot(a[1][1], c1, sg * s1);     // W16^1
        a[1][2] = crot(a[1][2], h, sg * h);       // W16^2
        a[1][3] = crot(a[1][3], s1, sg * c1);     // W16^3
        a[2][1] = crot(a[2][1], h, sg * h);       // W16^2
        a[2][2] = cis(a[2][2], sg);               // W16^4
        a[2][3] = crot(a[2][3], -h, sg * h);      // W16^6
        a[3][1] = crot(a[3][1], s1, sg * c1);     // W16^3
        a[3][2] = crot(a[3][2], -h, sg * h);      // W16^6
        a[3][3] = crot(a[3][3], -c1, -sg * s1);   // W16^9
#pragma unroll
        for (int k1 = 0; k1 < 4; ++k1) {
            cplx<T> p = a[0][k1], q = a[1][k1], r = a[2][k1], s = a[3][k1];
            dft4(p, q, r, s, sg);
            v[k1] = p; v[k1 + 4] = q; v[k1 + 8] = r; v[k1 + 12] = s;
        }
    } else if constexpr (R == 3) {
        const T s3 = (T)0.86602540378443864676;
        const cplx<T> a = v[0], t1 = cadd(v[1], v[2]), t3 = csub(v[1], v[2]);
        const cplx<T> t2 = {a.x - (T)0.5 * t1.x, a.y - (T)0.5 * t1.y};
        const cplx<T> r = cis(cplx<T>{s3 * t3.x, s3 * t3.y}, sg);
        v[0] = cadd(a, t1);
        v[1] = cadd(t2, r);
        v[2] = csub(t2, r);
    } else if constexpr (R == 7 || R == 9 || R == 11 || R == 13) {
        bfly_pairs<T, R>(v, sg);
    } else {
        static_assert(R == 5, "radix");
        const T c1 = (T)0.30901699437494742410, c2 = (T)-0.80901699437494742410;
        const T s1 = (T)0.95105651629515357212, s2 = (T)0.58778525229247312917;
        const cplx<T> a = v[0];
        const cplx<T> t1 = cadd(v[1], v[4]), t2 = cadd(v[2], v[3]), t3 = csub(v[1], v[4]), t4 = csub(v[2], v[3]);
        const cplx<T> m1 = {a.x + c1 * t1.x + c2 * t2.x, a.y + c1 * t1.y + c2 * t2.y};
        const cplx<T> m2 = {a.x + c2 * t1.x + c1 * t2.x, a.y + c2 * t1.y + c1 * t2.y};
        const cplx<T> n1 = cis(cplx<T>{s1 * t3.x + s2 * t4.x, s1 * t3.y + s2 * t4.y}, sg);
        const cplx<T> n2 = cis(cplx<T>{s2 * t3.x - s1 * t4.x, s2 * t3.y - s1 * t4.y}, sg);
        v[0] = cadd(a, cadd(t1, t2));
        v[1] = cadd(m1, n1);
        v[2] = cadd(m2, n2);
        v[3] = csub(m2, n2);
        v[4] = csub(m1, n1);
    }
}

// LDS index with one pad element per 16: the stride-R accesses of a Stockham
// stage then spread over the banks instead of a few of them.
__host__ __device__ constexpr int padi(int i) { return i + (i >> 4); }
// LDS line pitch (complex elements): long enough for the padded line and
// = 1 mod 32 (runtime plans: odd), so that threads walking across lines hit
// distinct banks.
__host__ __device__ constexpr int lds_pitch(int N, int n)
{
    if (N == 0) return n | 1;
    const int len = padi(N - 1) + 1;
    return ((len + 30) / 32) * 32 + 1;
}

// Runs the compile-time plan of N on nlines lines with one butterfly per
// thread per stage (nlines * ct_max_nb(N) <= blockDim.x).  Stage 0 reads its
// inputs through ld(l, i) -- global memory, or the LDS buffer itself when
// SRC_BUF; the other stages read buf.  Stages write back into buf in place
// (all reads of a stage complete before its writes), except that the last
// stage writes through sf(l, i, v) when DST_GLOBAL.  Every thread of the
// block must call it; the result is in buf (padded index) unless DST_GLOBAL.
template <typename T, int N, int ST, int NS, bool SRC_BUF, bool DST_GLOBAL, class LD, class SF>
__device__ __forceinline__ void ct_run(const LD& ld, const SF& sf, cplx<T>* buf, int nlines, int ldl,
                                       const cplx<T>* __restrict__ tw, int sign)
{
    constexpr int NST = ct_nst(N);
    if constexpr (ST < NST) {
        constexpr int R = ct_radix(N, ST);
        constexpr int NB = N / R;
        constexpr int TSTEP = N / (NS * R);
        constexpr bool from_buf = (ST > 0) || SRC_BUF;
        constexpr bool to_global = DST_GLOBAL && (ST == NST - 1);
        const T sg = (T)sign;
        const int w = threadIdx.x;
        const bool act = w < nlines * NB;
        const int l = w / NB, j = w - l * NB, k = j % NS;
        cplx<T> v[R];
        if (act) {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                cplx<T> x;
                if constexpr (ST == 0) x = ld(l, j + r * NB);
                else x = buf[l * ldl + padi(j + r * NB)];
                if constexpr (NS > 1) {
                    if (r > 0) x = cmul(x, root(tw, r * k * TSTEP, sign));
                }
                v[r] = x;
            }
        }
        if constexpr (from_buf && !to_global) __syncthreads();
        if (act) {
            bfly<T, R>(v, sg);
            const int o = (j / NS) * NS * R + k;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                if constexpr (to_global) sf(l, o + r * NS, v[r]);
                else buf[l * ldl + padi(o + r * NS)] = v[r];
            }
        }
        if constexpr (!to_global) __syncthreads();
        ct_run<T, N, ST + 1, NS * R, SRC_BUF, DST_GLOBAL>(ld, sf, buf, nlines, ldl, tw, sign);
    }
}

// ---------------------------------------------------------------------------
// Runtime-planned FFT (every other size): a Stockham FFT of nl <= 2^lg lines
// in LDS, ping-pong between two buffers, one register butterfly per thread
// and turn.  The lines run fastest over the threads (line pitch odd), so the
// reads and writes of a stage hit distinct banks whatever its strides, the
// twiddles are broadcasts, and the only divisions left are by the stage's Ns,
// done by a multiplication.

// a / b of a magic number from fft_magic(b): exact for a < 2^16
__device__ __forceinline__ int fdiv(int a, unsigned magic) { return (int)__umulhi((unsigned)a, magic); }

template <typename T, int R>
__device__ __forceinline__ void rt_stage(const cplx<T>* in, cplx<T>* out, int nl, int lg, int ldl, int nb, int Ns,
                                         unsigned mNs, const cplx<T>* __restrict__ tw, int sign)
{
    const T sg = (T)sign;
    const int tstep = Ns > 1 ? fdiv(nb, mNs) : nb;   // n / (Ns R)
    for (int w = threadIdx.x; w < (nb << lg); w += blockDim.x) {
        const int l = w & ((1 << lg) - 1), j = w >> lg;
        if (l >= nl) continue;
        const cplx<T>* src = in + l * ldl + j;
        cplx<T> v[R];
#pragma unroll
        for (int r = 0; r < R; ++r) v[r] = src[r * nb];
        int o = j * R;
        if (Ns > 1) {
            const int jq = fdiv(j, mNs), k = j - jq * Ns;
            o = jq * Ns * R + k;
#pragma unroll
            for (int r = 1; r < R; ++r) v[r] = cmul(v[r], root(tw, r * k * tstep, sign));
        }
        bfly<T, R>(v, sg);
        cplx<T>* dst = out + l * ldl + o;
#pragma unroll
        for (int r = 0; r < R; ++r) dst[r * Ns] = v[r];
    }
}

// A stage of any other prime R (17 and up): the pairs (r, R - r) become their
// sums and differences in place (after the twiddles), then every thread forms
// PQ output pairs q, R - q of one butterfly; the roots are the same for all
// lines (broadcasts), each sum and difference serves PQ outputs.
// 122 = 61 * 2, FP64, 122x122x101, one y pass: 114 us with one thread per
// output and a modulo per term, 20 us so (the x passes 88 and 84, now 24 and 21).
template <typename T>
__device__ __forceinline__ void rt_prime_stage(cplx<T>* in, cplx<T>* out, int R, int nl, int lg, int ldl, int nb,
                                               unsigned mnb, int Ns, unsigned mNs, const cplx<T>* __restrict__ tw,
                                               int sign)
{
    constexpr int PQ = 4;
    const T sg = (T)sign;
    const int H = R >> 1, tstep = Ns > 1 ? fdiv(nb, mNs) : nb, lm = (1 << lg) - 1;
    for (int w = threadIdx.x; w < ((nb * H) << lg); w += blockDim.x) {
        const int l = w & lm, e = w >> lg, r = fdiv(e, mnb) + (nb == 1 ? e : 0) + 1;
        const int j = nb == 1 ? 0 : e - (r - 1) * nb;
        if (l >= nl) continue;
        cplx<T>* p = in + l * ldl + j;
        cplx<T> a = p[r * nb], b = p[(R - r) * nb];
        if (Ns > 1) {
            const int k = j - fdiv(j, mNs) * Ns;
            a = cmul(a, root(tw, r * k * tstep, sign));
            b = cmul(b, root(tw, (R - r) * k * tstep, sign));
        }
        p[r * nb] = cadd(a, b);
        p[(R - r) * nb] = csub(a, b);
    }
    __syncthreads();
    const int ng = (H + PQ) / PQ;    // groups of PQ outputs over q = 0..H
    for (int w = threadIdx.x; w < ((nb * ng) << lg); w += blockDim.x) {
        const int l = w & lm, e = w >> lg, g = nb == 1 ? e : fdiv(e, mnb), j = e - g * nb;
        if (l >= nl) continue;
        const cplx<T>* p = in + l * ldl + j;
        const cplx<T> x0 = p[0];
        cplx<T> a[PQ], b[PQ];
        int m[PQ], q[PQ];
#pragma unroll
        for (int i = 0; i < PQ; ++i) {
            a[i] = x0;
            b[i] = {(T)0, (T)0};
            q[i] = min(g * PQ + i, H);
            m[i] = 0;
        }
        for (int r = 1; r <= H; ++r) {
            const cplx<T> s = p[r * nb], d = p[(R - r) * nb];
#pragma unroll
            for (int i = 0; i < PQ; ++i) {
                m[i] += q[i];
                m[i] -= m[i] >= R ? R : 0;
                const cplx<T> c = tw[m[i] * nb];   // cos, -sin of 2 pi r q / R
                a[i].x += c.x * s.x;
                a[i].y += c.x * s.y;
                b[i].x -= c.y * d.x;
                b[i].y -= c.y * d.y;
            }
        }
        const int jq = Ns > 1 ? fdiv(j, mNs) : j, k = Ns > 1 ? j - jq * Ns : 0;
        cplx<T>* dst = out + l * ldl + jq * Ns * R + k;
#pragma unroll
        for (int i = 0; i < PQ; ++i) {
            const cplx<T> ib = cis(b[i], sg);
            if (g * PQ + i <= H) {
                dst[q[i] * Ns] = cadd(a[i], ib);
                if (q[i] > 0) dst[(R - q[i]) * Ns] = csub(a[i], ib);
            }
        }
    }
}

// Runs plan pl on the lines A[l*ldl ..], l < nl; returns the buffer (A or B)
// that holds the result.  Unnormalised, sign -1 forward, +1 inverse.  Every
// thread of the block must call it, with A's writes behind a barrier.
template <typename T>
__device__ cplx<T>* rt_fft(cplx<T>* A, cplx<T>* B, const FftPlan& pl, int nl, int lg, int ldl,
                           const cplx<T>* __restrict__ tw, int sign)
{
    cplx<T>* in = A;
    cplx<T>* out = B;
    int Ns = 1;
    for (int st = 0; st < pl.nst; ++st) {
        const int R = pl.rad[st], nb = pl.nb[st];
        const unsigned mNs = pl.mns[st];
        switch (R) {
        case 2: rt_stage<T, 2>(in, out, nl, lg, ldl, nb, Ns, mNs, tw, sign); break;
        case 3: rt_stage<T, 3>(in, out, nl, lg, ldl, nb, Ns, mNs, tw, sign); break;
        case 4: rt_stage<T, 4>(in, out, nl, lg, ldl, nb, Ns, mNs, tw, sign); break;
        case 5: rt_stage<T, 5>(in, out, nl, lg, ldl, nb, Ns, mNs, tw, sign); break;
        case 7: rt_stage<T, 7>(in, out, nl, lg, ldl, nb, Ns, mNs, tw, sign); break;
        case 8: rt_stage<T, 8>(in, out, nl, lg, ldl, nb, Ns, mNs, tw, sign); break;
        case 9: rt_stage<T, 9>(in, out, nl, lg, ldl, nb, Ns, mNs, tw, sign); break;
        case 11: rt_stage<T, 11>(in, out, nl, lg, ldl, nb, Ns, mNs, tw, sign); break;
        case 13: rt_stage<T, 13>(in, out, nl, lg, ldl, nb, Ns, mNs, tw, sign); break;
        case 16: rt_stage<T, 16>(in, out, nl, lg, ldl, nb, Ns, mNs, tw, sign); break;
        default: rt_prime_stage<T>(in, out, R, nl, lg, ldl, nb, pl.mnb[st], Ns, mNs, tw, sign); break;
        }
        __syncthreads();
        cplx<T>* tmp = in;
        in = out;
        out = tmp;
        Ns *= R;
    }
    return in;
}

// A thread's turn over the count elements of a block's contiguous rows of n:
// U loads ld(l, i) in flight, then their stores st(l, i, v); mn = fft_magic(n)
template <int U, typename V, class LD, class ST>
__device__ __forceinline__ void rows_copy(int count, int n, unsigned mn, const LD& ld, const ST& st)
{
    for (int e0 = threadIdx.x; e0 < count; e0 += U * blockDim.x) {
        V v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int e = e0 + u * blockDim.x, l = fdiv(e, mn);
            if (e < count) v[u] = ld(l, e - l * n);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int e = e0 + u * blockDim.x, l = fdiv(e, mn);
            if (e < count) st(l, e - l * n, v[u]);
        }
    }
}

// a compile-time plan needs no argument (and no work on the host)
struct NoPlan {};
template <int N>
using PlanArg = std::conditional_t<(N > 0), NoPlan, FftPlan>;
template <int N>
PlanArg<N> plan_arg(int n)
{
    if constexpr (N > 0) return NoPlan{};
    else return make_fft_plan(n);
}

// Spectral layout (both precisions): [z-1][kx][ky], ky fastest, kx in
// [0, nx/2]: the y transforms run over contiguous lines and the z solve over
// contiguous modes m = kx*ny + ky.

// (1a) R2C along x of s = -q/eps on interior rows, two real rows per complex
// line.  A block takes up to 2*lpb = 2^(lg+1) consecutive rows y0.. of one
// plane (the last block of a plane what is left).  The spectrum is written
// transposed, 2*lpb consecutive ky per kx.
// LDS: twiddles (nx), line buffers (lpb lines; two for the runtime plan).
template <typename T, int N>
__global__ void __launch_bounds__(256) fftx_fwd_kernel(const PoissonJob* __restrict__ jobs,
                                                       const cplx<T>* __restrict__ tw, PlanArg<N> pl, int nx_rt,
                                                       int ny, int lpb, int lg)
{
    const PoissonJob& J = jobs[blockIdx.y];
    const int nx = N > 0 ? N : nx_rt;
    const int nxh = nx / 2 + 1;
    const int ldl = lds_pitch(N, nx);
    extern __shared__ unsigned char smem_raw[];
    cplx<T>* tws = reinterpret_cast<cplx<T>*>(smem_raw);
    cplx<T>* A = tws + nx;
    const int groups = (ny / 2 + lpb - 1) / lpb;
    const int zi = blockIdx.x / groups;              // interior plane index z-1
    if (zi >= J.n) return;                           // a shorter box of the batch
    const int y0 = (blockIdx.x - zi * groups) * 2 * lpb;
    const int nl = min(lpb, (ny - y0) / 2);
    EHD_GLOBAL const T* qp = gptr((const T*)J.q) + (size_t)(zi + 1) * nx * ny + (size_t)y0 * nx;
    EHD_GLOBAL cplx<T>* spec = gptr((cplx<T>*)J.spec);
    const double neps = -1.0 / J.eps;
    for (int i = threadIdx.x; i < nx; i += blockDim.x) tws[i] = tw[i];
    __syncthreads();
    cplx<T>* res;
    if constexpr (N > 0) {
        auto ld = [&](int l, int i) -> cplx<T> {
            return {(T)((double)qp[(size_t)(2 * l) * N + i] * neps),
                    (T)((double)qp[(size_t)(2 * l + 1) * N + i] * neps)};
        };
        auto sf = [](int, int, cplx<T>) {};
        ct_run<T, N, 0, 1, false, false>(ld, sf, A, nl, ldl, tws, -1);
        res = A;
    } else {
        cplx<T>* B = A + lpb * ldl;
        rows_copy<4, cplx<T>>(
            nl * nx, nx, pl.mn,
            [&](int l, int i) -> cplx<T> {
                return {(T)((double)qp[(size_t)(2 * l) * nx + i] * neps),
                        (T)((double)qp[(size_t)(2 * l + 1) * nx + i] * neps)};
            },
            [&](int l, int i, cplx<T> v) { A[l * ldl + i] = v; });
        __syncthreads();
        res = rt_fft<T>(A, B, pl, nl, lg, ldl, tws, -1);
    }
    const int rows = 2 << lg;
    EHD_GLOBAL cplx<T>* out = spec + (size_t)zi * nxh * ny + y0;
    for (int w = threadIdx.x; w < nxh * rows; w += blockDim.x) {
        const int k = w >> (lg + 1), r = w & (rows - 1);
        if (r >= 2 * nl) continue;
        const int l = r >> 1;
        const int kn = (nx - k) % nx;
        const cplx<T> zk = res[l * ldl + (N > 0 ? padi(k) : k)];
        const cplx<T> zn = res[l * ldl + (N > 0 ? padi(kn) : kn)];
        // A_k = (Z_k + conj Z_{n-k})/2 (row 2l), B_k = (Z_k - conj Z_{n-k})/(2i) (row 2l+1)
        const cplx<T> v = (r & 1) ? cplx<T>{(T)0.5 * (zk.y + zn.y), (T)-0.5 * (zk.x - zn.x)}
                                  : cplx<T>{(T)0.5 * (zk.x + zn.x), (T)0.5 * (zk.y - zn.y)};
        stc(out + (size_t)k * ny + r, v);
    }
}

// (1b)/(3a) complex DFT along y, in place, over contiguous lines of ny.
// A block takes G consecutive lines.
template <typename T, int N>
__global__ void __launch_bounds__(256) ffty_kernel(const PoissonJob* __restrict__ jobs, const cplx<T>* __restrict__ tw,
                                                   PlanArg<N> pl, int ny_rt, int nxh, int G, int lg, int sign)
{
    const PoissonJob& J = jobs[blockIdx.y];
    const int ny = N > 0 ? N : ny_rt;
    const int ldl = lds_pitch(N, ny);
    extern __shared__ unsigned char smem_raw[];
    cplx<T>* tws = reinterpret_cast<cplx<T>*>(smem_raw);
    cplx<T>* A = tws + ny;
    const int nlines = J.n * nxh;
    const int L0 = blockIdx.x * G;
    if (L0 >= nlines) return;                        // a shorter box of the batch
    const int nl = min(G, nlines - L0);
    EHD_GLOBAL cplx<T>* base = gptr((cplx<T>*)J.spec) + (size_t)L0 * ny;
    for (int i = threadIdx.x; i < ny; i += blockDim.x) tws[i] = tw[i];
    __syncthreads();
    if constexpr (N > 0) {
        auto ld = [&](int l, int i) -> cplx<T> { return ldc(base + (size_t)l * N + i); };
        auto sf = [&](int l, int i, cplx<T> v) { stc(base + (size_t)l * N + i, v); };
        ct_run<T, N, 0, 1, false, true>(ld, sf, A, nl, ldl, tws, sign);
    } else {
        cplx<T>* B = A + G * ldl;
        rows_copy<4, cplx<T>>(
            nl * ny, ny, pl.mn, [&](int l, int i) { return ldc(base + (size_t)l * ny + i); },
            [&](int l, int i, cplx<T> v) { A[l * ldl + i] = v; });
        __syncthreads();
        cplx<T>* res = rt_fft<T>(A, B, pl, nl, lg, ldl, tws, sign);
        rows_copy<4, cplx<T>>(
            nl * ny, ny, pl.mn, [&](int l, int i) { return res[l * ldl + i]; },
            [&](int l, int i, cplx<T> v) { stc(base + (size_t)l * ny + i, v); });
    }
}

// (2) per-mode tridiagonal solve along z, FP64, by the partition method.
// For each (kx,ky) mode the system is x[k-1] + b x[k] + x[k+1] = dz^2 s[k],
// k = 0..n-1, x[-1] = x[n] = 0, b = -(2 + k^2 dz^2).  A block holds MB =
// NT/P modes and P threads per mode, each owning a chunk of at most MAXM
// (<= ZS_MAXM) consecutive k; the threads of a wave hold consecutive modes,
// so every load and store of a chunk row is a contiguous run of modes.  Each
// thread loads its chunk straight into registers and solves with the
// chunk's own matrix T (Thomas)
//   T y = r,  T v = e_first,  (T w = e_last, w = reverse of v for Toeplitz T),
// so that x = y - x_left v - x_right w.  The interface unknowns (first and
// last x of every chunk) obey three recurrences along the chunks:
//   be_q = -vf_q - vl_q^2 be_{q-1} / (1 + vf_q be_{q-1})  (pivots),
//   ar_q = al_q + bt_q ar_{q-1},   xf_q = gr_q + de_q xf_{q+1}
// (vf, vl the first and last entries of the chunk's v), after which every
// chunk has its neighbours x_l(q-1) = ar_{q-1} + be_{q-1} xf_q and x_f(q+1)
// and finishes independently.  Per-chunk records go through LDS, fields
// outermost and modes innermost, so the threads of a wave hit consecutive
// banks.  Two ways to solve the recurrences:
// - FP64 spectrum (the parity path): one thread per mode runs them in order.
// - FP32 spectrum: three doubling (Hillis-Steele) scans over the P threads of
//   the mode: prefix products of the Moebius matrices
//   M_q = [[vl^2 - vf^2, -vf], [vf, 1]], be_q = N_q / D_q with
//   [N_q; D_q] = M_q [N_{q-1}; D_{q-1}], rescaled by powers of two; an affine
//   prefix for ar; an affine suffix for xf.  25 -> 21.5 us on the 256x256x128
//   FP32 spectrum.  The composed matrices lose more to rounding than the
//   ordered recurrence: against the oracle at 64x48x200 the FP64 solve was
//   7e-13 with scans and 3e-14 in order, so the FP64 spectrum keeps the order.
//   Rounded to float the two agree.
// LDS: 6 P MB doubles.
constexpr int ZS_MAXM = 16;

thread_local const char* g_failed_pass = "";

template <typename T, int P, int MAXM, int NT = 256>
__global__ void __launch_bounds__(NT) zsolve_kernel(const PoissonJob* __restrict__ jobs, int nmodes, int ny,
                                                      int split_mean, double inv_nxy)
{
    constexpr int MB = NT / P;
    const PoissonJob& J = jobs[blockIdx.y];
    EHD_GLOBAL cplx<T>* __restrict__ spec = gptr((cplx<T>*)J.spec);
    EHD_GLOBAL double* __restrict__ phibar = gptr(J.phibar);
    const int n = J.n;
    const double kxs = J.kxs, kys = J.kys, dz2 = J.dz2, voltage = J.voltage;
    extern __shared__ unsigned char smem_raw[];
    double* sc = reinterpret_cast<double*>(smem_raw);   // [6][P][MB] chunk records
    auto Y = [&](int f, int q, int cc) -> double& { return sc[(f * P + q) * MB + cc]; };
    const int m0 = blockIdx.x * MB;
    const int nm = min(MB, nmodes - m0);
    const int c = threadIdx.x % MB, p = threadIdx.x / MB;
    const int m = m0 + c;
    const int Peff = min(P, n);
    const bool active = (c < nm) && (p < Peff);
    const int k0 = (p * n) / Peff, len = ((p + 1) * n) / Peff - k0;
    T sx[MAXM], sy[MAXM];
#pragma unroll
    for (int i = 0; i < MAXM; ++i) {
        sx[i] = (T)0;
        sy[i] = (T)0;
        if (active && i < len) {
            const cplx<T> v = ldc(spec + (size_t)(k0 + i) * nmodes + m);
            sx[i] = v.x;
            sy[i] = v.y;
        }
    }
    const int kxi = m / ny, kyi = m - kxi * ny;
    const double kxv = kxi * kxs, kyv = (kyi <= ny / 2 ? kyi : kyi - ny) * kys;
    const double bd = -(2.0 + (kxv * kxv + kyv * kyv) * dz2);
    double cp[MAXM], yr[MAXM], yi[MAXM], v[MAXM];
    double e0 = 0.0, e1 = 0.0, e2 = 0.0, e3 = 0.0, vf = 0.0, vlq = 0.0;
    if (active) {
#pragma unroll
        for (int i = 0; i < MAXM; ++i) {
            if (i < len) {
                const double den = (i == 0) ? 1.0 / bd : 1.0 / (bd - cp[i - 1]);
                cp[i] = den;
                const double rr = dz2 * (double)sx[i], ri = dz2 * (double)sy[i];
                yr[i] = (i == 0 ? rr : rr - yr[i - 1]) * den;
                yi[i] = (i == 0 ? ri : ri - yi[i - 1]) * den;
                v[i] = (i == 0 ? 1.0 : -v[i - 1]) * den;
            }
        }
#pragma unroll
        for (int i = MAXM - 2; i >= 0; --i) {
            if (i < len - 1) {
                yr[i] -= cp[i] * yr[i + 1];
                yi[i] -= cp[i] * yi[i + 1];
                v[i] -= cp[i] * v[i + 1];
            }
        }
#pragma unroll
        for (int i = 0; i < MAXM; ++i)
            if (i == len - 1) {
                e2 = yr[i];
                e3 = yi[i];
                vlq = v[i];
            }
        e0 = yr[0]; e1 = yi[0]; vf = v[0];
    }
    double Lr = 0.0, Li = 0.0, Rr = 0.0, Ri = 0.0;
    if constexpr (sizeof(T) == sizeof(float)) {
        // (1) be_q = N_q / D_q, [N_q; D_q] = M_q [N_{q-1}; D_{q-1}], M_q = [[vl^2 - vf^2, -vf], [vf, 1]]:
        //     inclusive prefix products of the M by a doubling scan (identity for inactive chunks)
        double a = 1.0, b = 0.0, cc2 = 0.0, d = 1.0;
        if (active) { a = vlq * vlq - vf * vf; b = -vf; cc2 = vf; d = 1.0; }
#pragma unroll
        for (int off = 1; off < P; off <<= 1) {
            Y(0, p, c) = a; Y(1, p, c) = b; Y(2, p, c) = cc2; Y(3, p, c) = d;
            __syncthreads();
            if (p >= off) {
                const double a2 = Y(0, p - off, c), b2 = Y(1, p - off, c), c2 = Y(2, p - off, c), d2 = Y(3, p - off, c);
                const double na = a * a2 + b * c2, nb = a * b2 + b * d2, nc = cc2 * a2 + d * c2, nd = cc2 * b2 + d * d2;
                const double mx = fmax(fmax(fabs(na), fabs(nb)), fmax(fabs(nc), fabs(nd)));
                const int e = __builtin_amdgcn_frexp_exp(mx);
                a = ldexp(na, -e); b = ldexp(nb, -e); cc2 = ldexp(nc, -e); d = ldexp(nd, -e);
            }
            __syncthreads();
        }
        // exclusive value (N_{p-1}, D_{p-1}) = P_{p-1} [0; 1]
        Y(0, p, c) = b; Y(1, p, c) = d;
        __syncthreads();
        const double Nq = (p > 0) ? Y(0, p - 1, c) : 0.0, Dq = (p > 0) ? Y(1, p - 1, c) : 1.0;
        __syncthreads();
        double den = 0.0, de = 0.0, be = 0.0, al = 0.0, ali = 0.0, bt = 1.0;
        if (active) {
            const double inv = 1.0 / (Dq + vf * Nq);
            den = Dq * inv;
            const double bden = Nq * inv;
            de = -vlq * den;
            be = vlq * vlq * bden - vf;
            al = e2 - vlq * bden * e0;
            ali = e3 - vlq * bden * e1;
            bt = -vlq * den;
        } else {
            bt = 1.0; al = 0.0; ali = 0.0;
        }
        // (2) ar_q = al_q + bt_q ar_{q-1}: doubling scan of affine maps (identity for inactive chunks)
        double sa = al, sai = ali, sb = bt;
#pragma unroll
        for (int off = 1; off < P; off <<= 1) {
            Y(0, p, c) = sa; Y(1, p, c) = sai; Y(2, p, c) = sb;
            __syncthreads();
            if (p >= off) {
                const double pa = Y(0, p - off, c), pai = Y(1, p - off, c), pb = Y(2, p - off, c);
                sa = sa + sb * pa;
                sai = sai + sb * pai;
                sb = sb * pb;
            }
            __syncthreads();
        }
        // sa = ar_p; exclusive ar_{p-1} from the left neighbour
        Y(0, p, c) = sa; Y(1, p, c) = sai;
        __syncthreads();
        const double arp = (p > 0) ? Y(0, p - 1, c) : 0.0, aip = (p > 0) ? Y(1, p - 1, c) : 0.0;
        __syncthreads();
        const double gr = active ? (e0 - vf * arp) * den : 0.0, gi = active ? (e1 - vf * aip) * den : 0.0;
        // (3) xf_q = gr_q + de_q xf_{q+1}, xf_Peff = 0: doubling scan from the right
        double xa = gr, xai = gi, xb = active ? de : 1.0;
#pragma unroll
        for (int off = 1; off < P; off <<= 1) {
            Y(0, p, c) = xa; Y(1, p, c) = xai; Y(2, p, c) = xb;
            __syncthreads();
            if (p + off < P) {
                const double na = Y(0, p + off, c), nai = Y(1, p + off, c), nb = Y(2, p + off, c);
                xa = xa + xb * na;
                xai = xai + xb * nai;
                xb = xb * nb;
            }
            __syncthreads();
        }
        // xa = x_f(p); neighbours: x_f(p+1) from the right, x_l(p-1) = ar_{p-1} + be_{p-1} x_f(p)
        Y(0, p, c) = xa; Y(1, p, c) = xai; Y(2, p, c) = be;
        __syncthreads();
        Rr = (p + 1 < Peff) ? Y(0, p + 1, c) : 0.0;
        Ri = (p + 1 < Peff) ? Y(1, p + 1, c) : 0.0;
        const double bem = (p > 0) ? Y(2, p - 1, c) : 0.0;
        Lr = (p > 0) ? arp + bem * xa : 0.0;
        Li = (p > 0) ? aip + bem * xai : 0.0;
    } else {
        if (active) {
            Y(0, p, c) = e0; Y(1, p, c) = e1; Y(2, p, c) = e2; Y(3, p, c) = e3; Y(4, p, c) = vf;
            Y(5, p, c) = vlq;
        }
        __syncthreads();
        if (p == 0 && c < nm) {
            double ar = 0.0, ai = 0.0, be = 0.0;
#pragma unroll
            for (int qq = 0; qq < P; ++qq) {
                if (qq >= Peff) break;
                const double f0 = Y(0, qq, c), f1 = Y(1, qq, c), f2 = Y(2, qq, c), f3 = Y(3, qq, c);
                const double wl = Y(4, qq, c), wf = Y(5, qq, c);   // w reversed v: w_l = v_f, w_f = v_l
                const double dn = 1.0 / (1.0 + wl * be);
                const double gr = (f0 - wl * ar) * dn;
                const double gi = (f1 - wl * ai) * dn;
                const double de = -wf * dn;
                const double nar = f2 - wf * ar - wf * be * gr;
                const double nai = f3 - wf * ai - wf * be * gi;
                const double nbe = -wf * be * de - wl;
                ar = nar; ai = nai; be = nbe;
                Y(0, qq, c) = gr; Y(1, qq, c) = gi; Y(2, qq, c) = de; Y(3, qq, c) = ar; Y(4, qq, c) = ai;
                Y(5, qq, c) = be;
            }
            // back: record q gets (x_l(q-1), x_f(q+1)) in fields 0..3, written
            // after the record's own coefficients are read
            double xfr = 0.0, xfi = 0.0;
#pragma unroll
            for (int qq = P - 1; qq >= 0; --qq) {
                if (qq >= Peff) continue;
                const double gr = Y(0, qq, c), gi = Y(1, qq, c), de = Y(2, qq, c);
                const double ar = Y(3, qq, c), ai = Y(4, qq, c), be = Y(5, qq, c);
                const double xlr = ar + be * xfr, xli = ai + be * xfi;
                Y(2, qq, c) = xfr;
                Y(3, qq, c) = xfi;
                if (qq + 1 < Peff) {
                    Y(0, qq + 1, c) = xlr;
                    Y(1, qq + 1, c) = xli;
                }
                const double nxr = gr + de * xfr, nxi = gi + de * xfi;
                xfr = nxr;
                xfi = nxi;
            }
            Y(0, 0, c) = 0.0;
            Y(1, 0, c) = 0.0;
        }
        __syncthreads();
        if (active) {
            Lr = Y(0, p, c); Li = Y(1, p, c); Rr = Y(2, p, c); Ri = Y(3, p, c);
        }
    }
    if (active) {
        double wn = 0.0;
#pragma unroll
        for (int i = MAXM - 1; i >= 0; --i) {
            if (i < len) {
                const double wi = (i == len - 1) ? cp[i] : -cp[i] * wn;
                wn = wi;
                const double xr = yr[i] - Lr * v[i] - Rr * wi;
                const double xi = yi[i] - Li * v[i] - Ri * wi;
                EHD_GLOBAL cplx<T>* dst = spec + (size_t)(k0 + i) * nmodes + m;
                if (split_mean && m == 0) {
                    const int z = k0 + i + 1;
                    phibar[z] = voltage * (1.0 - (double)z / (double)(n + 1)) + xr * inv_nxy;
                    stc(dst, cplx<T>{(T)0, (T)0});
                } else {
                    stc(dst, cplx<T>{(T)xr, (T)xi});
                }
            }
        }
    }
    if (split_mean && m0 == 0 && threadIdx.x == 0) {
        phibar[0] = voltage;
        phibar[n + 1] = 0.0;
    }
}

// Dirichlet values of the potential on the walls (odd_extract,
// poisson.cu:158-165) for the rows first .. first + count of a plane, beside the
// first and the last interior plane (FP64; FP32S keeps them in the plane means)
template <typename T>
__device__ __forceinline__ void wall_rows(EHD_GLOBAL T* phi, int zi, int n, int nx, int ny, int first, int count,
                                          double voltage)
{
    for (int w = 0; w < 2; ++w) {
        if (zi != (w ? n - 1 : 0)) continue;
        EHD_GLOBAL T* p = phi + (size_t)(w ? n + 1 : 0) * nx * ny + (size_t)first * nx;
        for (int i = threadIdx.x; i < count * nx; i += blockDim.x) p[i] = w ? (T)0 : (T)voltage;
    }
}

// (3b) C2R along x, two real rows per complex line, scaled by 1/(nx*ny), plus
// the wall potential (F64) or nothing (FP32S fluctuation).  A block takes up
// to 2*lpb consecutive rows y0.. of one plane; the transposed spectrum is read
// as (row 2l, row 2l+1) pairs, coalesced along ky, and rebuilt in LDS as
// Z = A + i B with the Hermitian half.
template <typename T, int N>
__global__ void __launch_bounds__(256) fftx_inv_kernel(const PoissonJob* __restrict__ jobs,
                                                       const cplx<T>* __restrict__ tw, PlanArg<N> pl, int nx_rt,
                                                       int ny, int lpb, int lg, int add_linear)
{
    const PoissonJob& J = jobs[blockIdx.y];
    const int nx = N > 0 ? N : nx_rt;
    const int nxh = nx / 2 + 1;
    const int ldl = lds_pitch(N, nx);
    extern __shared__ unsigned char smem_raw[];
    cplx<T>* tws = reinterpret_cast<cplx<T>*>(smem_raw);
    cplx<T>* A = tws + nx;
    const int groups = (ny / 2 + lpb - 1) / lpb;
    const int zi = blockIdx.x / groups;
    if (zi >= J.n) return;                           // a shorter box of the batch
    const int y0 = (blockIdx.x - zi * groups) * 2 * lpb;
    const int nl = min(lpb, (ny - y0) / 2);
    const int z = zi + 1;
    const int nz = J.n + 2;
    const double voltage = J.voltage;
    EHD_GLOBAL const cplx<T>* spec = gptr((const cplx<T>*)J.spec);
    EHD_GLOBAL T* phi = gptr((T*)J.phi);
    for (int i = threadIdx.x; i < nx; i += blockDim.x) tws[i] = tw[i];
    EHD_GLOBAL const cplx<T>* in = spec + (size_t)zi * nxh * ny + y0;
    // XI_LOADS row pairs in flight per thread before the LDS stores
    constexpr int XI_LOADS = 4;
    // lanes beyond a last block's lines fill theirs with copies of its last one
    const int lanes = 1 << lg;
    for (int w0 = threadIdx.x; w0 < nxh * lanes; w0 += blockDim.x * XI_LOADS) {
        cplx<T> av[XI_LOADS], bv[XI_LOADS];
#pragma unroll
        for (int u = 0; u < XI_LOADS; ++u) {
            const int w = w0 + u * blockDim.x;
            const int k = w >> lg, l = min(w & (lanes - 1), nl - 1);
            if (w < nxh * lanes) {
                av[u] = ldc(in + (size_t)k * ny + 2 * l);
                bv[u] = ldc(in + (size_t)k * ny + 2 * l + 1);
            }
        }
#pragma unroll
        for (int u = 0; u < XI_LOADS; ++u) {
            const int w = w0 + u * blockDim.x;
            const int k = w >> lg, l = w & (lanes - 1);
            if (w < nxh * lanes) {
                cplx<T> a = av[u], b = bv[u];
                if (k == 0 || 2 * k == nx) {
                    a.y = (T)0;
                    b.y = (T)0;
                }
                // Z_k = A_k + i B_k; Z_{n-k} = conj(A_k) + i conj(B_k)
                A[l * ldl + (N > 0 ? padi(k) : k)] = {a.x - b.y, a.y + b.x};
                if (k > 0 && 2 * k < nx) {
                    const int kn = nx - k;
                    A[l * ldl + (N > 0 ? padi(kn) : kn)] = {a.x + b.y, b.x - a.y};
                }
            }
        }
    }
    __syncthreads();
    const double inv = 1.0 / ((double)nx * (double)ny);
    const double lin = add_linear ? voltage * (1.0 - (double)z / (double)(nz - 1)) : 0.0;
    EHD_GLOBAL T* row0 = phi + (size_t)z * nx * ny + (size_t)y0 * nx;
    if (add_linear) wall_rows(phi, zi, J.n, nx, ny, y0, 2 * nl, voltage);
    if constexpr (N > 0) {
        auto ld = [&](int l, int i) -> cplx<T> { return A[l * ldl + padi(i)]; };
        auto sf = [&](int l, int i, cplx<T> v) {
            row0[(size_t)(2 * l) * N + i] = (T)((double)v.x * inv + lin);
            row0[(size_t)(2 * l + 1) * N + i] = (T)((double)v.y * inv + lin);
        };
        ct_run<T, N, 0, 1, true, true>(ld, sf, A, nl, ldl, tws, +1);
    } else {
        cplx<T>* B = A + lpb * ldl;
        cplx<T>* res = rt_fft<T>(A, B, pl, nl, lg, ldl, tws, +1);
        rows_copy<4, cplx<T>>(
            nl * nx, nx, pl.mn, [&](int l, int i) { return res[l * ldl + i]; },
            [&](int l, int i, cplx<T> v) {
                row0[(size_t)(2 * l) * nx + i] = (T)((double)v.x * inv + lin);
                row0[(size_t)(2 * l + 1) * nx + i] = (T)((double)v.y * inv + lin);
            });
    }
}

// (1) and (3) for a small plane in one launch each: a block holds a whole
// plane, transforms its row pairs, turns them into the nx/2+1 lines along y in
// LDS and transforms those, or the other way round.  The same line programs
// and, in the planes that with_plane admits, the same plan as the separate
// passes, so the same numbers bit for bit.  Two launches and a spectrum round
// trip less: solves back to back, five launches / three, FP32S 32x32x16 16.6 /
// 13.1 us, 64x64x64 22.3 / 16.9; FP64 64x64x32 26.1 / 20.6 us.
constexpr int kPlaneThreads = 512;

// A sign that the compiler does not know: the y pass takes its as an
// argument, and with a constant one the conjugated twiddles' products are
// fused into their sums the other way round, which moves the last bit.
__device__ __forceinline__ int unknown_sign(int s)
{
    asm("" : "+s"(s));
    return s;
}

constexpr int plane_pitch(int N, int n) { return N > 0 ? (padi(N - 1) + 1) | 1 : n | 1; }

// lines and elements of the two LDS buffers of a plane
template <int N>
struct PlaneBufs {
    int ldx, ldy, size;      // pitches, elements per buffer
    __host__ __device__ PlaneBufs(int nx, int ny)
        : ldx(plane_pitch(N, nx)), ldy(plane_pitch(N, ny)),
          size((ny / 2) * ldx > (nx / 2 + 1) * ldy ? (ny / 2) * ldx : (nx / 2 + 1) * ldy)
    {
    }
};

template <typename T, int N>
__global__ void __launch_bounds__(kPlaneThreads) plane_fwd_kernel(const PoissonJob* __restrict__ jobs,
                                                                  const cplx<T>* __restrict__ twx,
                                                                  const cplx<T>* __restrict__ twy, PlanArg<N> plx,
                                                                  PlanArg<N> ply, int nx_rt, int ny_rt, int lgx,
                                                                  int lgy)
{
    const PoissonJob& J = jobs[blockIdx.y];
    const int zi = blockIdx.x;
    if (zi >= J.n) return;                           // a shorter box of the batch
    const int nx = N > 0 ? N : nx_rt, ny = N > 0 ? N : ny_rt, nxh = nx / 2 + 1, nl = ny / 2;
    const PlaneBufs<N> pb(nx, ny);
    extern __shared__ unsigned char smem_raw[];
    cplx<T>* tx = reinterpret_cast<cplx<T>*>(smem_raw);
    cplx<T>* ty = tx + nx;
    cplx<T>* A = ty + ny;
    cplx<T>* B = A + pb.size;
    EHD_GLOBAL const T* qp = gptr((const T*)J.q) + (size_t)(zi + 1) * nx * ny;
    EHD_GLOBAL cplx<T>* out = gptr((cplx<T>*)J.spec) + (size_t)zi * nxh * ny;
    const double neps = -1.0 / J.eps;
    for (int i = threadIdx.x; i < nx; i += blockDim.x) tx[i] = twx[i];
    for (int i = threadIdx.x; i < ny; i += blockDim.x) ty[i] = twy[i];
    auto row_pair = [&](int l, int i) -> cplx<T> {
        return {(T)((double)qp[(size_t)(2 * l) * nx + i] * neps), (T)((double)qp[(size_t)(2 * l + 1) * nx + i] * neps)};
    };
    cplx<T>* res = A;
    if constexpr (N > 0) {
        __syncthreads();
        auto sf = [](int, int, cplx<T>) {};
        ct_run<T, N, 0, 1, false, false>(row_pair, sf, A, nl, pb.ldx, tx, -1);
    } else {
        rows_copy<4, cplx<T>>(nl * nx, nx, plx.mn, row_pair,
                              [&](int l, int i, cplx<T> v) { A[l * pb.ldx + i] = v; });
        __syncthreads();
        res = rt_fft<T>(A, B, plx, nl, lgx, pb.ldx, tx, -1);
    }
    // the lines along y: as fftx_fwd_kernel writes them, into the other buffer
    cplx<T>* lines = res == A ? B : A;
    const int lanes = 1 << lgx;
    for (int w = threadIdx.x; w < nxh * lanes; w += blockDim.x) {
        const int k = w >> lgx, l = w & (lanes - 1);
        if (l >= nl) continue;
        const int kn = k == 0 ? 0 : nx - k;
        const cplx<T> zk = res[l * pb.ldx + (N > 0 ? padi(k) : k)], zn = res[l * pb.ldx + (N > 0 ? padi(kn) : kn)];
        cplx<T>* p = lines + k * pb.ldy;
        p[N > 0 ? padi(2 * l) : 2 * l] = {(T)0.5 * (zk.x + zn.x), (T)0.5 * (zk.y - zn.y)};
        p[N > 0 ? padi(2 * l + 1) : 2 * l + 1] = {(T)0.5 * (zk.y + zn.y), (T)-0.5 * (zk.x - zn.x)};
    }
    __syncthreads();
    if constexpr (N > 0) {
        auto ld = [&](int l, int i) -> cplx<T> { return lines[l * pb.ldy + padi(i)]; };
        auto sf = [&](int l, int i, cplx<T> v) { stc(out + (size_t)l * N + i, v); };
        ct_run<T, N, 0, 1, true, true>(ld, sf, lines, nxh, pb.ldy, ty, unknown_sign(-1));
    } else {
        const cplx<T>* r = rt_fft<T>(lines, res, ply, nxh, lgy, pb.ldy, ty, unknown_sign(-1));
        rows_copy<4, cplx<T>>(
            nxh * ny, ny, ply.mn, [&](int l, int i) { return r[l * pb.ldy + i]; },
            [&](int l, int i, cplx<T> v) { stc(out + (size_t)l * ny + i, v); });
    }
}

template <typename T, int N>
__global__ void __launch_bounds__(kPlaneThreads) plane_inv_kernel(const PoissonJob* __restrict__ jobs,
                                                                  const cplx<T>* __restrict__ twx,
                                                                  const cplx<T>* __restrict__ twy, PlanArg<N> plx,
                                                                  PlanArg<N> ply, int nx_rt, int ny_rt, int lgx,
                                                                  int lgy, int add_linear)
{
    const PoissonJob& J = jobs[blockIdx.y];
    const int zi = blockIdx.x;
    if (zi >= J.n) return;                           // a shorter box of the batch
    const int nx = N > 0 ? N : nx_rt, ny = N > 0 ? N : ny_rt, nxh = nx / 2 + 1, nl = ny / 2;
    const PlaneBufs<N> pb(nx, ny);
    extern __shared__ unsigned char smem_raw[];
    cplx<T>* tx = reinterpret_cast<cplx<T>*>(smem_raw);
    cplx<T>* ty = tx + nx;
    cplx<T>* A = ty + ny;
    cplx<T>* B = A + pb.size;
    EHD_GLOBAL const cplx<T>* in = gptr((const cplx<T>*)J.spec) + (size_t)zi * nxh * ny;
    EHD_GLOBAL T* phi = gptr((T*)J.phi);
    for (int i = threadIdx.x; i < nx; i += blockDim.x) tx[i] = twx[i];
    for (int i = threadIdx.x; i < ny; i += blockDim.x) ty[i] = twy[i];
    auto line = [&](int l, int i) -> cplx<T> { return ldc(in + (size_t)l * ny + i); };
    cplx<T>* res = A;
    if constexpr (N > 0) {
        __syncthreads();
        auto sf = [](int, int, cplx<T>) {};
        ct_run<T, N, 0, 1, false, false>(line, sf, A, nxh, pb.ldy, ty, unknown_sign(+1));
    } else {
        rows_copy<4, cplx<T>>(nxh * ny, ny, ply.mn, line, [&](int l, int i, cplx<T> v) { A[l * pb.ldy + i] = v; });
        __syncthreads();
        res = rt_fft<T>(A, B, ply, nxh, lgy, pb.ldy, ty, unknown_sign(+1));
    }
    // the row pairs: as fftx_inv_kernel builds them, into the other buffer
    cplx<T>* rows = res == A ? B : A;
    const int lanes = 1 << lgx;
    for (int w = threadIdx.x; w < nxh * lanes; w += blockDim.x) {
        const int k = w >> lgx, l = w & (lanes - 1);
        if (l >= nl) continue;
        const cplx<T>* p = res + k * pb.ldy;
        cplx<T> a = p[N > 0 ? padi(2 * l) : 2 * l], b = p[N > 0 ? padi(2 * l + 1) : 2 * l + 1];
        if (k == 0 || 2 * k == nx) {
            a.y = (T)0;
            b.y = (T)0;
        }
        cplx<T>* z = rows + l * pb.ldx;
        z[N > 0 ? padi(k) : k] = {a.x - b.y, a.y + b.x};
        if (k > 0 && 2 * k < nx) z[N > 0 ? padi(nx - k) : nx - k] = {a.x + b.y, b.x - a.y};
    }
    __syncthreads();
    const double inv = 1.0 / ((double)nx * (double)ny);
    const double lin = add_linear ? J.voltage * (1.0 - (double)(zi + 1) / (double)(J.n + 1)) : 0.0;
    EHD_GLOBAL T* row0 = phi + (size_t)(zi + 1) * nx * ny;
    if (add_linear) wall_rows(phi, zi, J.n, nx, ny, 0, ny, J.voltage);
    auto put = [&](int l, int i, cplx<T> v) {
        row0[(size_t)(2 * l) * nx + i] = (T)((double)v.x * inv + lin);
        row0[(size_t)(2 * l + 1) * nx + i] = (T)((double)v.y * inv + lin);
    };
    if constexpr (N > 0) {
        auto ld = [&](int l, int i) -> cplx<T> { return rows[l * pb.ldx + padi(i)]; };
        ct_run<T, N, 0, 1, true, true>(ld, put, rows, nl, pb.ldx, tx, +1);
    } else {
        const cplx<T>* r = rt_fft<T>(rows, res, plx, nl, lgx, pb.ldx, tx, +1);
        rows_copy<4, cplx<T>>(nl * nx, nx, plx.mn, [&](int l, int i) { return r[l * pb.ldx + i]; }, put);
    }
}

// The tables of a solve, made where they are used: the roots exp(-2 pi i j/n)
// of both sides, in FP64 by sincospi (the argument exact but for one rounding)
// and rounded to the path's type, and the one-entry job table.  Uploaded from
// the host they cost a call without workspace of its own three small copies
// and a wait in between: ehd_poisson_noalloc at 64x64x32 53.8 -> 35.9 us, at
// 256x256x128 172.7 -> 150.6 us.
template <typename T>
__global__ void __launch_bounds__(256) setup_kernel(PoissonJob job, PoissonJob* dst, cplx<T>* twx, int nx,
                                                    cplx<T>* twy, int ny)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0) *dst = job;
    if (i >= nx + ny) return;
    const int n = i < nx ? nx : ny, j = i < nx ? i : i - nx;
    double s, c;
    sincospi(2.0 * (double)j / (double)n, &s, &c);
    (i < nx ? twx : twy)[j] = {(T)c, (T)-s};
}

constexpr size_t kMaxLds = 65536;

int pow2_floor(int v)
{
    int p = 1;
    while (2 * p <= v) p *= 2;
    return p;
}

// Lines per block of a pass that fit its LDS and, with a compile-time plan,
// one butterfly per thread and stage; a power of two (the lanes count lines
// by shifts), at most 16 with a runtime plan.  0: not even one line fits.
template <typename T, int N>
int lines_that_fit(int n)
{
    const size_t cs = sizeof(cplx<T>);
    const int ldl = lds_pitch(N, n), bufs = N > 0 ? 1 : 2;
    int l = N > 0 ? pow2_floor(256 / ct_max_nb(N > 0 ? N : 1)) : 16;
    while (l > 0 && (size_t)n * cs + (size_t)bufs * l * ldl * cs > kMaxLds) l /= 2;
    return l;
}

// Largest line count per block for an x pass: the power of two that holds a
// plane's ny/2 row pairs cut evenly among as few blocks as fit.
template <typename T, int N>
int x_lines_per_block(int nx, int ny)
{
    const int fit = lines_that_fit<T, N>(nx), half = ny / 2;
    if (fit == 0) return 0;
    const int groups = (half + fit - 1) / fit, l = (half + groups - 1) / groups;
    return pow2_floor(2 * l - 1);
}

template <typename T, int N>
int y_lines_per_block(int ny)
{
    return lines_that_fit<T, N>(ny);
}

// z-solve partition: P (16, 8 or 32) threads per mode with chunks of at most
// ZS_MAXM; fixed by n so that a box gives the same numbers alone and in a
// batch.
// LDS of a z-solve block: six doubles per (chunk, mode), P chunks x 256/P modes
size_t zsolve_lds(int P) { return (size_t)6 * P * (256 / P) * sizeof(double); }

int zsolve_partition(int n, size_t cs)
{
    (void)cs;
    // 16 threads per mode first (measured fastest at n = 126 on the 256x256
    // FP32 spectrum: 21.5 us with scans against 28 us for 32; in order 25 us
    // against 42 us for 8 and 51 us for 32)
    for (int cand : {16, 8, 32})
        if ((n + cand - 1) / cand <= ZS_MAXM && zsolve_lds(cand) <= kMaxLds) return cand;
    return 0;
}

// The passes of a group: each runs the compile-time plan of its own side
// length where there is one, so a box of unequal sides uses one per side.
template <typename T, int N>
hipError_t launch_x(const PoissonGroup& g, bool inverse, hipStream_t st)
{
    static_assert(N == 0 || ct_complete(N), "compile-time sizes must factor into powers of two, 3 and 5");
    const int most = x_lines_per_block<T, N>(g.nx, g.ny);
    if (most == 0 || g.lpb > most) return hipErrorInvalidValue;
    const int lpb = pow2_floor(g.lpb > 0 ? g.lpb : most), lg = __builtin_ctz(lpb);
    const size_t cs = sizeof(cplx<T>);
    const size_t sh = (size_t)g.nx * cs + (size_t)(N > 0 ? 1 : 2) * lpb * lds_pitch(N, g.nx) * cs;
    const dim3 grid(g.max_n * ((g.ny / 2 + lpb - 1) / lpb), g.njobs);
    const PlanArg<N> pl = plan_arg<N>(g.nx);
    const cplx<T>* tw = (const cplx<T>*)g.twx;
    if (inverse)
        fftx_inv_kernel<T, N><<<grid, 256, sh, st>>>(g.jobs, tw, pl, g.nx, g.ny, lpb, lg, g.split_mean ? 0 : 1);
    else
        fftx_fwd_kernel<T, N><<<grid, 256, sh, st>>>(g.jobs, tw, pl, g.nx, g.ny, lpb, lg);
    return hipSuccess;
}

template <typename T, int N>
hipError_t launch_y(const PoissonGroup& g, bool inverse, hipStream_t st)
{
    const int most = y_lines_per_block<T, N>(g.ny), nxh = g.nx / 2 + 1;
    int G = g.ylines > 0 ? g.ylines : most;
    if (most == 0 || G > most) return hipErrorInvalidValue;
    if (N == 0) G = pow2_floor(G);
    const size_t cs = sizeof(cplx<T>);
    const size_t sh = (size_t)g.ny * cs + (size_t)(N > 0 ? 1 : 2) * G * lds_pitch(N, g.ny) * cs;
    const dim3 grid((g.max_n * nxh + G - 1) / G, g.njobs);
    ffty_kernel<T, N><<<grid, 256, sh, st>>>(g.jobs, (const cplx<T>*)g.twy, plan_arg<N>(g.ny), g.ny, nxh, G,
                                            __builtin_ctz(pow2_floor(G)), inverse ? +1 : -1);
    return hipSuccess;
}

int log2_ceil(int v)
{
    int lg = 0;
    while ((1 << lg) < v) ++lg;
    return lg;
}

// Planes of up to 64 x 64 points take the one-launch transforms where their two
// buffers fit.  Larger ones keep too few blocks busy for too long, five launches /
// three: FP32S 96x96x64 26.3 / 39 us, 100x80x64 29.6 / 35.5, 128x128x64 33 / 47
// (62x62x40, the slowest kind of plan within the line, 34.5 / 30.6).
template <typename T, int N>
size_t plane_lds(int nx, int ny)
{
    return ((size_t)nx + ny + 2 * (size_t)PlaneBufs<N>(nx, ny).size) * sizeof(cplx<T>);
}
constexpr int kPlaneMost = 4096;
constexpr size_t kPlaneLds = 80 << 10;   // two blocks per compute unit

template <typename T, int N>
bool plane_fits(int nx, int ny)
{
    if (N > 0 && (nx != ny || (nx / 2 + 1) * ct_max_nb(N > 0 ? N : 1) > kPlaneThreads)) return false;
    return nx * ny <= kPlaneMost && plane_lds<T, N>(nx, ny) <= kPlaneLds;
}

template <typename T, int N>
hipError_t launch_plane(const PoissonGroup& g, bool inverse, hipStream_t st)
{
    const dim3 grid(g.max_n, g.njobs);
    const size_t sh = plane_lds<T, N>(g.nx, g.ny);
    const cplx<T>*twx = (const cplx<T>*)g.twx, *twy = (const cplx<T>*)g.twy;
    const int lgx = log2_ceil(g.ny / 2), lgy = log2_ceil(g.nx / 2 + 1);
    const PlanArg<N> plx = plan_arg<N>(g.nx), ply = plan_arg<N>(g.ny);
    if (sh > kMaxLds) {   // more than a launch may ask for by itself
        const void* kernel = inverse ? (const void*)plane_inv_kernel<T, N> : (const void*)plane_fwd_kernel<T, N>;
        const hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)sh);
        if (e != hipSuccess) return e;
    }
    if (inverse)
        plane_inv_kernel<T, N><<<grid, kPlaneThreads, sh, st>>>(g.jobs, twx, twy, plx, ply, g.nx, g.ny, lgx, lgy,
                                                                g.split_mean ? 0 : 1);
    else
        plane_fwd_kernel<T, N><<<grid, kPlaneThreads, sh, st>>>(g.jobs, twx, twy, plx, ply, g.nx, g.ny, lgx, lgy);
    return hipGetLastError();
}

// f(constant N) with the compile-time plan's length, 0 for a runtime plan
template <class F>
auto with_plan(int n, const F& f)
{
    switch (n) {
    case 32: return f(std::integral_constant<int, 32>{});
    case 48: return f(std::integral_constant<int, 48>{});
    case 64: return f(std::integral_constant<int, 64>{});
    case 80: return f(std::integral_constant<int, 80>{});
    case 96: return f(std::integral_constant<int, 96>{});
    case 128: return f(std::integral_constant<int, 128>{});
    case 256: return f(std::integral_constant<int, 256>{});
    case 512: return f(std::integral_constant<int, 512>{});
    default: return f(std::integral_constant<int, 0>{});
    }
}

// f(constant N) with the plane kernels' plan, if there is one: a plane takes
// them only where both sides run the plan that their passes would run, so that
// the potential is the passes' bit for bit and a run's history does not depend
// on which of the two serves its planes.  That is a square with a compile-time
// plan of powers of two (32 or 64; with a factor of three the forward plane
// kernel fuses other products into sums than the passes do) and two sides
// without one (the runtime plan).  Other pairs are left to the passes, whose
// compile-time plans are mostly the faster ones too: a whole FP32S solve of 9
// interior planes, plane kernels with the runtime plan / passes, 32x64 19.1 /
// 18.3 us, 48x64 20.8 / 18.7, 32x128 21.9 / 18.9, 96x36 22.9 / 21.0; one side
// of 32 or 64 beside a runtime plan 64x40 20.3 / 22.2, 100x32 20.7 / 23.7.
template <typename T, class F>
bool with_plane(int nx, int ny, const F& f)
{
    auto planned = [](int n) { return with_plan(n, [](auto N) { return decltype(N)::value > 0; }); };
    if (nx == 32 && plane_fits<T, 32>(nx, ny)) f(std::integral_constant<int, 32>{});
    else if (nx == 64 && plane_fits<T, 64>(nx, ny)) f(std::integral_constant<int, 64>{});
    else if (!planned(nx) && !planned(ny) && plane_fits<T, 0>(nx, ny)) f(std::integral_constant<int, 0>{});
    else return false;
    return true;
}

// One Poisson solve for every job of a group (same nx, ny, precision; the
// jobs' plane counts may differ): each kernel runs once over the group, the
// job index in blockIdx.y.
template <typename T>
hipError_t poisson_t(const PoissonGroup& g, hipStream_t st)
{
    const int nx = g.nx, ny = g.ny, nxh = nx / 2 + 1;
    const int nmax = g.max_n;
    const size_t cs = sizeof(cplx<T>);
    auto x_pass = [&](bool inverse) {
        return with_plan(nx, [&](auto n) { return launch_x<T, decltype(n)::value>(g, inverse, st); });
    };
    auto y_pass = [&](bool inverse) {
        return with_plan(ny, [&](auto n) { return launch_y<T, decltype(n)::value>(g, inverse, st); });
    };
    // debug_sync: each pass synchronised and checked on its own
    auto check = [&](const char* pass) -> hipError_t {
        if (!g.debug_sync) return hipSuccess;
        hipError_t e = hipGetLastError();
        if (e == hipSuccess) e = hipStreamSynchronize(st);
        if (e != hipSuccess) g_failed_pass = pass;
        return e;
    };
    hipError_t ec = hipSuccess;
    auto plane_pass = [&](bool inverse) {
        if (g.debug_sync == 2) return false;
        return with_plane<T>(nx, ny, [&](auto n) { ec = launch_plane<T, decltype(n)::value>(g, inverse, st); });
    };
    if (plane_pass(false)) {
        if (ec != hipSuccess || (ec = check("forward x and y transforms")) != hipSuccess) return ec;
    } else {
        if ((ec = x_pass(false)) != hipSuccess) return ec;
        if ((ec = check("forward x transform")) != hipSuccess) return ec;
        if ((ec = y_pass(false)) != hipSuccess) return ec;
        if ((ec = check("forward y transform")) != hipSuccess) return ec;
    }

    const int nmodes = nxh * ny;
    const int Pz = zsolve_partition(nmax, cs);
    if (Pz == 0 || Pz != g.zs_partition) return hipErrorInvalidValue;
    const int mb = 256 / Pz;
    const size_t shz = zsolve_lds(Pz);
    const dim3 gz((nmodes + mb - 1) / mb, g.njobs);
    const double inv_nxy = 1.0 / ((double)nx * (double)ny);
    const int sm = g.split_mean;
    // chunk registers sized to the longest chunk: MAXM = 16, 8 or 4
    const int chunk = (nmax + Pz - 1) / Pz;
    hipError_t ez = hipErrorInvalidValue;
    if (Pz == 8) {
        zsolve_kernel<T, 8, 16><<<gz, 256, shz, st>>>(g.jobs, nmodes, ny, sm, inv_nxy);
        ez = hipSuccess;
    } else if (Pz == 16) {
        if (chunk <= 8) zsolve_kernel<T, 16, 8><<<gz, 256, shz, st>>>(g.jobs, nmodes, ny, sm, inv_nxy);
        else zsolve_kernel<T, 16, 16><<<gz, 256, shz, st>>>(g.jobs, nmodes, ny, sm, inv_nxy);
        ez = hipSuccess;
    } else if (Pz == 32) {
        if (chunk <= 4) zsolve_kernel<T, 32, 4><<<gz, 256, shz, st>>>(g.jobs, nmodes, ny, sm, inv_nxy);
        else if (chunk <= 8) zsolve_kernel<T, 32, 8><<<gz, 256, shz, st>>>(g.jobs, nmodes, ny, sm, inv_nxy);
        else zsolve_kernel<T, 32, 16><<<gz, 256, shz, st>>>(g.jobs, nmodes, ny, sm, inv_nxy);
        ez = hipSuccess;
    }
    if (ez != hipSuccess) return ez;
    if ((ec = check("z solve")) != hipSuccess) return ec;

    if (plane_pass(true)) {
        if (ec != hipSuccess || (ec = check("inverse y and x transforms")) != hipSuccess) return ec;
    } else {
        if ((ec = y_pass(true)) != hipSuccess) return ec;
        if ((ec = check("inverse y transform")) != hipSuccess) return ec;
        if ((ec = x_pass(true)) != hipSuccess) return ec;
        if ((ec = check("inverse x transform")) != hipSuccess) return ec;
    }
    return hipGetLastError();
}

template <typename T>
int max_x_lines(int nx, int ny)
{
    return with_plan(nx, [&](auto n) { return x_lines_per_block<T, decltype(n)::value>(nx, ny); });
}

template <typename T>
int max_y_lines(int ny)
{
    return with_plan(ny, [&](auto n) { return y_lines_per_block<T, decltype(n)::value>(ny); });
}

}  // namespace

PoissonJob make_poisson_job(const LbmParams& P, const PoissonBufs& pb, const void* q, void* phi, double voltage,
                            double eps)
{
    PoissonJob j{};
    j.q = q;
    j.spec = pb.spec;
    j.phi = phi;
    j.phibar = pb.phibar;
    j.n = pb.nz - 2;
    j.kxs = 2.0 * 3.14159265358979323846 / (pb.nx * P.dx);
    j.kys = 2.0 * 3.14159265358979323846 / (pb.ny * P.dy);
    j.dz2 = P.dz * P.dz;
    j.eps = eps;
    j.voltage = voltage;
    return j;
}

PoissonShape poisson_shape(Prec prec, int nx, int ny, int nz)
{
    PoissonShape s{};
    const bool f64 = prec == Prec::F64;
    s.max_x_lines = f64 ? max_x_lines<double>(nx, ny) : max_x_lines<float>(nx, ny);
    s.max_y_lines = f64 ? max_y_lines<double>(ny) : max_y_lines<float>(ny);
    s.zs_partition = zsolve_partition(nz - 2, f64 ? 16 : 8);
    return s;
}

bool poisson_planes(Prec prec, int nx, int ny)
{
    auto any = [](auto) {};
    return prec == Prec::F64 ? with_plane<double>(nx, ny, any) : with_plane<float>(nx, ny, any);
}

hipError_t launch_poisson_setup(Prec prec, const PoissonJob& job, PoissonJob* dst, void* twx, int nx, void* twy, int ny,
                                hipStream_t st)
{
    const unsigned grid = (unsigned)(nx + ny + 255) / 256;
    if (prec == Prec::F64)
        setup_kernel<double><<<grid, 256, 0, st>>>(job, dst, (cplx<double>*)twx, nx, (cplx<double>*)twy, ny);
    else setup_kernel<float><<<grid, 256, 0, st>>>(job, dst, (cplx<float>*)twx, nx, (cplx<float>*)twy, ny);
    return hipGetLastError();
}

hipError_t launch_poisson_group(Prec prec, const PoissonGroup& g, hipStream_t st)
{
    if (prec == Prec::F64) return poisson_t<double>(g, st);
    return poisson_t<float>(g, st);
}

const char* poisson_failed_pass() { return g_failed_pass; }

}  // namespace ehd
