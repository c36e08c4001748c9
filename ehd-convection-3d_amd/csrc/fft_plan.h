// fft_plan.h -- radix schedule of the runtime-planned LDS FFTs.
#pragma once

namespace ehd {

// multiplier of fdiv: (a * fft_magic(b)) >> 32 = a / b for a, b < 2^16, b > 1
inline unsigned fft_magic(int b) { return b > 1 ? (unsigned)((1ull << 32) / (unsigned)b + 1) : 0u; }

struct FftPlan {
    int n;
    int nst;            // number of stages
    unsigned mn;        // fft_magic(n)
    int rad[16];        // radix of each stage
    int nb[16];         // butterflies of a line, n / radix
    unsigned mnb[16];   // fft_magic(nb)
    unsigned mns[16];   // fft_magic(Ns), Ns = product of the radices before
};

// Prime factors above 13 first (their stage needs no twiddles there), then
// 13, 11, 7, 5, pairs of threes as 9 and a last 3, then the power of two in
// ceil(p/4) balanced stages of 2..16.
inline FftPlan make_fft_plan(int n)
{
    FftPlan p{};
    p.n = n;
    p.mn = fft_magic(n);
    int r = n, ns = 1;
    auto stage = [&](int radix) {
        p.rad[p.nst] = radix;
        p.nb[p.nst] = n / radix;
        p.mnb[p.nst] = fft_magic(n / radix);
        p.mns[p.nst] = fft_magic(ns);
        ns *= radix;
        ++p.nst;
    };
    int twos = 0;
    while (r % 2 == 0) {
        r /= 2;
        ++twos;
    }
    int small = 1;      // the part of the odd factors with a register butterfly
    for (int f : {13, 11, 7, 5, 3})
        while (r % f == 0) {
            r /= f;
            small *= f;
        }
    for (int f = 17; r > 1; f += 2)
        while (r % f == 0) {
            stage(f);
            r /= f;
        }
    for (int f : {13, 11, 7, 5, 9, 3})
        while (small % f == 0) {
            stage(f);
            small /= f;
        }
    const int s2 = (twos + 3) / 4;
    for (int s = 0; s < s2; ++s) stage(1 << (twos / s2 + (s < twos % s2 ? 1 : 0)));
    return p;
}

}  // namespace ehd
