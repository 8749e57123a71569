// LDS-staged mixed-radix (2, 3, 4, 5) Stockham FFT for gfx950.
//
// Replaces the Temperton/NCAR FFT99/CFFT99 passes (libs/fft99/VPASSM.f90,
// CFFT99.f90) used by the Poisson solver.  Same transform definitions:
// forward exp(-2 pi i jk/n), inverse exp(+2 pi i jk/n), both unnormalised
// here (the 1/(L N) factor of FFT99's forward real transform and of the
// reference's UN3M is applied once, in the wall-normal solve).
//
// A block transforms `howmany` vectors held in LDS; each Stockham stage reads
// one buffer and writes the other (autosort, no bit reversal), so any length
// whose factors are 2, 3, 4 and 5 works, as FFT99 allows.
#pragma once

#include <utility>

#include "chs_common.hpp"

namespace chs {

struct FftPlan {
    int n;
    int nst;
    int rad[20];
};

// radix-R DFT of v[0..R-1] in registers; dir = -1 forward, +1 inverse
template <int R, typename C, typename Rl>
__device__ __forceinline__ void dft_small(C (&v)[5], int dir) {
    if constexpr (R == 2) {
        C t = v[0];
        v[0] = cadd(t, v[1]);
        v[1] = csub(t, v[1]);
    } else if constexpr (R == 4) {
        C t0 = cadd(v[0], v[2]), t1 = csub(v[0], v[2]);
        C t2 = cadd(v[1], v[3]), t3 = cmul_i(csub(v[1], v[3]), dir);
        v[0] = cadd(t0, t2);
        v[2] = csub(t0, t2);
        v[1] = cadd(t1, t3);
        v[3] = csub(t1, t3);
    } else if constexpr (R == 3) {
        const Rl c = Rl(-0.5), s = Rl(0.86602540378443864676372317075294);  // cos, sin(2 pi/3)
        C sum = cadd(v[1], v[2]);
        C dif = csub(v[1], v[2]);
        C m = C{v[0].x + c * sum.x, v[0].y + c * sum.y};
        C t = cmul_i(C{s * dif.x, s * dif.y}, dir);
        v[0] = cadd(v[0], sum);
        v[1] = cadd(m, t);
        v[2] = csub(m, t);
    } else if constexpr (R == 5) {
        const Rl c1 = Rl(0.30901699437494742410229341718282);   // cos(2 pi/5)
        const Rl c2 = Rl(-0.80901699437494742410229341718282);  // cos(4 pi/5)
        const Rl s1 = Rl(0.95105651629515357211643933337938);   // sin(2 pi/5)
        const Rl s2 = Rl(0.58778525229247312916870595463907);   // sin(4 pi/5)
        C a14 = cadd(v[1], v[4]), d14 = csub(v[1], v[4]);
        C a23 = cadd(v[2], v[3]), d23 = csub(v[2], v[3]);
        C m1 = C{v[0].x + c1 * a14.x + c2 * a23.x, v[0].y + c1 * a14.y + c2 * a23.y};
        C m2 = C{v[0].x + c2 * a14.x + c1 * a23.x, v[0].y + c2 * a14.y + c1 * a23.y};
        C t1 = cmul_i(C{s1 * d14.x + s2 * d23.x, s1 * d14.y + s2 * d23.y}, dir);
        C t2 = cmul_i(C{s2 * d14.x - s1 * d23.x, s2 * d14.y - s1 * d23.y}, dir);
        v[0] = cadd(v[0], cadd(a14, a23));
        v[1] = cadd(m1, t1);
        v[4] = csub(m1, t1);
        v[2] = cadd(m2, t2);
        v[3] = csub(m2, t2);
    }
}

// One Stockham stage of radix R over `howmany` vectors: x -> y.
template <int R, typename Rl>
__device__ __forceinline__ void stockham_stage(const cpx_t<Rl>* x, cpx_t<Rl>* y, int n, int howmany, int bstride,
                                               int Ns, const cpx_t<Rl>* tw, int dir) {
    using C = cpx_t<Rl>;
    const int nb = n / R;
    const int tstep = n / (Ns * R);
    for (int w = threadIdx.x; w < howmany * nb; w += blockDim.x) {
        const int bidx = w / nb, j = w - bidx * nb;
        const C* src = x + bidx * bstride;
        C* dst = y + bidx * bstride;
        const int k = j % Ns;
        C v[5];
#pragma unroll
        for (int r = 0; r < R; ++r) v[r] = src[j + r * nb];
        if (Ns > 1) {
#pragma unroll
            for (int r = 1; r < R; ++r) {
                C t = tw[r * k * tstep];
                if (dir > 0) t.y = -t.y;
                v[r] = cmul(v[r], t);
            }
        }
        dft_small<R, C, Rl>(v, dir);
        const int idxD = (j / Ns) * Ns * R + k;
#pragma unroll
        for (int r = 0; r < R; ++r) dst[idxD + r * Ns] = v[r];
    }
}

// Full transform; returns the buffer holding the result (x or y).
template <typename Rl>
__device__ cpx_t<Rl>* fft_lds(cpx_t<Rl>* x, cpx_t<Rl>* y, int howmany, int bstride, const FftPlan& p,
                              const cpx_t<Rl>* tw, int dir) {
    int Ns = 1;
    for (int s = 0; s < p.nst; ++s) {
        const int R = p.rad[s];
        switch (R) {
            case 4: stockham_stage<4, Rl>(x, y, p.n, howmany, bstride, Ns, tw, dir); break;
            case 2: stockham_stage<2, Rl>(x, y, p.n, howmany, bstride, Ns, tw, dir); break;
            case 3: stockham_stage<3, Rl>(x, y, p.n, howmany, bstride, Ns, tw, dir); break;
            default: stockham_stage<5, Rl>(x, y, p.n, howmany, bstride, Ns, tw, dir); break;
        }
        __syncthreads();
        cpx_t<Rl>* t = x;
        x = y;
        y = t;
        Ns *= R;
    }
    return x;
}

// Host: factor n into radices 4, 2, 3, 5 (FFTFAX-style factor list).
inline bool fft_plan(int n, FftPlan* p) {
    p->n = n;
    p->nst = 0;
    int m = n;
    while (m % 4 == 0) { p->rad[p->nst++] = 4; m /= 4; }
    while (m % 2 == 0) { p->rad[p->nst++] = 2; m /= 2; }
    while (m % 3 == 0) { p->rad[p->nst++] = 3; m /= 3; }
    while (m % 5 == 0) { p->rad[p->nst++] = 5; m /= 5; }
    return m == 1 && p->nst <= 20;
}

// ---------------------------------------------------------------------------
// Register transforms: a length n = R1 R2 (radices up to 16) or R1 R2 R3 (up
// to 10) as that many Stockham stages, each a whole radix-R DFT in a thread's
// registers.  The first stage reads global memory and the last writes it (or
// the caller's LDS rows), so a transform crosses LDS once per stage boundary.
// ---------------------------------------------------------------------------

// cos and sin of 2 pi m / r at compile time: the angle reduced to an octant,
// then the Taylor series to below one ulp
constexpr double trig_series(double x, bool sine) {
    double t = sine ? x : 1.0, s = 0.0;
    double term[14] = {};
    for (int q = 0; q < 14; ++q) {
        term[q] = t;
        const double a = 2.0 * q + (sine ? 2.0 : 1.0);
        t = -t * x * x / (a * (a + 1.0));
    }
    for (int q = 13; q >= 0; --q) s += term[q];
    return s;
}
constexpr double trig_2pi(int m, int r, bool sine) {
    m %= r;
    if (m < 0) m += r;
    int o = 8 * m / r;                   // octant of the angle
    const double pi4 = 0.78539816339744830961566084581988;
    // the angle within the octant, from its nearer multiple of pi/2
    const bool odd = o & 1;
    const int num = odd ? (o + 1) * r - 8 * m : 8 * m - o * r;   // in eighths of 1/r
    const double x = pi4 * (double)num / (double)r;
    const double c = trig_series(x, false), s = trig_series(x, true);
    // the angle is (o/2) pi/2 + x (even octants) or ((o+1)/2) pi/2 - x (odd)
    const int quad = ((o + 1) / 2) % 4;
    const double sx = odd ? -s : s;
    const double cosv = quad == 0 ? c : quad == 1 ? -sx : quad == 2 ? -c : sx;
    const double sinv = quad == 0 ? sx : quad == 1 ? c : quad == 2 ? -sx : -c;
    return sine ? sinv : cosv;
}
template <int M, int R>
struct UnitRoot {
    static constexpr double c = trig_2pi(M, R, false), s = trig_2pi(M, R, true);
};
// z W_R^m (forward) or its conjugate (inverse), m and R compile-time
template <int M, int R, int DIR>
__device__ __forceinline__ double2 mul_root(double2 z) {
    if constexpr (M % R == 0) {
        return z;
    } else {
        constexpr double c = UnitRoot<M, R>::c, s = DIR > 0 ? UnitRoot<M, R>::s : -UnitRoot<M, R>::s;
        return make_double2(z.x * c - z.y * s, z.x * s + z.y * c);
    }
}

constexpr int dft_first(int r) { return r == 16 ? 4 : r % 3 == 0 && r != 6 ? 3 : 2; }   // R = A B: the first factor

template <int R, int A, int B, int DIR, int... I>
__device__ __forceinline__ void dft_reg_columns(double2 (&v)[R], double2 (&y)[R], std::integer_sequence<int, I...>);

// In-place DFT of v[0..R-1], natural order in and out; DIR -1 forward, +1 inverse
template <int R, int DIR>
__device__ __forceinline__ void dft_reg(double2 (&v)[R]) {
    if constexpr (R == 2 || R == 3 || R == 4 || R == 5) {
        double2 t[5];
#pragma unroll
        for (int q = 0; q < R; ++q) t[q] = v[q];
        dft_small<R, double2, double>(t, DIR);
#pragma unroll
        for (int q = 0; q < R; ++q) v[q] = t[q];
    } else {
        constexpr int A = dft_first(R), B = R / A;
        double2 y[R];
        dft_reg_columns<R, A, B, DIR>(v, y, std::make_integer_sequence<int, R>{});
#pragma unroll
        for (int k1 = 0; k1 < A; ++k1) {   // DFT-B over n2: X[k1 + A k2]
            double2 t[B];
#pragma unroll
            for (int n2 = 0; n2 < B; ++n2) t[n2] = y[A * n2 + k1];
            dft_reg<B, DIR>(t);
#pragma unroll
            for (int k2 = 0; k2 < B; ++k2) v[k1 + A * k2] = t[k2];
        }
    }
}
// n = B n1 + n2: DFT-A over n1, times W_R^(n2 k1), to y[A n2 + k1]
template <int R, int A, int B, int DIR, int... I>
__device__ __forceinline__ void dft_reg_columns(double2 (&v)[R], double2 (&y)[R], std::integer_sequence<int, I...>) {
#pragma unroll
    for (int n2 = 0; n2 < B; ++n2) {
        double2 t[A];
#pragma unroll
        for (int n1 = 0; n1 < A; ++n1) t[n1] = v[B * n1 + n2];
        dft_reg<A, DIR>(t);
#pragma unroll
        for (int k1 = 0; k1 < A; ++k1) y[A * n2 + k1] = t[k1];
    }
    ((y[I] = mul_root<(I / A) * (I % A), R, DIR>(y[I])), ...);
}

// The stages of a register transform: radices r, butterflies per stage nb =
// n / r, threads per transform T = the largest nb
struct RegPlan {
    int n, nst;
    int r[3], nb[3];
    int T;
    float Tinv;
};

// Two stages where radices up to 16 allow, three (up to 10) otherwise; the
// split with the fewest threads per transform.  The first stage reads runs of
// n / r[0] consecutive elements and the last writes runs of n / r[nst - 1]:
// small_first makes the first run the longer one.  False: no such split with
// at most 128 threads per transform.
inline bool reg_plan(int n, bool small_first, RegPlan* p) {
    const int r2[] = {2, 3, 4, 5, 6, 8, 9, 10, 12, 15, 16}, r3[] = {4, 5, 6, 8, 9, 10};
    p->n = n;
    p->nst = 0;
    p->T = 1 << 20;
    auto take = [&](int nst, int a, int b, int c) {
        const int r[3] = {a, b, c};
        int T = 0;
        for (int q = 0; q < nst; ++q) T = T > n / r[q] ? T : n / r[q];
        if (T >= p->T) return;
        p->T = T;
        p->nst = nst;
        for (int q = 0; q < 3; ++q) {
            p->r[q] = q < nst ? r[q] : 1;
            p->nb[q] = q < nst ? n / r[q] : 0;
        }
    };
    for (int b : r2)
        for (int a : r2)
            if (a >= b && a * b == n) small_first ? take(2, b, a, 1) : take(2, a, b, 1);
    if (p->nst == 0)
        for (int a : r3)
            for (int b : r3)
                for (int c : r3)
                    if (a >= b && b >= c && a * b * c == n) small_first ? take(3, c, b, a) : take(3, a, b, c);
    p->Tinv = 1.0f / (float)p->T;
    return p->nst != 0 && p->T <= 128;
}

}  // namespace chs
