// m3d_fft.hpp -- complex arithmetic and the in-register butterflies of the
// LDS-resident Stockham FFTs (gfx950).
//
// A workgroup owns a tile of lines in LDS and transforms all of them with a
// sequence of in-place Stockham passes: every thread loads the R inputs of
// each of its butterflies into registers, the butterflies are computed, the
// workgroup synchronises and stores them to their autosorted positions.  No
// bit reversal pass is needed and the output is in natural order.  The
// passes themselves are in m3d_fast.hpp (compile-time line lengths) and
// m3d_flex.hpp (any product of primes up to 13).
//
// Twiddles come from a per-axis table tw[m] = exp(-2 pi i m / Ltab); a pass
// over lines of length L uses stride Ltab/L into it.
#pragma once
#include <hip/hip_runtime.h>

namespace m3d {

template <typename T>
struct cx {
    T re, im;
};

template <typename T>
__device__ __forceinline__ cx<T> mk(T a, T b) { return cx<T>{a, b}; }
template <typename T>
__device__ __forceinline__ cx<T> operator+(cx<T> a, cx<T> b) { return cx<T>{a.re + b.re, a.im + b.im}; }
template <typename T>
__device__ __forceinline__ cx<T> operator-(cx<T> a, cx<T> b) { return cx<T>{a.re - b.re, a.im - b.im}; }
template <typename T>
__device__ __forceinline__ cx<T> cmul(cx<T> a, cx<T> b)
{
    return cx<T>{a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
}
template <typename T>
__device__ __forceinline__ cx<T> cscale(cx<T> a, T s) { return cx<T>{a.re * s, a.im * s}; }
template <typename T>
__device__ __forceinline__ cx<T> cconj(cx<T> a) { return cx<T>{a.re, -a.im}; }
// multiply by -i (forward, DIR<0) or +i (inverse, DIR>0)
template <int DIR, typename T>
__device__ __forceinline__ cx<T> rot90(cx<T> a)
{
    return DIR < 0 ? cx<T>{a.im, -a.re} : cx<T>{-a.im, a.re};
}

// radix sequence of one axis' line FFT
struct FftAxis {
    int L;                   // transform length
    int np;                  // number of passes (<= 16)
    unsigned long long rad;  // radix - 1 of pass p in bits [4p, 4p+4) (kept packed so the
                             // kernel never indexes its by-value arguments dynamically)
    __host__ __device__ int radix(int p) const { return (int)((rad >> (4 * p)) & 15ull) + 1; }
};

// cos and sin of 2 pi p / q as compile-time constants: the angle is reduced
// to [0, pi/4] in exact integer arithmetic and carried as x + lo (Dekker's
// product gives the rounding of x), then summed by its Taylor series from the
// smallest term
constexpr double root_series(long long p, long long q, bool cosine)
{
    const double pi2 = 2 * 3.14159265358979323846, pi2_lo = 2 * 1.2246467991473532e-16;
    const double x = pi2 * (double)p / (double)q;
    auto split = [](double a, double& h, double& l) {
        const double c = 134217729.0 * a; // 2^27 + 1
        h = c - (c - a);
        l = a - h;
    };
    auto prod_err = [&](double a, double b) { // a b - fl(a b)
        double ah = 0, al = 0, bh = 0, bl = 0;
        split(a, ah, al);
        split(b, bh, bl);
        return ((ah * bh - a * b) + ah * bl + al * bh) + al * bl;
    };
    const double num = pi2 * (double)p, back = x * (double)q;
    const double lo = ((num - back) + (prod_err(pi2, (double)p) - prod_err(x, (double)q)) + pi2_lo * (double)p) / (double)q;
    double c = 0, s = 0; // cos x - 1 and (sin x - x) by Horner's rule
    for (int i = 26; i >= 2; i -= 2) {
        c = -x * x / (double)((i - 1) * i) * (1.0 + c);
        s = -x * x / (double)(i * (i + 1)) * (1.0 + s);
    }
    return cosine ? 1.0 + (c - lo * x) : x + (x * s + lo * (1.0 + c));
}
constexpr double root_sin(long long p, long long q);
constexpr double root_cos(long long p, long long q)
{
    p %= q;
    if (p < 0) p += q;
    if (2 * p > q) p = q - p;                                   // cos(2 pi - a) = cos a
    if (4 * p > q) return -root_cos(q - 2 * p, 2 * q);          // cos(pi - a) = -cos a
    if (8 * p > q) return root_series(q - 4 * p, 4 * q, false); // cos a = sin(pi/2 - a)
    return root_series(p, q, true);
}
constexpr double root_sin(long long p, long long q) { return root_cos(4 * p - q, 4 * q); } // cos(a - pi/2)
template <int N>
struct RootTab {
    double c[N] = {}, s[N] = {}; // of 2 pi m / N
    constexpr RootTab()
    {
        for (int m = 0; m < N; ++m) {
            c[m] = root_cos(m, N);
            s[m] = root_sin(m, N);
        }
    }
};

template <typename T, int R, int DIR>
__device__ __forceinline__ void butterfly(cx<T> (&v)[R]);

// R = A B points: A-point DFTs over n1 of v[B n1 + n2], twiddles W_R^(n2 k1),
// B-point DFTs over n2; X[k1 + A k2] lands in v[k1 + A k2]
template <typename T, int A, int B, int DIR>
__device__ __forceinline__ void butterfly_ab(cx<T> (&v)[A * B])
{
    constexpr RootTab<A * B> rt;
    cx<T> y[B][A];
#pragma unroll
    for (int n2 = 0; n2 < B; ++n2) {
        cx<T> t[A];
#pragma unroll
        for (int n1 = 0; n1 < A; ++n1) t[n1] = v[B * n1 + n2];
        butterfly<T, A, DIR>(t);
#pragma unroll
        for (int k1 = 0; k1 < A; ++k1) {
            if (n2 * k1 == 0) y[n2][k1] = t[k1];
            else {
                const T c = T(rt.c[n2 * k1]), s = T(DIR > 0 ? rt.s[n2 * k1] : -rt.s[n2 * k1]);
                y[n2][k1] = cx<T>{t[k1].re * c - t[k1].im * s, t[k1].re * s + t[k1].im * c};
            }
        }
    }
#pragma unroll
    for (int k1 = 0; k1 < A; ++k1) {
        cx<T> u[B];
#pragma unroll
        for (int n2 = 0; n2 < B; ++n2) u[n2] = y[n2][k1];
        butterfly<T, B, DIR>(u);
#pragma unroll
        for (int k2 = 0; k2 < B; ++k2) v[k1 + A * k2] = u[k2];
    }
}

template <typename T, int R, int DIR>
__device__ __forceinline__ void butterfly(cx<T> (&v)[R])
{
    if constexpr (R == 2) {
        cx<T> a = v[0], b = v[1];
        v[0] = a + b;
        v[1] = a - b;
    } else if constexpr (R == 3) {
        const T c = T(-0.5);
        const T s = T(0.86602540378443864676372317075294); // sin(2 pi / 3)
        cx<T> t1 = v[1] + v[2];
        cx<T> t2 = v[1] - v[2];
        cx<T> m = cx<T>{v[0].re + c * t1.re, v[0].im + c * t1.im};
        // forward: X1 = m - i s t2, X2 = m + i s t2
        cx<T> r = rot90<DIR>(t2);
        v[0] = v[0] + t1;
        v[1] = cx<T>{m.re + s * r.re, m.im + s * r.im};
        v[2] = cx<T>{m.re - s * r.re, m.im - s * r.im};
    } else if constexpr (R == 4) {
        cx<T> s02 = v[0] + v[2], d02 = v[0] - v[2];
        cx<T> s13 = v[1] + v[3], d13 = rot90<DIR>(v[1] - v[3]);
        v[0] = s02 + s13;
        v[2] = s02 - s13;
        v[1] = d02 + d13;
        v[3] = d02 - d13;
    } else if constexpr (R == 8) {
        const T h = T(0.70710678118654752440084436210485);
        cx<T> e[4] = {v[0], v[2], v[4], v[6]};
        cx<T> o[4] = {v[1], v[3], v[5], v[7]};
        // 4-point DFTs
        {
            cx<T> s02 = e[0] + e[2], d02 = e[0] - e[2];
            cx<T> s13 = e[1] + e[3], d13 = rot90<DIR>(e[1] - e[3]);
            e[0] = s02 + s13; e[2] = s02 - s13; e[1] = d02 + d13; e[3] = d02 - d13;
        }
        {
            cx<T> s02 = o[0] + o[2], d02 = o[0] - o[2];
            cx<T> s13 = o[1] + o[3], d13 = rot90<DIR>(o[1] - o[3]);
            o[0] = s02 + s13; o[2] = s02 - s13; o[1] = d02 + d13; o[3] = d02 - d13;
        }
        // twiddles W8^k (forward: exp(-i pi k / 4))
        cx<T> o1 = o[1], o2 = o[2], o3 = o[3];
        cx<T> r1 = rot90<DIR>(o1);
        o1 = cx<T>{h * (o1.re + r1.re), h * (o1.im + r1.im)}; // (1 -/+ i)/sqrt2
        o2 = rot90<DIR>(o2);
        cx<T> r3 = rot90<DIR>(o3);
        o3 = cx<T>{h * (r3.re - o3.re), h * (r3.im - o3.im)}; // (-1 -/+ i)/sqrt2
        v[0] = e[0] + o[0];
        v[4] = e[0] - o[0];
        v[1] = e[1] + o1;
        v[5] = e[1] - o1;
        v[2] = e[2] + o2;
        v[6] = e[2] - o2;
        v[3] = e[3] + o3;
        v[7] = e[3] - o3;
    } else if constexpr (R == 16) {
        // 16 = 4 x 4: 4-point DFTs over n1 of x[4 n1 + n2], twiddles
        // W16^(n2 k1), 4-point DFTs over n2; X[k1 + 4 k2] lands in v[k1 + 4 k2]
        const T c1 = T(0.92387953251128675612818318939679); // cos(pi/8)
        const T s1 = T(0.38268343236508977172845998403040); // sin(pi/8)
        const T h = T(0.70710678118654752440084436210485);
        cx<T> y[4][4];
#pragma unroll
        for (int n2 = 0; n2 < 4; ++n2) {
            const cx<T> a = v[n2], b = v[n2 + 4], c = v[n2 + 8], d = v[n2 + 12];
            const cx<T> s02 = a + c, d02 = a - c, s13 = b + d, d13 = rot90<DIR>(b - d);
            y[n2][0] = s02 + s13;
            y[n2][1] = d02 + d13;
            y[n2][2] = s02 - s13;
            y[n2][3] = d02 - d13;
        }
        // W16^m = (cos, DIR*sin)(2 pi m / 16): forward exp(-i ...), inverse exp(+i ...)
        auto tmul = [](cx<T> z, T wr, T wi) { return cx<T>{z.re * wr - z.im * wi, z.re * wi + z.im * wr}; };
        const T sd = DIR > 0 ? T(1) : T(-1);
        y[1][1] = tmul(y[1][1], c1, sd * s1);   // m = 1
        y[1][2] = tmul(y[1][2], h, sd * h);     // m = 2
        y[1][3] = tmul(y[1][3], s1, sd * c1);   // m = 3
        y[2][1] = tmul(y[2][1], h, sd * h);     // m = 2
        y[2][2] = rot90<DIR>(y[2][2]);          // m = 4: -i forward, +i inverse
        y[2][3] = tmul(y[2][3], -h, sd * h);    // m = 6
        y[3][1] = tmul(y[3][1], s1, sd * c1);   // m = 3
        y[3][2] = tmul(y[3][2], -h, sd * h);    // m = 6
        y[3][3] = tmul(y[3][3], -c1, -sd * s1); // m = 9
#pragma unroll
        for (int k1 = 0; k1 < 4; ++k1) {
            const cx<T> a = y[0][k1], b = y[1][k1], c = y[2][k1], d = y[3][k1];
            const cx<T> s02 = a + c, d02 = a - c, s13 = b + d, d13 = rot90<DIR>(b - d);
            v[k1] = s02 + s13;
            v[k1 + 4] = d02 + d13;
            v[k1 + 8] = s02 - s13;
            v[k1 + 12] = d02 - d13;
        }
    } else if constexpr (R == 6) {
        butterfly_ab<T, 3, 2, DIR>(v);
    } else if constexpr (R == 9) {
        butterfly_ab<T, 3, 3, DIR>(v);
    } else if constexpr (R == 10) {
        butterfly_ab<T, 5, 2, DIR>(v);
    } else if constexpr (R == 12) {
        butterfly_ab<T, 3, 4, DIR>(v);
    } else if constexpr (R == 14) {
        butterfly_ab<T, 7, 2, DIR>(v);
    } else if constexpr (R == 15) {
        butterfly_ab<T, 5, 3, DIR>(v);
    } else {
        // odd prime: sums and differences of the pairs (m, R - m), then
        //   X_q, X_(R-q) = A_q -/+ i B_q,  A_q = v0 + sum_m cos(2 pi q m / R) (v_m + v_(R-m)),
        //   B_q = sum_m sin(2 pi q m / R) (v_m - v_(R-m))     (signs for the forward transform)
        static_assert(R == 5 || R == 7 || R == 11 || R == 13, "radix");
        constexpr int H = (R - 1) / 2;
        constexpr RootTab<R> rt;
        cx<T> t[H], d[H];
        cx<T> x0 = v[0];
#pragma unroll
        for (int m = 1; m <= H; ++m) {
            t[m - 1] = v[m] + v[R - m];
            d[m - 1] = v[m] - v[R - m];
            x0 = x0 + t[m - 1];
        }
#pragma unroll
        for (int q = 1; q <= H; ++q) {
            cx<T> a = v[0], b{T(0), T(0)};
#pragma unroll
            for (int m = 1; m <= H; ++m) {
                const T c = T(rt.c[q * m % R]), s = T(rt.s[q * m % R]);
                a = cx<T>{a.re + c * t[m - 1].re, a.im + c * t[m - 1].im};
                b = cx<T>{b.re + s * d[m - 1].re, b.im + s * d[m - 1].im};
            }
            b = rot90<DIR>(b);
            v[q] = a + b;
            v[R - q] = a - b;
        }
        v[0] = x0;
    }
}

} // namespace m3d
