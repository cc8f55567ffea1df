// In-register DFTs (2 to 24 points), forward and inverse.
#pragma once
#include "common.h"

namespace fans {

template <typename T, int R, bool INV>
__device__ __forceinline__ void dft(cplx<T> (&v)[R]);


template <>
__device__ __forceinline__ void dft<double, 2, false>(cplx<double> (&v)[2])
{
    cplx<double> a = v[0];
    v[0]           = a + v[1];
    v[1]           = a - v[1];
}
template <>
__device__ __forceinline__ void dft<double, 2, true>(cplx<double> (&v)[2])
{
    dft<double, 2, false>(v);
}
template <>
__device__ __forceinline__ void dft<float, 2, false>(cplx<float> (&v)[2])
{
    cplx<float> a = v[0];
    v[0]          = a + v[1];
    v[1]          = a - v[1];
}
template <>
__device__ __forceinline__ void dft<float, 2, true>(cplx<float> (&v)[2])
{
    dft<float, 2, false>(v);
}

template <typename T, bool INV>
__device__ __forceinline__ void dft3(cplx<T> (&v)[3])
{
    const T      s3 = (T) 0.86602540378443864676;
    cplx<T>      t1 = v[1] + v[2];
    cplx<T>      t2 = v[0] - cscale(t1, (T) 0.5);
    cplx<T>      t3 = mul_mi<T, INV>(cscale(v[1] - v[2], s3));
    v[0]            = v[0] + t1;
    v[1]            = t2 + t3;
    v[2]            = t2 - t3;
}
template <>
__device__ __forceinline__ void dft<double, 3, false>(cplx<double> (&v)[3]) { dft3<double, false>(v); }
template <>
__device__ __forceinline__ void dft<double, 3, true>(cplx<double> (&v)[3]) { dft3<double, true>(v); }
template <>
__device__ __forceinline__ void dft<float, 3, false>(cplx<float> (&v)[3]) { dft3<float, false>(v); }
template <>
__device__ __forceinline__ void dft<float, 3, true>(cplx<float> (&v)[3]) { dft3<float, true>(v); }

template <typename T, bool INV>
__device__ __forceinline__ void dft4(cplx<T> (&v)[4])
{
    cplx<T> t0 = v[0] + v[2], t1 = v[0] - v[2], t2 = v[1] + v[3];
    cplx<T> t3 = mul_mi<T, INV>(v[1] - v[3]);
    v[0]       = t0 + t2;
    v[2]       = t0 - t2;
    v[1]       = t1 + t3;
    v[3]       = t1 - t3;
}
template <>
__device__ __forceinline__ void dft<double, 4, false>(cplx<double> (&v)[4]) { dft4<double, false>(v); }
template <>
__device__ __forceinline__ void dft<double, 4, true>(cplx<double> (&v)[4]) { dft4<double, true>(v); }
template <>
__device__ __forceinline__ void dft<float, 4, false>(cplx<float> (&v)[4]) { dft4<float, false>(v); }
template <>
__device__ __forceinline__ void dft<float, 4, true>(cplx<float> (&v)[4]) { dft4<float, true>(v); }

template <typename T, bool INV>
__device__ __forceinline__ void dft5(cplx<T> (&v)[5])
{
    const T c1 = (T) 0.30901699437494742410, c2 = (T) -0.80901699437494742410;
    const T s1 = (T) 0.95105651629515357212, s2 = (T) 0.58778525229247312917;
    cplx<T> a1 = v[1] + v[4], b1 = v[1] - v[4], a2 = v[2] + v[3], b2 = v[2] - v[3];
    cplx<T> p1 = v[0] + cscale(a1, c1) + cscale(a2, c2);
    cplx<T> p2 = v[0] + cscale(a1, c2) + cscale(a2, c1);
    cplx<T> q1 = mul_mi<T, INV>(cscale(b1, s1) + cscale(b2, s2));
    cplx<T> q2 = mul_mi<T, INV>(cscale(b1, s2) - cscale(b2, s1));
    v[0]       = v[0] + a1 + a2;
    v[1]       = p1 + q1;
    v[4]       = p1 - q1;
    v[2]       = p2 + q2;
    v[3]       = p2 - q2;
}
template <>
__device__ __forceinline__ void dft<double, 5, false>(cplx<double> (&v)[5]) { dft5<double, false>(v); }
template <>
__device__ __forceinline__ void dft<double, 5, true>(cplx<double> (&v)[5]) { dft5<double, true>(v); }
template <>
__device__ __forceinline__ void dft<float, 5, false>(cplx<float> (&v)[5]) { dft5<float, false>(v); }
template <>
__device__ __forceinline__ void dft<float, 5, true>(cplx<float> (&v)[5]) { dft5<float, true>(v); }

template <typename T, bool INV>
__device__ __forceinline__ void dft8(cplx<T> (&v)[8])
{
    const T r = (T) 0.70710678118654752440;
    cplx<T> a[4], b[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        a[t] = v[t] + v[t + 4];
        b[t] = v[t] - v[t + 4];
    }
    // b[1] *= W8, b[2] *= W8^2, b[3] *= W8^3  (W8 = exp(-+ 2 pi i / 8))
    {
        cplx<T> x = b[1];
        b[1]      = INV ? cplx<T>{(x.x - x.y) * r, (x.x + x.y) * r} : cplx<T>{(x.x + x.y) * r, (x.y - x.x) * r};
        b[2]      = mul_mi<T, INV>(b[2]);
        x         = b[3];
        b[3]      = INV ? cplx<T>{(-x.x - x.y) * r, (x.x - x.y) * r} : cplx<T>{(x.y - x.x) * r, (-x.x - x.y) * r};
    }
    dft4<T, INV>(a);
    dft4<T, INV>(b);
    v[0] = a[0];
    v[2] = a[1];
    v[4] = a[2];
    v[6] = a[3];
    v[1] = b[0];
    v[3] = b[1];
    v[5] = b[2];
    v[7] = b[3];
}
template <>
__device__ __forceinline__ void dft<double, 8, false>(cplx<double> (&v)[8]) { dft8<double, false>(v); }
template <>
__device__ __forceinline__ void dft<double, 8, true>(cplx<double> (&v)[8]) { dft8<double, true>(v); }
template <>
__device__ __forceinline__ void dft<float, 8, false>(cplx<float> (&v)[8]) { dft8<float, false>(v); }
template <>
__device__ __forceinline__ void dft<float, 8, true>(cplx<float> (&v)[8]) { dft8<float, true>(v); }

// in-register DFT of length 16 as 4 x 4 with constant internal twiddles
template <typename T, bool INV>
__device__ __forceinline__ void dft16(cplx<T> (&v)[16])
{
    const T c = (T) 0.92387953251128675613, s = (T) 0.38268343236508977173, r = (T) 0.70710678118654752440;
    cplx<T> y[4][4];
#pragma unroll
    for (int i2 = 0; i2 < 4; ++i2) {
        cplx<T> a[4] = {v[i2], v[i2 + 4], v[i2 + 8], v[i2 + 12]};
        dft4<T, INV>(a);
#pragma unroll
        for (int k1 = 0; k1 < 4; ++k1)
            y[i2][k1] = a[k1];
    }
    // y[i2][k1] *= W16^(i2 k1); forward W16^p = (cos, -sin)(2 pi p / 16)
    auto tw = [&](cplx<T> a, T wr, T wi) { return INV ? cplx<T>{a.x * wr + a.y * wi, a.y * wr - a.x * wi}
                                                       : cplx<T>{a.x * wr - a.y * wi, a.x * wi + a.y * wr}; };
    // (wr, wi) below are the forward twiddles; the lambda conjugates for INV
    y[1][1] = tw(y[1][1], c, -s);
    y[1][2] = tw(y[1][2], r, -r);
    y[1][3] = tw(y[1][3], s, -c);
    y[2][1] = tw(y[2][1], r, -r);
    y[2][2] = tw(y[2][2], (T) 0, (T) -1);
    y[2][3] = tw(y[2][3], -r, -r);
    y[3][1] = tw(y[3][1], s, -c);
    y[3][2] = tw(y[3][2], -r, -r);
    y[3][3] = tw(y[3][3], -c, s);
#pragma unroll
    for (int k1 = 0; k1 < 4; ++k1) {
        cplx<T> a[4] = {y[0][k1], y[1][k1], y[2][k1], y[3][k1]};
        dft4<T, INV>(a);
#pragma unroll
        for (int k2 = 0; k2 < 4; ++k2)
            v[k1 + 4 * k2] = a[k2];
    }
}

// exp(-2 pi i k / n) for compile-time k, n: the angle reduced to a quadrant
// and a Taylor series there (terms below 1e-20 of the result)
constexpr double ct_taylor(double x, bool sine)
{
    // sin: x - x^3/3! + ...; cos: 1 - x^2/2! + ...
    double t = sine ? x : 1.0, s = t;
    for (int m = 1; m < 14; ++m) {
        const double a = sine ? 2.0 * m : 2.0 * m - 1.0;
        t *= -x * x / (a * (a + 1.0));
        s += t;
    }
    return s;
}
struct CtW {
    double re, im;
};
constexpr CtW ct_twiddle(int k, int n)
{
    k %= n;
    const int    q  = (4 * k) / n;  // quadrant of 2 pi k / n
    const double r  = 1.57079632679489661923 * (double) (4 * k - q * n) / (double) n;
    const double cr = ct_taylor(r, false), sr = ct_taylor(r, true);
    // angle q pi/2 + r: rotate (cos r, sin r) by q quarter turns
    const double c = q == 0 ? cr : (q == 1 ? -sr : (q == 2 ? -cr : sr));
    const double s = q == 0 ? sr : (q == 1 ? cr : (q == 2 ? -sr : -cr));
    return CtW{c, -s};
}

template <typename T, int N, bool INV>
__device__ __forceinline__ void dft_reg(cplx<T> (&v)[N]);

// in-register DFT of length P Q by Cooley-Tukey: P-point DFTs over the
// stride-Q subsequences, the twiddles W_PQ^(i2 k1), Q-point DFTs; input
// index i2 + Q m, output k1 + P k2 (dft16's order for P = Q = 4)
template <typename T, int P, int Q, bool INV>
__device__ __forceinline__ void dft_pq(cplx<T> (&v)[P * Q])
{
    cplx<T> y[Q][P];
#pragma unroll
    for (int i2 = 0; i2 < Q; ++i2) {
        cplx<T> a[P];
#pragma unroll
        for (int m = 0; m < P; ++m)
            a[m] = v[i2 + Q * m];
        dft_reg<T, P, INV>(a);
#pragma unroll
        for (int k1 = 0; k1 < P; ++k1) {
            if (i2 * k1 == 0) {
                y[i2][k1] = a[k1];
            } else {
                constexpr int n = P * Q;
                const CtW     w = ct_twiddle(i2 * k1, n);
                const T       wr = (T) w.re, wi = INV ? (T) -w.im : (T) w.im;
                y[i2][k1]        = cplx<T>{a[k1].x * wr - a[k1].y * wi, a[k1].x * wi + a[k1].y * wr};
            }
        }
    }
#pragma unroll
    for (int k1 = 0; k1 < P; ++k1) {
        cplx<T> b[Q];
#pragma unroll
        for (int i2 = 0; i2 < Q; ++i2)
            b[i2] = y[i2][k1];
        dft_reg<T, Q, INV>(b);
#pragma unroll
        for (int k2 = 0; k2 < Q; ++k2)
            v[k1 + P * k2] = b[k2];
    }
}

template <typename T, int N, bool INV>
__device__ __forceinline__ void dft_reg(cplx<T> (&v)[N])
{
    if constexpr (N == 2 || N == 3 || N == 5)
        dft<T, N, INV>(v);
    else if constexpr (N == 4)
        dft4<T, INV>(v);
    else if constexpr (N == 8)
        dft8<T, INV>(v);
    else if constexpr (N == 16)
        dft16<T, INV>(v);
    else if constexpr (N == 6)
        dft_pq<T, 3, 2, INV>(v);
    else if constexpr (N == 9)
        dft_pq<T, 3, 3, INV>(v);
    else if constexpr (N == 10)
        dft_pq<T, 5, 2, INV>(v);
    else if constexpr (N == 12)
        dft_pq<T, 3, 4, INV>(v);
    else if constexpr (N == 15)
        dft_pq<T, 5, 3, INV>(v);
    else if constexpr (N == 20)
        dft_pq<T, 5, 4, INV>(v);
    else {
        static_assert(N == 24, "unsupported register DFT length");
        dft_pq<T, 3, 8, INV>(v);
    }
}

}  // namespace fans
