// fft_device.hpp — device building blocks of the gfx950 FFT.
//
// One kernel template, fft_pass_body<L, C, V, IO>, computes a tile of C
// independent DFTs of compile-time length L inside one work-group (V is the
// compile-time variant: pre-op, post-op, Bluestein; see Variant below):
//
//   * each DFT ("instance") is worked on by T = L / R0 threads, R0 being the
//     first radix of the compile-time radix plan of L;
//   * the stages are Stockham autosort steps: a thread reads R values at
//     j + r*L/R from LDS, multiplies by the stage twiddles W_{Ns*R}^{r*(j%Ns)}
//     (a table built in FP64 and rounded once), does an in-register DFT_R and
//     writes them to (j/Ns)*Ns*R + j%Ns + r*Ns, so the result comes out in
//     natural order with no bit reversal;
//   * global memory is walked in one of three ways per side (rk_pass_args
//     load_mode/store_mode): DIRECT (each thread its own elements: coalesced
//     when the axis is contiguous), COLUMN (lanes across adjacent instances,
//     staged through LDS: coalesced when instances are adjacent, i.e. strided
//     axes and the inner passes of a multi-pass transform), FLAT (the tile is
//     one contiguous block, streamed linearly through LDS);
//   * the Bluestein variant runs the whole chirp-z convolution in one tile:
//     chirp on load, forward DFT_L, multiply by the kernel spectrum and
//     conjugate, forward DFT_L again, conjugate, chirp and truncate on store.
//
// The inverse transform is the forward one on conjugated data
// (IFFT(x) = conj(FFT(conj x)) / N), so the direction is the run-time
// in_sign / out_sign / out_scale of the pass arguments, not a kernel variant.
//
// The IO policy supplies the element load/store so that fused input/output
// transformations (generated at run time) reuse the same kernel body.
#ifndef RK_FFT_DEVICE_HPP
#define RK_FFT_DEVICE_HPP

#if !defined(__HIPCC_RTC__)
#include <hip/hip_runtime.h>
#endif

#include "fft_args.h"

#define RK_HD __host__ __device__ __forceinline__

namespace rkfft {

// ------------------------------------------------------------------------
// complex arithmetic (x = re, y = im) on complex64 (float2) and complex128
// (double2) values; a pass's element type is its IO policy's value_type
// ------------------------------------------------------------------------
template <class F> using rk_v2 = F __attribute__((ext_vector_type(2)));

// The values of two adjacent instances at one position, part by part: a pass
// whose value type is cpair2 computes two instances per thread with the same
// code (elementwise arithmetic; PairIO below).
struct cpair2 {
    rk_v2<float> x, y;
};

template <class X> struct RealOf;
template <> struct RealOf<float2> { typedef float type; };
template <> struct RealOf<double2> { typedef double type; };
template <> struct RealOf<cpair2> { typedef rk_v2<float> type; };
template <class X> using real_t = typename RealOf<X>::type;

// Instances per thread of a value type, and its single complex value (the
// element type of its tables).
template <class X> struct ScalarOf { typedef X type; };
template <> struct ScalarOf<cpair2> { typedef float2 type; };
template <class X> using scalar_t = typename ScalarOf<X>::type;
template <class X> RK_HD constexpr int pair_width() { return (int)(sizeof(X) / sizeof(scalar_t<X>)); }

template <class X> RK_HD X cx(real_t<X> re, real_t<X> im);
template <> RK_HD float2 cx<float2>(float re, float im) { return make_float2(re, im); }
template <> RK_HD double2 cx<double2>(double re, double im) { return make_double2(re, im); }
template <> RK_HD cpair2 cx<cpair2>(rk_v2<float> re, rk_v2<float> im) {
    cpair2 r;
    r.x = re;
    r.y = im;
    return r;
}

template <class X> RK_HD X c_add(X a, X b) { return cx<X>(a.x + b.x, a.y + b.y); }
template <class X> RK_HD X c_sub(X a, X b) { return cx<X>(a.x - b.x, a.y - b.y); }
// b: a value of the same type, or one complex factor for both of a cpair2's
template <class X, class W> RK_HD X c_mul(X a, W b) { return cx<X>(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x); }
template <class X> RK_HD X c_conj(X a) { return cx<X>(a.x, -a.y); }
template <class X> RK_HD X c_mul_mi(X a) { return cx<X>(a.y, -a.x); }   // a * (-i)
template <class X> RK_HD X c_scale(X a, real_t<X> s) { return cx<X>(a.x * s, a.y * s); }
// cond ? a : b part by part (a select of the whole 16-byte complex128 value
// is lowered through scratch memory)
template <class X> RK_HD X c_select(bool cond, X a, X b) { return cx<X>(cond ? a.x : b.x, cond ? a.y : b.y); }

// Butterfly constants: double literals, rounded once to the element's real
// type where they are used ((F)RK_C8 and so on).
#define RK_C8 0.7071067811865476      // cos(pi/4)
#define RK_C16 0.9238795325112867     // cos(pi/8)
#define RK_S16 0.3826834323650898     // sin(pi/8)
#define RK_S3 0.8660254037844387      // sin(2pi/3)
#define RK_C5_1 0.30901699437494745   // cos(2pi/5)
#define RK_C5_2 -0.8090169943749473   // cos(4pi/5)
#define RK_S5_1 0.9510565162951535    // sin(2pi/5)
#define RK_S5_2 0.5877852522924732    // sin(4pi/5)
#define RK_C7_1 0.6234898018587336
#define RK_C7_2 -0.22252093395631434
#define RK_C7_3 -0.900968867902419
#define RK_S7_1 0.7818314824680298
#define RK_S7_2 0.9749279121818236
#define RK_S7_3 0.43388373911755823
#define RK_C9_1 0.766044443118978     // cos(2pi/9)
#define RK_S9_1 0.6427876096865394
#define RK_C9_2 0.17364817766693036   // cos(4pi/9)
#define RK_S9_2 0.984807753012208
#define RK_C9_4 -0.9396926207859084   // cos(8pi/9)
#define RK_S9_4 0.3420201433256687

// ------------------------------------------------------------------------
// in-register forward DFTs, y_k = sum_n v_n exp(-2 pi i n k / R), in place
// ------------------------------------------------------------------------
template <class X> RK_HD void dft2(X& a, X& b) {
    X t = a;
    a = c_add(t, b);
    b = c_sub(t, b);
}

template <class X> RK_HD void dft4(X& a0, X& a1, X& a2, X& a3) {
    X t0 = c_add(a0, a2), t1 = c_sub(a0, a2);
    X t2 = c_add(a1, a3), t3 = c_mul_mi(c_sub(a1, a3));
    a0 = c_add(t0, t2);
    a2 = c_sub(t0, t2);
    a1 = c_add(t1, t3);
    a3 = c_sub(t1, t3);
}

// multiply by W8^1 = (1 - i)/sqrt2 and W8^3 = (-1 - i)/sqrt2
template <class X> RK_HD X c_w8_1(X a) {
    using F = real_t<X>;
    return cx<X>((F)RK_C8 * (a.x + a.y), (F)RK_C8 * (a.y - a.x));
}
template <class X> RK_HD X c_w8_3(X a) {
    using F = real_t<X>;
    return cx<X>((F)RK_C8 * (a.y - a.x), -(F)RK_C8 * (a.x + a.y));
}

template <class X> RK_HD void dft8(X* v) {
    X e0 = v[0], e1 = v[2], e2 = v[4], e3 = v[6];
    X o0 = v[1], o1 = v[3], o2 = v[5], o3 = v[7];
    dft4(e0, e1, e2, e3);
    dft4(o0, o1, o2, o3);
    o1 = c_w8_1(o1);
    o2 = c_mul_mi(o2);
    o3 = c_w8_3(o3);
    v[0] = c_add(e0, o0); v[4] = c_sub(e0, o0);
    v[1] = c_add(e1, o1); v[5] = c_sub(e1, o1);
    v[2] = c_add(e2, o2); v[6] = c_sub(e2, o2);
    v[3] = c_add(e3, o3); v[7] = c_sub(e3, o3);
}

// 16 = 4 x 4: DFT4 over n2 for each n1 (x[n1 + 4 n2]), twiddle W16^{n1 k2},
// DFT4 over n1 for each k2, output y[k2 + 4 k1].
template <class X> RK_HD void dft16_second(X* v);
template <class X> RK_HD void dft16(X* v) {
    dft4(v[0], v[4], v[8], v[12]);
    dft4(v[1], v[5], v[9], v[13]);
    dft4(v[2], v[6], v[10], v[14]);
    dft4(v[3], v[7], v[11], v[15]);
    dft16_second(v);
}

// The twiddles and the second DFT4s of dft16.
template <class X> RK_HD void dft16_second(X* v) {
    using F = real_t<X>;
    const X w1 = cx<X>((F)RK_C16, -(F)RK_S16);
    const X w3 = cx<X>((F)RK_S16, -(F)RK_C16);
    const X w9 = cx<X>(-(F)RK_C16, (F)RK_S16);
    v[5] = c_mul(v[5], w1);
    v[9] = c_w8_1(v[9]);
    v[13] = c_mul(v[13], w3);
    v[6] = c_w8_1(v[6]);
    v[10] = c_mul_mi(v[10]);
    v[14] = c_w8_3(v[14]);
    v[7] = c_mul(v[7], w3);
    v[11] = c_w8_3(v[11]);
    v[15] = c_mul(v[15], w9);
    dft4(v[0], v[1], v[2], v[3]);
    dft4(v[4], v[5], v[6], v[7]);
    dft4(v[8], v[9], v[10], v[11]);
    dft4(v[12], v[13], v[14], v[15]);
    // v[4 k2 + k1] holds y[k2 + 4 k1]: transpose the 4x4 block
    X t;
    t = v[1]; v[1] = v[4]; v[4] = t;
    t = v[2]; v[2] = v[8]; v[8] = t;
    t = v[3]; v[3] = v[12]; v[12] = t;
    t = v[6]; v[6] = v[9]; v[9] = t;
    t = v[7]; v[7] = v[13]; v[13] = t;
    t = v[11]; v[11] = v[14]; v[14] = t;
}

template <class X> RK_HD void dft3(X* v) {
    using F = real_t<X>;
    X t = c_add(v[1], v[2]);
    X m = cx<X>(v[0].x - (F)0.5 * t.x, v[0].y - (F)0.5 * t.y);
    X d = c_sub(v[1], v[2]);
    X s = cx<X>((F)RK_S3 * d.y, -(F)RK_S3 * d.x);   // -i sin(2pi/3) d
    v[0] = c_add(v[0], t);
    v[1] = c_add(m, s);
    v[2] = c_sub(m, s);
}

template <class X> RK_HD void dft5(X* v) {
    using F = real_t<X>;
    const F c1 = (F)RK_C5_1, c2 = (F)RK_C5_2, s1 = (F)RK_S5_1, s2 = (F)RK_S5_2;
    X t1 = c_add(v[1], v[4]), t2 = c_add(v[2], v[3]);
    X t3 = c_sub(v[1], v[4]), t4 = c_sub(v[2], v[3]);
    X a0 = v[0];
    X b1 = cx<X>(a0.x + c1 * t1.x + c2 * t2.x, a0.y + c1 * t1.y + c2 * t2.y);
    X b2 = cx<X>(a0.x + c2 * t1.x + c1 * t2.x, a0.y + c2 * t1.y + c1 * t2.y);
    // u1 = s1 t3 + s2 t4, u2 = s2 t3 - s1 t4; y1 = b1 - i u1, y2 = b2 - i u2
    X u1 = cx<X>(s1 * t3.x + s2 * t4.x, s1 * t3.y + s2 * t4.y);
    X u2 = cx<X>(s2 * t3.x - s1 * t4.x, s2 * t3.y - s1 * t4.y);
    v[0] = cx<X>(a0.x + t1.x + t2.x, a0.y + t1.y + t2.y);
    v[1] = c_add(b1, c_mul_mi(u1));
    v[4] = c_sub(b1, c_mul_mi(u1));
    v[2] = c_add(b2, c_mul_mi(u2));
    v[3] = c_sub(b2, c_mul_mi(u2));
}

// Odd prime radix 7: y_k = A_k - i B_k, y_{7-k} = A_k + i B_k with
// A_k = a0 + sum_n cos(2 pi n k/7)(a_n + a_{7-n}), B_k = sum_n sin(2 pi n k/7)(a_n - a_{7-n}).
template <class X> RK_HD void dft7(X* v) {
    using F = real_t<X>;
    const F c[4] = {(F)1, (F)RK_C7_1, (F)RK_C7_2, (F)RK_C7_3};
    const F s[4] = {(F)0, (F)RK_S7_1, (F)RK_S7_2, (F)RK_S7_3};
    X p[4], m[4];
    for (int n = 1; n <= 3; ++n) {
        p[n] = c_add(v[n], v[7 - n]);
        m[n] = c_sub(v[n], v[7 - n]);
    }
    X a0 = v[0];
    v[0] = cx<X>(a0.x + p[1].x + p[2].x + p[3].x, a0.y + p[1].y + p[2].y + p[3].y);
    for (int k = 1; k <= 3; ++k) {
        X A = a0, B = cx<X>((F)0, (F)0);
        for (int n = 1; n <= 3; ++n) {
            int nk = (n * k) % 7;
            F cc = nk <= 3 ? c[nk] : c[7 - nk];
            F ss = nk <= 3 ? s[nk] : -s[7 - nk];
            A.x += cc * p[n].x; A.y += cc * p[n].y;
            B.x += ss * m[n].x; B.y += ss * m[n].y;
        }
        v[k] = c_add(A, c_mul_mi(B));
        v[7 - k] = c_sub(A, c_mul_mi(B));
    }
}

template <int R, class X> RK_HD void dft(X* v);

// N1 x N2 points, N1 and N2 coprime: with n = N2 n1 + N1 n2 and k = N2 a k1 +
// N1 b k2 modulo N (a, b the inverses of N2 modulo N1 and N1 modulo N2) the
// DFT separates without twiddles (Good 1958).
constexpr int inverse_mod(int x, int m) {
    for (int y = 1; y < m; ++y)
        if ((x * y) % m == 1) return y;
    return 1;
}
template <int N1, int N2, class X> RK_HD void dft_coprime(X* v) {
    constexpr int N = N1 * N2, E1 = N2 * inverse_mod(N2, N1), E2 = N1 * inverse_mod(N1, N2);
    X t[N];
#pragma unroll
    for (int n2 = 0; n2 < N2; ++n2) {
        X c[N1];
#pragma unroll
        for (int n1 = 0; n1 < N1; ++n1) c[n1] = v[(N2 * n1 + N1 * n2) % N];
        dft<N1>(c);
#pragma unroll
        for (int k1 = 0; k1 < N1; ++k1) t[k1 * N2 + n2] = c[k1];
    }
#pragma unroll
    for (int k1 = 0; k1 < N1; ++k1) {
        dft<N2>(&t[k1 * N2]);
#pragma unroll
        for (int k2 = 0; k2 < N2; ++k2) v[(E1 * k1 + E2 * k2) % N] = t[k1 * N2 + k2];
    }
}

// a * (c + cl - i (s + sl)), the constants' rounding errors included: 9 = 3 x 3
// multiplies by the same three twiddles wherever it occurs, and their errors,
// shared by all of a transform's butterflies, made 729 = 9 * 9 * 9 2.4 % less
// accurate than 3^6 with its tables.
template <class X> RK_HD X mul_w9(X a, real_t<X> c, real_t<X> cl, real_t<X> s, real_t<X> sl) {
    return cx<X>(a.x * c + (a.y * s + (a.y * sl + a.x * cl)), a.y * c - (a.x * s + (a.x * sl - a.y * cl)));
}

// 9 = 3 x 3: DFT3 over n2 for each n1 (x[n1 + 3 n2]), twiddle W9^{n1 k2},
// DFT3 over n1 for each k2, output y[k2 + 3 k1].
template <class X> RK_HD void dft9(X* v) {
    using F = real_t<X>;
    // one value's real type: a double subtracted from a pair's vector is rounded
    // to float first, which leaves no residual
    using S = real_t<scalar_t<X>>;
    X t[9];
#pragma unroll
    for (int n1 = 0; n1 < 3; ++n1) {
        X c[3] = {v[n1], v[n1 + 3], v[n1 + 6]};
        dft3(c);
#pragma unroll
        for (int k2 = 0; k2 < 3; ++k2) t[3 * k2 + n1] = c[k2];
    }
    const F c1 = (S)RK_C9_1, c1l = (S)(RK_C9_1 - (S)RK_C9_1 + 2.175e-17), s1 = (S)RK_S9_1, s1l = (S)(RK_S9_1 - (S)RK_S9_1 - 3.660e-17);
    const F c2 = (S)RK_C9_2, c2l = (S)(RK_C9_2 - (S)RK_C9_2 - 1.009e-17), s2 = (S)RK_S9_2, s2l = (S)(RK_S9_2 - (S)RK_S9_2 + 3.905e-17);
    const F c4 = (S)RK_C9_4, c4l = (S)(RK_C9_4 - (S)RK_C9_4 + 4.385e-17), s4 = (S)RK_S9_4, s4l = (S)(RK_S9_4 - (S)RK_S9_4 + 2.014e-17);
    t[4] = mul_w9(t[4], c1, c1l, s1, s1l);
    t[5] = mul_w9(t[5], c2, c2l, s2, s2l);
    t[7] = mul_w9(t[7], c2, c2l, s2, s2l);
    t[8] = mul_w9(t[8], c4, c4l, s4, s4l);
#pragma unroll
    for (int k2 = 0; k2 < 3; ++k2) {
        dft3(&t[3 * k2]);
#pragma unroll
        for (int k1 = 0; k1 < 3; ++k1) v[k2 + 3 * k1] = t[3 * k2 + k1];
    }
}

template <int R, class X> RK_HD void dft(X* v) {
    if constexpr (R == 2) dft2(v[0], v[1]);
    else if constexpr (R == 3) dft3(v);
    else if constexpr (R == 4) dft4(v[0], v[1], v[2], v[3]);
    else if constexpr (R == 5) dft5(v);
    else if constexpr (R == 7) dft7(v);
    else if constexpr (R == 6) dft_coprime<2, 3>(v);
    else if constexpr (R == 8) dft8(v);
    else if constexpr (R == 9) dft9(v);
    else if constexpr (R == 10) dft_coprime<2, 5>(v);
    else if constexpr (R == 12) dft_coprime<4, 3>(v);
    else if constexpr (R == 15) dft_coprime<3, 5>(v);
    else if constexpr (R == 16) dft16(v);
    else static_assert(R == 1, "radix without a butterfly");
}

// The same with zeros in the upper half of the inputs (even R): the first
// stage of a Bluestein transform, whose M >= 2N-1 points hold N <= M/2 values.
template <class X> RK_HD void dft4_lower(X& a0, X& a1, X& a2, X& a3) {
    const X x = a0, y = a1, t = c_mul_mi(a1);
    a0 = c_add(x, y);
    a2 = c_sub(x, y);
    a1 = c_add(x, t);
    a3 = c_sub(x, t);
}

template <int R, class X> RK_HD void dft_lower(X* v) {
    using F = real_t<X>;
    if constexpr (R == 2) {
        v[1] = v[0];
    } else if constexpr (R == 4) {
        dft4_lower(v[0], v[1], v[2], v[3]);
    } else if constexpr (R == 8) {
        X e0 = v[0], e1 = v[2], e2, e3, o0 = v[1], o1 = v[3], o2, o3;
        dft4_lower(e0, e1, e2, e3);
        dft4_lower(o0, o1, o2, o3);
        o1 = c_w8_1(o1);
        o2 = c_mul_mi(o2);
        o3 = c_w8_3(o3);
        v[0] = c_add(e0, o0); v[4] = c_sub(e0, o0);
        v[1] = c_add(e1, o1); v[5] = c_sub(e1, o1);
        v[2] = c_add(e2, o2); v[6] = c_sub(e2, o2);
        v[3] = c_add(e3, o3); v[7] = c_sub(e3, o3);
    } else if constexpr (R == 16) {
        dft4_lower(v[0], v[4], v[8], v[12]);
        dft4_lower(v[1], v[5], v[9], v[13]);
        dft4_lower(v[2], v[6], v[10], v[14]);
        dft4_lower(v[3], v[7], v[11], v[15]);
        dft16_second(v);
    } else {
        const X zero = cx<X>((F)0, (F)0);
#pragma unroll
        for (int r = R / 2; r < R; ++r) v[r] = zero;
        dft<R>(v);
    }
}

// ------------------------------------------------------------------------
// compile-time radix plan of a length L = 2^a 3^b 5^c 7^d
// ------------------------------------------------------------------------
struct RadixList {
    int n;
    int r[24];
};

// Prime powers only: 16s, the rest of the powers of two, 7s, 5s, 3s, the
// largest in front (it fixes T = L / r[0] threads per instance).
__host__ __device__ constexpr RadixList prime_power_list(int L) {
    RadixList s = {0, {0}};
    int x = L, p2 = 0, n3 = 0, n5 = 0, n7 = 0;
    while (x % 2 == 0) { x /= 2; ++p2; }
    while (x % 3 == 0) { x /= 3; ++n3; }
    while (x % 5 == 0) { x /= 5; ++n5; }
    while (x % 7 == 0) { x /= 7; ++n7; }
    while (p2 >= 4) { s.r[s.n++] = 16; p2 -= 4; }
    if (p2 > 0) s.r[s.n++] = 1 << p2;
    for (int k = 0; k < n7; ++k) s.r[s.n++] = 7;
    for (int k = 0; k < n5; ++k) s.r[s.n++] = 5;
    for (int k = 0; k < n3; ++k) s.r[s.n++] = 3;
    if (s.n == 0) s.r[s.n++] = 1;
    // move the largest radix to the front (e.g. [4, 5, 5] -> [5, 4, 5])
    int imax = 0;
    for (int k = 1; k < s.n; ++k)
        if (s.r[k] > s.r[imax]) imax = k;
    int t = s.r[0]; s.r[0] = s.r[imax]; s.r[imax] = t;
    return s;
}

// Cost of a radix sequence (make_radix_list); fits: at most 20 values per thread.
__host__ __device__ constexpr long long radix_cost(int L, const int* r, int n, bool* fits) {
    const int kCost[17] = {0, 0, 4, 16, 16, 40, 40, 84, 60, 120, 100, 0, 112, 0, 0, 200, 168};
    const int T = L / r[0];
    long long c = r[0] == 15 ? 200 : 0;
    for (int s = 0; s < n; ++s) {
        const int q = (L / r[s] + T - 1) / T;
        if (fits) *fits = *fits && q * r[s] <= 20;
        c += q * (kCost[r[s]] + 14 * r[s]);
    }
    return c * T + 6ll * n * L;
}

// The radix plan of a length (build.py radix_list mirrors it).  Powers of two
// take their 16s.  Other lengths take, of all factorisations into the radices
// below, the cheapest: a stage costs every thread of T = L / r[0] its
// ceil(L / R / T) butterflies (operations of the DFT, plus 14 per value for
// twiddles, LDS and addresses), idle threads included, and each stage its
// barriers (6 per value of the instance); a 15 in front, whose outputs lie 16
// padded slots apart in LDS, pays for its bank conflicts.  The prime powers stay
// unless that is 10 % cheaper, and rows of at least 32 threads keep them (below
// 32 a contiguous side is staged through LDS), as those of at least 20 do
// rather than go below 10 (30000 x 81: 9.7 us with 27 threads, 10.6 with 9) and
// those of at least 15 rather than go below 6 (30000 x 75: 9.4 us with 15
// threads, 12.2 with 5, whose tiles of 51 instances leave a CU four
// work-groups).  Composite radices leave 1000 = 10 * 10 * 10 where prime powers gave 8 * 5 * 5 * 5 and 1080 = 12 * 15 * 6
// for 8 * 5 * 3 * 3 * 3: fewer exchanges and fewer idle threads.  At most 20
// values per thread, and at most 256 threads up to 4096 points (the batch
// kernel's work-group).  Prime powers / composite radices, us: rows 4096 x
// 1000 15.3 / 12.9, 2048 x 2000 22.4 / 16.0, 500 x 1200 9.4 / 6.0; columns
// 1440 x 1440 17.5 / 11.9, 200 x 360000 543 / 509; 192 cubed 68.0 / 62.1,
// 160 cubed 45.2 / 40.9.
__host__ __device__ constexpr RadixList make_radix_list(int L) {
    const int kR[12] = {16, 15, 12, 10, 9, 8, 7, 6, 5, 4, 3, 2};
    RadixList best = prime_power_list(L);
    if ((L & (L - 1)) == 0 || L < 6) return best;
    long long best_cost = radix_cost(L, best.r, best.n, nullptr) * 9 / 10;
    const int T0 = L / best.r[0];
    // depth-first over non-increasing radix sequences: idx[d] is the radix of
    // depth d, rem[d] what is left to factor before it
    int idx[16] = {0}, rem[17] = {0}, d = 0;
    rem[0] = L;
    idx[0] = -1;
    while (d >= 0) {
        int k = idx[d] + 1;
        while (k < 12 && rem[d] % kR[k] != 0) ++k;
        if (k == 12 || d > 7) {
            --d;
            continue;
        }
        idx[d] = k;
        rem[d + 1] = rem[d] / kR[k];
        if (rem[d + 1] > 1) {
            idx[d + 1] = k - 1;   // non-increasing: start at the same radix
            ++d;
            continue;
        }
        const int n = d + 1;
        for (int f = 0; f < n; ++f) {   // each distinct radix in front
            if (f > 0 && idx[f] == idx[f - 1]) continue;
            const int T = L / kR[idx[f]];
            if (T > 1024 || (L <= 4096 && T > 256) || (T < 32 && T0 >= 32) || (T < 10 && T0 >= 20) || (T < 6 && T0 >= 15)) continue;
            int r[16] = {kR[idx[f]]}, m = 1;
            for (int s = 0; s < n; ++s)
                if (s != f) r[m++] = kR[idx[s]];
            bool fits = true;
            const long long c = radix_cost(L, r, n, &fits);
            if (!fits || c >= best_cost) continue;
            best_cost = c;
            best.n = n;
            for (int s = 0; s < n; ++s) best.r[s] = r[s];
        }
    }
    return best;
}

__host__ __device__ constexpr bool is_supported_length(int L) {
    int x = L;
    if (x < 1) return false;
    while (x % 2 == 0) x /= 2;
    while (x % 3 == 0) x /= 3;
    while (x % 5 == 0) x /= 5;
    while (x % 7 == 0) x /= 7;
    return x == 1;
}

template <int L> struct Plan {
    static constexpr RadixList RL = make_radix_list(L);
    static constexpr int NSTAGE = RL.n;
    static constexpr int R0 = RL.r[0];
    static constexpr int T = L / R0;
    static constexpr int radix(int s) { return RL.r[s]; }
    static constexpr int ns(int s) {
        int p = 1;
        for (int k = 0; k < s; ++k) p *= RL.r[k];
        return p;
    }
    static constexpr int nb(int s) { return L / RL.r[s]; }
    static constexpr int q(int s) { return (L / RL.r[s] + T - 1) / T; }
    static constexpr int vmax() {
        int m = 0;
        for (int s = 0; s < RL.n; ++s)
            if (q(s) * RL.r[s] > m) m = q(s) * RL.r[s];
        return m;
    }
};

// LDS layout of one instance: one padding slot every 16 complex values.
RK_HD constexpr int lds_pad(int p) { return p + (p >> 4); }
// lds_pad(b + c) for a run-time b >= 0 with b % 16 < BM and a c >= 0 that is a
// constant once the caller's loops are unrolled.  When b % 16 + c % 16 < 16
// no padding slot falls between b and b + c, and the padded position is
// lds_pad(b) + lds_pad(c): one address register per exchange, the constant in
// the LDS instruction's offset field, where the plain form costs a register
// and three instructions per value (the compiler does not split a shift of a
// sum whose low bits it cannot see).
template <int BM> RK_HD constexpr int lds_pad_add(int b, int c) {
    return (BM - 1) + (c & 15) < 16 ? lds_pad(b) + lds_pad(c) : lds_pad(b + c);
}
// Base row pitch of the instances of a tile: odd, so that lanes walking
// adjacent instances hit distinct banks.
RK_HD constexpr int lds_pitch_base(int L) {
    int s = lds_pad(L - 1) + 1;
    return (s % 2 == 0) ? s + 1 : s;
}
// A tile's exchanges go through halves (real parts, then imaginary parts)
// when it needs more than 80 KB at the base pitch; ES is the element size
// (8 bytes complex64, 16 complex128).
RK_HD constexpr bool lds_split(int L, int C, int ES = 8) { return C * lds_pitch_base(L) * ES > 80 * 1024; }
// Row pitch of a tile of C instances of L points (T threads each).  Under the
// column mapping a wave covers C instances x 64/C threads.  For C a power of
// two from 2 to 16 (32 when split) and T >= 16, an odd pitch stacks the C
// instances' accesses on the same banks; a pitch of m/C modulo m (m = 32
// slots of 64-bit accesses, or 64 banks of split 32-bit accesses) gives each
// instance its own share of the banks.  (A bank model of every exchange of
// every catalogue tile: 1.2-3x fewer conflict cycles where this applies,
// averaged over load/store modes and both mappings; the other tiles keep the
// odd pitch, which the model favours for them.)  Complex128 tiles keep the
// odd pitch (the rule is for 64-bit accesses and their 32-bit halves).
RK_HD constexpr int lds_pitch_for(int L, int C, int T, bool force_split = false, int ES = 8) {
    if (ES != 8) return lds_pitch_base(L);
    const bool split = force_split || lds_split(L, C);
    const bool pow2 = C > 0 && (C & (C - 1)) == 0;
    if (!pow2 || C < 2 || T < 16 || C > (split ? 32 : 16)) return lds_pitch_base(L);
    const int m = split ? 64 : 32;
    const int target = m / C;
    int p = lds_pad(L - 1) + 1;
    while (p % m != target) ++p;
    return p;
}

// Row pitch (in 64-bit slots) and LDS bytes of a pair tile of C instances:
// C/2 rows of 64-bit values, the pitch rule of 64-bit accesses above.
RK_HD constexpr int lds_pitch_pair(int L, int C, int T) {
    const int CP = C / 2;
    const bool pow2 = CP > 0 && (CP & (CP - 1)) == 0;
    if (!pow2 || CP < 2 || T < 16 || CP > 16) return lds_pitch_base(L);
    int p = lds_pad(L - 1) + 1;
    while (p % 32 != 32 / CP) ++p;
    return p;
}
RK_HD constexpr int pair_lds_bytes(int L, int C, int T) { return (C / 2) * lds_pitch_pair(L, C, T) * 8; }

// ------------------------------------------------------------------------
// per-instance coordinates
// ------------------------------------------------------------------------
struct Inst {
    rk_u64 o, i, l;
    rk_u64 jpass;    // h*NS + l: axis position of input element 0
    rk_u64 kbase;    // h*NS*L + l: axis position of output element 0
    rk_i64 in_base, out_base;
    bool valid;
};

// x / d for x < 2^31 with the host's round-up multiplier m and shift s.
__device__ __forceinline__ rk_u32 magic_div(rk_u32 x, rk_u32 m, rk_u32 s) { return (__umulhi(x, m) + x) >> s; }

template <int L>
__device__ __forceinline__ Inst decompose(const rk_pass_args& a, rk_u64 inst) {
    Inst r;
    r.valid = inst < a.n_inst;
    rk_u64 x = r.valid ? inst : 0;
    rk_u64 i = 0, l = 0, h = 0;
    if (a.div_magic) {   // a multiply and a shift per division instead of a division sequence
        rk_u32 y = (rk_u32)x, q;
        if (a.dim_I > 1) { q = magic_div(y, a.mag_I, a.sh_I); i = y - q * (rk_u32)a.dim_I; y = q; }
        if (a.dim_NS > 1) { q = magic_div(y, a.mag_NS, a.sh_NS); l = y - q * (rk_u32)a.dim_NS; y = q; }
        if (a.dim_H > 1) { q = magic_div(y, a.mag_H, a.sh_H); h = y - q * (rk_u32)a.dim_H; y = q; }
        x = y;
    } else {
        if (a.dim_I > 1) { i = x % a.dim_I; x /= a.dim_I; }
        if (a.dim_NS > 1) { l = x % a.dim_NS; x /= a.dim_NS; }
        if (a.dim_H > 1) { h = x % a.dim_H; x /= a.dim_H; }
    }
    r.o = x;
    r.i = i;
    r.l = l;
    r.jpass = h * a.dim_NS + l;
    r.kbase = h * a.dim_NS * (rk_u64)L + l;
    r.in_base = a.in_off + (rk_i64)x * a.in_so + (rk_i64)i * a.in_si;
    r.out_base = a.out_off + (rk_i64)x * a.out_so + (rk_i64)i * a.out_si;
    return r;
}

// Axis position of a pair's second instance minus its first's: pairs are
// adjacent along the innermost of the dims I, NS, H that is longer than one.
__device__ __forceinline__ rk_u64 pair_step(const rk_pass_args& a) { return a.dim_I > 1 ? 0 : 1; }

// W_N^e for 0 <= e < N from two FP64 tables; the product is formed in FP64
// and rounded once to the element's real type.
__device__ __forceinline__ double2 d_mul(double2 a, double2 b) {
    return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

__device__ __forceinline__ double2 twiddle_n64(const rk_pass_args& a, rk_u64 e) {
    return d_mul(a.tw_hi[e >> a.tw_shift], a.tw_lo[e & a.tw_mask]);
}

// The inter-pass twiddles of one thread, W_N^{p*l*tw_mult} for p = p0, p0+dp,
// p0+2dp, ...: two table lookups for the first one and the step, then an FP64
// recurrence; every value is rounded once to the element's real type.
struct TwiddleWalk {
    double2 w, s;
    __device__ __forceinline__ void init(const rk_pass_args& a, rk_u64 l, rk_u64 p0, rk_u64 dp) {
        const rk_u64 lm = l * a.tw_mult;
        w = twiddle_n64(a, p0 * lm);
        s = twiddle_n64(a, dp * lm);
    }
    template <class X> __device__ __forceinline__ X next() {
        const X r = cx<X>((real_t<X>)w.x, (real_t<X>)w.y);
        w = d_mul(w, s);
        return r;
    }
};

// The inter-pass twiddles of one thread's values x[r] at positions p0 + r*dp
// of instance l.  (An exact FP32 table of W_{NS*L}^j read at index l*p was
// measured instead: on 64 x 2^20 the 128-point middle pass went from 181 to
// 226 us, its lanes' table reads scattered over many cache lines per load,
// while the FP64 walk costs VALU only.)
template <int NV, class X>
__device__ __forceinline__ void apply_pass_twiddles(const rk_pass_args& a, rk_u64 l, int p0, int dp, X* x) {
    TwiddleWalk tw;
    tw.init(a, l, (rk_u64)p0, (rk_u64)dp);
#pragma unroll
    for (int r = 0; r < NV; ++r) x[r] = c_mul(x[r], tw.template next<X>());
}

// Two instances per thread: one walk per instance (equal when the pair
// differs in its inner batch index only).
template <int NV>
__device__ __forceinline__ void apply_pass_twiddles(const rk_pass_args& a, rk_u64 l, int p0, int dp, cpair2* x) {
    TwiddleWalk tw0, tw1;
    tw0.init(a, l, (rk_u64)p0, (rk_u64)dp);
    tw1.init(a, l + pair_step(a), (rk_u64)p0, (rk_u64)dp);
#pragma unroll
    for (int r = 0; r < NV; ++r) {
        const float2 w0 = tw0.template next<float2>(), w1 = tw1.template next<float2>();
        cpair2 w;
        w.x = rk_v2<float>{w0.x, w1.x};
        w.y = rk_v2<float>{w0.y, w1.y};
        x[r] = c_mul(x[r], w);
    }
}

// The table pointers of the pass arguments, as the element type X of a pass
// (complex64 or complex128 tables; the host builds the ones its plan needs).
template <class X> __device__ __forceinline__ const scalar_t<X>* table(const float2* p) {
    return reinterpret_cast<const scalar_t<X>*>(p);
}

// The output scale (1/N on the last pass of an inverse transform) in the
// element's real type: complex128 passes take the FP64 value.
template <class X> __device__ __forceinline__ real_t<X> out_scale_of(const rk_pass_args& a) {
    if constexpr (sizeof(real_t<scalar_t<X>>) == 8) return a.out_scale64;
    else return a.out_scale;
}

// Plain strided element access: the identity IO policy.
// An IO policy is an object with load(a, o, m, i, addr) and
// store(a, o, k, i, addr, v): o / i are the flat indices over the dims before /
// after the transformed axis, m / k the axis position, addr the plain strided
// element address.  Fused transformations (generated at run time) use o, m, i.
// kBranchFree: a lane with nothing to load loads a valid element instead (its
// instance's first position, or the tile's first instance: valid indices o,
// m, i and a valid address) and discards it, so every load of a thread is
// issued without a branch around it (a branch per load serialises them on
// their completion).
// Streaming variant (NT = true): every load and store carries the
// nontemporal hint, so a pass whose input and output far exceed the 256 MB
// Infinity Cache does not fill it and the L2 with lines nothing reads again
// (measured on 64 x 2^20: 0.640 -> 0.599 ms; a hand-written copy of 512 MiB
// runs at 5.8 TB/s plain and 6.0 TB/s with the hint).  Passes whose data fit
// in that cache keep the plain accesses: the hint costs the 256^3 transform,
// whose in-place passes re-read what the previous pass just wrote, 22 %.
// The hint is chosen per side (NTL loads, NTS stores): a chunked chain whose
// intermediate stays in that cache between passes streams only its first
// pass's loads and its last pass's stores.  X is the element type
// (complex64 float2, complex128 double2); every IO policy names it value_type.
// kPtr: elements are also reached by their 64-bit address in global memory
// (load_p / store_p), so a thread walks its elements with one address.
#define RK_GLOBAL(T, p) reinterpret_cast<T __attribute__((address_space(1)))*>(p)
template <class IO, class = void> struct HasPtr { static constexpr bool value = false; };
template <class IO> struct HasPtr<IO, decltype((void)IO::kPtr)> { static constexpr bool value = true; };

template <bool NTL, bool NTS = NTL, class X = float2> struct GlobalIO {
    using value_type = X;
    static constexpr bool kBranchFree = true;
    static constexpr bool kPtr = true;
    __device__ __forceinline__ X load(const rk_pass_args& a, rk_u64 /*o*/, rk_u64 /*m*/, rk_u64 /*i*/,
                                      rk_i64 addr) const {
        return load_p(reinterpret_cast<rk_u64>(reinterpret_cast<const X*>(a.in) + addr));
    }
    __device__ __forceinline__ X load_p(rk_u64 p) const {
        auto q = RK_GLOBAL(const rk_v2<real_t<X>>, p);
        rk_v2<real_t<X>> x;
        if constexpr (NTL) x = __builtin_nontemporal_load(q);
        else x = *q;
        return cx<X>(x.x, x.y);
    }
    __device__ __forceinline__ void store(const rk_pass_args& a, rk_u64 /*o*/, rk_u64 /*k*/, rk_u64 /*i*/,
                                          rk_i64 addr, X v) const {
        store_p(reinterpret_cast<rk_u64>(reinterpret_cast<X*>(a.out) + addr), v);
    }
    __device__ __forceinline__ void store_p(rk_u64 p, X v) const {
        auto q = RK_GLOBAL(rk_v2<real_t<X>>, p);
        const rk_v2<real_t<X>> x = {v.x, v.y};
        if constexpr (NTS) __builtin_nontemporal_store(x, q);
        else *q = x;
    }
};
using PlainIO = GlobalIO<false>;
using StreamIO = GlobalIO<true>;

// Two adjacent instances per thread (complex64, column tiles): their elements
// at one position are neighbours in memory, so a load or store moves 16 bytes
// per lane, half as many vector-memory instructions per element.  The element
// address need not be 16-byte aligned (an instance pair starts at any even
// element of the caller's view).
typedef float rk_v4u __attribute__((ext_vector_type(4), aligned(8)));
template <bool NTL, bool NTS = NTL> struct PairIO {
    using value_type = cpair2;
    static constexpr bool kBranchFree = true;
    static constexpr bool kPtr = true;
    __device__ __forceinline__ cpair2 load_p(rk_u64 p) const {
        auto q = RK_GLOBAL(const rk_v4u, p);
        rk_v4u v;
        if constexpr (NTL) v = __builtin_nontemporal_load(q);
        else v = *q;
        return cx<cpair2>(rk_v2<float>{v.x, v.z}, rk_v2<float>{v.y, v.w});
    }
    // two consecutive complex values at p
    __device__ __forceinline__ void store_run(rk_u64 p, float x0, float y0, float x1, float y1) const {
        auto q = RK_GLOBAL(rk_v4u, p);
        const rk_v4u v = {x0, y0, x1, y1};
        if constexpr (NTS) __builtin_nontemporal_store(v, q);
        else *q = v;
    }
    __device__ __forceinline__ void store_p(rk_u64 p, cpair2 v) const { store_run(p, v.x.x, v.y.x, v.x.y, v.y.y); }
};

// Plain strided IO whose loads and stores are coherent across the whole
// device (relaxed agent-scope atomics: they bypass the caches that are not
// shared by all CUs).  Used where one kernel launch hands data from one
// work-group to another: after the producer's stores have completed, a
// counter in memory is enough to publish them, with no cache write-back or
// invalidation in between.  (Choosing cached or coherent accesses per pass
// with a run-time branch was measured: the second code path raised the
// batch kernel from 160 to 200 VGPRs and cost more than it saved.)
struct CoherentIO {
    using value_type = float2;
    static constexpr bool kBranchFree = true;
    static constexpr bool kPtr = true;
    __device__ __forceinline__ float2 load(const rk_pass_args& a, rk_u64 /*o*/, rk_u64 /*m*/, rk_u64 /*i*/,
                                           rk_i64 addr) const {
        return load_p(reinterpret_cast<rk_u64>(a.in + addr));
    }
    __device__ __forceinline__ float2 load_p(rk_u64 p) const {
        const rk_u64 bits = __hip_atomic_load(RK_GLOBAL(rk_u64, p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return make_float2(__uint_as_float((unsigned)bits), __uint_as_float((unsigned)(bits >> 32)));
    }
    __device__ __forceinline__ void store(const rk_pass_args& a, rk_u64 /*o*/, rk_u64 /*k*/, rk_u64 /*i*/,
                                          rk_i64 addr, float2 v) const {
        store_p(reinterpret_cast<rk_u64>(a.out + addr), v);
    }
    __device__ __forceinline__ void store_p(rk_u64 p, float2 v) const {
        const rk_u64 bits = (rk_u64)__float_as_uint(v.x) | ((rk_u64)__float_as_uint(v.y) << 32);
        __hip_atomic_store(RK_GLOBAL(rk_u64, p), bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
};

// Compile-time pass variant: which pre-/post-ops the pass applies and whether
// it is the single-kernel Bluestein convolution.  Keeping them out of the
// run-time arguments keeps plain passes free of table loads (and registers).
#define RK_VAR_PRE_NONE 0
#define RK_VAR_PRE_TWIDDLE 1
#define RK_VAR_PRE_CHIRP 2
#define RK_VAR_POST_NONE 0
#define RK_VAR_POST_KMUL_CONJ 1
#define RK_VAR_POST_CONJ_CHIRP 2
#define RK_VARIANT(pre, post, blue) ((pre) | ((post) << 2) | ((blue) << 4))
// Bit of a catalogue kernel's variant number (not of Variant<V>): the kernel
// uses StreamIO instead of PlainIO.
#define RK_VAR_STREAM 128
// Bits of a catalogue kernel's variant number: the kernel has the pass's load
// and store modes compiled in (DIRECT/DIRECT, DIRECT/FLAT, FLAT/FLAT) instead of reading
// them from the pass arguments.  The run-time switch keeps the code of every
// mode alive in one kernel: a 96-point tile holds 146 VGPRs with it and 75-82
// with its modes fixed.
#define RK_VAR_MODE_DD 256
#define RK_VAR_MODE_DF 512
#define RK_VAR_MODE_FF 1024
// Bits of a catalogue kernel's variant number: nontemporal loads only / stores
// only (GlobalIO<true, false> / GlobalIO<false, true>; RK_VAR_STREAM is both).
#define RK_VAR_NT_LOAD 2048
#define RK_VAR_NT_STORE 4096
// Bit of a catalogue kernel's variant number: the row mapping is compiled in
// and each wave holds whole instances (64 % T == 0), so the exchanges between
// Stockham stages stay inside one wave and need no work-group barrier; only
// the staged global sides (COLUMN, FLAT) exchange across waves.
#define RK_VAR_WAVE 8192
// Bit of a catalogue kernel's variant number: the persistent, software-
// pipelined body (fft_pass_body_pipe; DIRECT loads only).
#define RK_VAR_PIPE 16384
// Bit of a catalogue kernel's variant number: the tile's exchanges go through
// re/im halves even when the whole tile would fit (half the LDS per
// work-group, twice the resident work-groups).
#define RK_VAR_HALF 32768
// Bit of a catalogue kernel's variant number: the launch bounds ask for as
// many resident work-groups per CU as the tile's LDS allows, so the register
// budget does not cut the residency to fewer.
#define RK_VAR_OCC 65536
// Bit of a kernel's variant number: complex128 elements (FP64 butterflies,
// twiddles and tables); such kernels come from the run-time compiler only.
#define RK_VAR_F64 131072
// Bit of a kernel's variant number: two adjacent instances per thread (PairIO;
// DIRECT/DIRECT or DIRECT/FLAT compiled in, complex64).
#define RK_VAR_PAIR 262144
// MODES template argument of fft_pass_tile: 0 reads the modes from the pass
// arguments, RK_MODES(load, store) compiles them in.
#define RK_MODES(load, store) (16 | (int)(load) | ((int)(store) << 2))
template <int V> struct Variant {
    static constexpr int PRE = V & 3;
    static constexpr int POST = (V >> 2) & 3;
    static constexpr bool BLUE = ((V >> 4) & 1) != 0;
};

// Padded sides: only a Bluestein chirp pass reads positions beyond its data
// (the input beyond n_valid_in reads as zero) and only the last pass of a
// Bluestein chain leaves positions unwritten (beyond n_valid_out); every
// other pass reads and writes all N positions of its axis (the planners check
// this), so its elements need no per-element bounds.
template <int V> __host__ __device__ constexpr bool pad_in() { return Variant<V>::PRE == RK_VAR_PRE_CHIRP; }
template <int V> __host__ __device__ constexpr bool pad_out() { return Variant<V>::POST == RK_VAR_POST_CONJ_CHIRP; }

// A Bluestein transform of N <= M/2 values over its M points (the planners
// check this): the inputs of a chirp pass at or beyond the middle of its axis
// are zero and the outputs of its last pass there are not stored, so with an
// even radix R the upper R/2 of a thread's first-stage inputs need no load, no
// chirp and no addition, and the upper R/2 of its last-stage outputs no store
// (lower_in, lower_out).
template <int V> __host__ __device__ constexpr bool lower_in(int R) { return pad_in<V>() && R % 2 == 0; }
template <int V> __host__ __device__ constexpr bool lower_out(int R) { return pad_out<V>() && R % 2 == 0; }

// One thread's walk over the positions p0 + c of one instance on one side
// (c a compile-time offset): axis position and element address of position p0
// and their uniform steps per unit of c, formed once per thread.
struct Walk {
    rk_u64 m0, mstep;   // axis position of position p0, and per unit of c
    rk_i64 a0, astep;   // element address of position p0, and per unit of c
};

__device__ __forceinline__ Walk in_walk(const rk_pass_args& a, const Inst& ic, int p0) {
    Walk w;
    w.m0 = ic.jpass + (rk_u64)p0 * a.pos_mult;
    w.mstep = a.pos_mult;
    w.a0 = ic.in_base + (rk_i64)w.m0 * a.in_sa;
    w.astep = (rk_i64)a.pos_mult * a.in_sa;
    return w;
}

// output position k of an instance sits at axis position kbase + k * dim_NS
__device__ __forceinline__ Walk out_walk(const rk_pass_args& a, const Inst& ic, int k0) {
    Walk w;
    w.m0 = ic.kbase + (rk_u64)k0 * a.dim_NS;
    w.mstep = a.dim_NS;
    w.a0 = ic.out_base + (rk_i64)w.m0 * a.out_sa;
    w.astep = (rk_i64)a.dim_NS * a.out_sa;
    return w;
}

// Address or offset + step, hidden from the optimiser: an element then costs
// one 64-bit add.  Left alone, the compiler rewrites a thread's unrolled
// addresses p0 + r * step into one or two quarter-rate 64-bit multiply-adds and
// register moves per element, a quarter of the 256-point column tile's VALU
// cycles; the same for the stage-twiddle offsets.  walk_step is the uniform
// byte step, kept in scalar registers.  With the direction's conjugation and
// scale behind a branch instead of selects: 33 x 65521 87 -> 74 us, 4096 x 997
// 38.8 -> 35.2, 64 x 2^20 393 -> 375, 1 x 2^20 28.7 -> 26.8.
__device__ __forceinline__ rk_i64 walk_step(rk_i64 step) {
    asm("" : "+s"(step));
    return step;
}
__device__ __forceinline__ rk_u64 step_addr(rk_u64 p, rk_i64 step) {
    p += (rk_u64)step;
    asm("" : "+v"(p));
    return p;
}
__device__ __forceinline__ rk_u32 step_off(rk_u32 off, rk_u32 step) {
    off += step;
    asm("" : "+v"(off));
    return off;
}

// Loads the values x[i] at positions p0 + i*CS of the walk's instance (raw: no
// sign, no pre-op).  An invalid instance (past n_inst) was decomposed as
// instance 0, so its addresses are valid: it reads them and its results are
// never stored.  On a padded side a lane with nothing to load reads its
// instance's first position (a valid address, different per instance: one
// shared clamp address would be a hot spot for loads that bypass the caches),
// which the zeros behind the chirp table's end turn into zero; N > M/4 (M is
// the smallest length the planner takes), so positions of the first quarter
// need no bound (NQ values).
template <int V, int NV, int CS, int NQ, class IO>
__device__ __forceinline__ void load_run(const rk_pass_args& a, const IO& io, const Inst& ic, const Walk& w,
                                         typename IO::value_type* x) {
    using X = typename IO::value_type;
    constexpr bool PAD = pad_in<V>();
    const rk_u64 spare_m = PAD && ic.jpass >= a.n_valid_in ? 0 : ic.jpass;
    const rk_i64 spare = ic.in_base + (rk_i64)spare_m * a.in_sa;
    if constexpr (HasPtr<IO>::value) {
        rk_u64 p = reinterpret_cast<rk_u64>(table<X>(a.in) + w.a0);
        const rk_u64 sp = reinterpret_cast<rk_u64>(table<X>(a.in) + spare);
        const rk_i64 st = walk_step(CS * w.astep * (rk_i64)sizeof(scalar_t<X>));
        rk_u64 m = w.m0;
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            if (PAD && i >= NQ) x[i] = io.load_p(m < a.n_valid_in ? p : sp);
            else x[i] = io.load_p(p);
            if (i + 1 < NV) p = step_addr(p, st);
            m += (rk_u64)CS * w.mstep;
        }
    } else {
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const rk_u64 m = w.m0 + (rk_u64)(i * CS) * w.mstep;
            const rk_i64 addr = w.a0 + (rk_i64)(i * CS) * w.astep;
            const bool ok = ic.valid && (!PAD || m < a.n_valid_in);
            if constexpr (IO::kBranchFree && PAD)
                x[i] = io.load(a, ic.o, m < a.n_valid_in ? m : spare_m, ic.i, m < a.n_valid_in ? addr : spare);
            else if constexpr (IO::kBranchFree)
                x[i] = io.load(a, ic.o, m, ic.i, addr);
            else
                x[i] = ok ? io.load(a, ic.o, m, ic.i, addr) : cx<X>((real_t<X>)0, (real_t<X>)0);
        }
    }
}

// Input-side pre-processing of the values of load_run: conjugation for the
// inverse direction (first passes only, which have no inter-pass twiddle; the
// empty asm keeps the uniform branch a branch instead of selects per value),
// then the Bluestein chirp (compile-time).  The inter-pass twiddle
// (PRE_TWIDDLE) is applied by the caller's TwiddleWalk.
template <int V, int NV, int CS, class X>
__device__ __forceinline__ void pre_ops(const rk_pass_args& a, const Walk& w, X* x) {
    if constexpr (Variant<V>::PRE != RK_VAR_PRE_TWIDDLE) {
        if (a.in_sign < 0.0f) {
            asm volatile("");
#pragma unroll
            for (int i = 0; i < NV; ++i) x[i].y = -x[i].y;
        }
    }
    if constexpr (Variant<V>::PRE == RK_VAR_PRE_CHIRP) {
        rk_u64 p = reinterpret_cast<rk_u64>(table<X>(a.chirp) + w.m0);
        const rk_i64 st = walk_step(CS * (rk_i64)w.mstep * (rk_i64)sizeof(scalar_t<X>));
        const GlobalIO<false, false, scalar_t<X>> tab;
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            x[i] = c_mul(x[i], tab.load_p(p));
            if (i + 1 < NV) p = step_addr(p, st);
        }
    }
}

// The direction's conjugation and scale of an output value.
template <class X> __device__ __forceinline__ X adjust_out(const rk_pass_args& a, X y) {
    y.y *= (real_t<X>)a.out_sign;
    return c_scale(y, out_scale_of<X>(a));
}
template <int N, class X> __device__ __forceinline__ void adjust_all(const rk_pass_args& a, X* y, bool adjust) {
    if (adjust) {
        asm volatile("");   // a branch, not selects per value
#pragma unroll
        for (int i = 0; i < N; ++i) y[i] = adjust_out(a, y[i]);
    }
}

// Stores the values y[q*RS + r] at positions k0 + q*SQ + r*SR of the walk's
// instance (q < NQ, r < NR; the caller skips invalid instances): the
// compile-time post-op, the direction's adjustment, the store.  valid(q)
// excludes a thread's idle butterflies; a padded side skips positions at or
// beyond n_valid_out (those of its first quarter never are: NU values of r).
template <int V, int NQ, int SQ, int NR, int SR, int RS, int NU, class IO, class FV>
__device__ __forceinline__ void store_run(const rk_pass_args& a, const IO& io, const Inst& ic, const Walk& w,
                                          typename IO::value_type* y, bool adjust, FV valid) {
    using X = typename IO::value_type;
    constexpr int POST = Variant<V>::POST;
    if constexpr (POST != RK_VAR_POST_NONE) {
        const rk_i64 es = (rk_i64)sizeof(scalar_t<X>);
        const rk_i64 sr = walk_step(SR * (rk_i64)w.mstep * es), sq = walk_step(SQ * (rk_i64)w.mstep * es);
        rk_u64 pr = reinterpret_cast<rk_u64>(table<X>(POST == RK_VAR_POST_KMUL_CONJ ? a.bspec : a.chirp) + w.m0);
        const GlobalIO<false, false, scalar_t<X>> tab;
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            rk_u64 p = pr;
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                X& v = y[q * RS + r];
                if (valid(q)) {
                    if constexpr (POST == RK_VAR_POST_KMUL_CONJ) v = c_conj(c_mul(v, tab.load_p(p)));
                    else v = c_mul(c_conj(v), tab.load_p(p));
                }
                if (q + 1 < NQ) p = step_addr(p, sq);
            }
            if (r + 1 < NR) pr = step_addr(pr, sr);
        }
    }
    adjust_all<(NQ - 1) * RS + NR>(a, y, adjust);
    const rk_u64 k00 = w.m0;
    if constexpr (HasPtr<IO>::value) {
        const rk_i64 es = (rk_i64)sizeof(scalar_t<X>);
        const rk_i64 sr = walk_step(SR * w.astep * es), sq = walk_step(SQ * w.astep * es);
        rk_u64 pr = reinterpret_cast<rk_u64>(table<X>(a.out) + w.a0);
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            rk_u64 p = pr;
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                const bool ok = !pad_out<V>() || r < NU || k00 + (rk_u64)(q * SQ + r * SR) * w.mstep < a.n_valid_out;
                if (valid(q) && ok) io.store_p(p, y[q * RS + r]);
                if (q + 1 < NQ) p = step_addr(p, sq);
            }
            if (r + 1 < NR) pr = step_addr(pr, sr);
        }
    } else {
#pragma unroll
        for (int r = 0; r < NR; ++r) {
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                const int c = q * SQ + r * SR;
                const rk_u64 kabs = k00 + (rk_u64)c * w.mstep;
                const bool ok = !pad_out<V>() || kabs < a.n_valid_out;
                if (valid(q) && ok) io.store(a, ic.o, kabs, ic.i, w.a0 + (rk_i64)c * w.astep, y[q * RS + r]);
            }
        }
    }
}

// ------------------------------------------------------------------------
// LDS exchange between two register layouts
// ------------------------------------------------------------------------
// Every value a thread holds in `w` is written to LDS at wpos(i) (skipped
// when negative) and every value of `r` is read from rpos(i).  With SPLIT the
// real and imaginary parts travel separately through a buffer of floats, so
// the tile needs half the LDS (two work-groups then fit on a CU); `w` and `r`
// may be the same array.
// Ordering point of an exchange.  Work-group scope: a barrier with
// work-group fences (__syncthreads).  Wave scope (every position a lane
// writes or reads belongs to instances its own wave holds): no barrier; the
// wave-scope fences keep the compiler from moving LDS accesses across the
// point, and the wait for the wave's outstanding LDS operations
// (lgkmcnt(0): s_waitcnt encoding 0xc07f leaves vmcnt and expcnt at their
// maxima) completes its writes before its reads.
template <bool WAVE> __device__ __forceinline__ void exchange_sync() {
    if constexpr (WAVE) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_s_waitcnt(0xc07f);
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    } else {
        __syncthreads();
    }
}

// LEAD: LDS may still be read from an earlier exchange, so the writes wait for
// every thread (not needed by a tile's first exchange).
template <bool SPLIT, int NW, int NR, bool WAVE = false, bool LEAD = true, class X, class FW, class FR>
__device__ __forceinline__ void lds_exchange(void* base, const X* w, X* r, FW wpos, FR rpos) {
    using F = real_t<X>;
    if constexpr (!SPLIT) {
        X* lds = reinterpret_cast<X*>(base);
        if constexpr (LEAD) exchange_sync<WAVE>();
#pragma unroll
        for (int i = 0; i < NW; ++i) {
            const int p = wpos(i);
            if (p >= 0) lds[p] = w[i];
        }
        exchange_sync<WAVE>();
#pragma unroll
        for (int i = 0; i < NR; ++i) {
            const int p = rpos(i);
            if (p >= 0) r[i] = lds[p];
        }
    } else {
        F* f = reinterpret_cast<F*>(base);
        F wy[NW], rx[NR];
#pragma unroll
        for (int i = 0; i < NW; ++i) wy[i] = w[i].y;
        if constexpr (LEAD) exchange_sync<WAVE>();
#pragma unroll
        for (int i = 0; i < NW; ++i) {
            const int p = wpos(i);
            if (p >= 0) f[p] = w[i].x;
        }
        exchange_sync<WAVE>();
#pragma unroll
        for (int i = 0; i < NR; ++i) {
            const int p = rpos(i);
            rx[i] = p >= 0 ? f[p] : (F)0;
        }
        exchange_sync<WAVE>();
#pragma unroll
        for (int i = 0; i < NW; ++i) {
            const int p = wpos(i);
            if (p >= 0) f[p] = wy[i];
        }
        exchange_sync<WAVE>();
#pragma unroll
        for (int i = 0; i < NR; ++i) {
            const int p = rpos(i);
            if (p >= 0) r[i] = cx<X>(rx[i], f[p]);
        }
    }
}

// ------------------------------------------------------------------------
// the Stockham stages of one tile
// ------------------------------------------------------------------------
// Stage s holds, in thread t, the butterflies j = t + q*T (q < Q_s, j < NB_s);
// v[q*R + r] is input r of butterfly j, at position j + r*NB_s of the
// instance.  The butterfly's outputs go to (j/Ns)*Ns*R + j%Ns + r*Ns, which is
// where stage s+1 reads them; after the last stage v[q*R + r] holds output
// k = j + r*NB.
template <int L, int S>
RK_HD constexpr bool stage_valid(int t, int q) {
    using P = Plan<L>;
    return (P::nb(S) % P::T) == 0 || (t + q * P::T) < P::nb(S);
}

template <int L, int S>
RK_HD constexpr int stage_in_pos(int t, int i) {   // input position of v[i]
    using P = Plan<L>;
    constexpr int R = P::radix(S);
    const int q = i / R, r = i % R;
    return (t + q * P::T) + r * P::nb(S);
}

template <int L, int S>
RK_HD constexpr int stage_out_pos(int t, int i) {  // output position of v[i]
    using P = Plan<L>;
    constexpr int R = P::radix(S);
    constexpr int NS = P::ns(S);
    const int q = i / R, r = i % R;
    const int j = t + q * P::T;
    return (j / NS) * NS * R + (j % NS) + r * NS;
}

// The padded LDS positions of stage_in_pos / stage_out_pos (lds_pad of them),
// written as a per-thread part plus a per-value constant where lds_pad_add
// allows.  Input: t + (q*T + r*NB) with t < T.  Output: when T % NS == 0,
// j / NS = t / NS + q*T/NS and j % NS = t % NS, so the position is
// (t/NS)*NS*R + t%NS + (q*T*R + r*NS), whose per-thread part is below NS
// modulo 16 when NS < 16 and NS*R % 16 == 0; when the stage has no more
// butterflies than NS (j < NS) it is t + (q*T + r*NS).
template <int L, int S>
RK_HD constexpr int stage_in_lds(int t, int i) {
    using P = Plan<L>;
    constexpr int R = P::radix(S);
    constexpr int T = P::T;
    const int q = i / R, r = i % R;
    return lds_pad_add<(T < 16 ? T : 16)>(t, q * T + r * P::nb(S));
}

template <int L, int S>
RK_HD constexpr int stage_out_lds(int t, int i) {
    using P = Plan<L>;
    constexpr int R = P::radix(S);
    constexpr int NS = P::ns(S);
    constexpr int T = P::T;
    const int q = i / R, r = i % R;
    if constexpr (T % NS == 0) {
        constexpr int BM = (NS < 16 && (NS * R) % 16 == 0) ? NS : 16;
        return lds_pad_add<BM>((t / NS) * NS * R + t % NS, q * T * R + r * NS);
    } else if constexpr (P::nb(S) <= NS) {
        return lds_pad_add<(T < 16 ? T : 16)>(t, q * T + r * NS);
    } else {
        return lds_pad(stage_out_pos<L, S>(t, i));
    }
}

// Padded LDS position, within a tile of pitch LP, of element it of thread tid
// on an instance-linear (FLAT) side: e = tid + it*NT is instance e / L,
// position e % L.  When NT is a multiple of L every thread stays on one
// position of its instances; when L is a multiple of NT, iteration it covers
// positions (it*NT) % L + tid of instance (it*NT) / L.
template <int L, int NT, int LP>
RK_HD constexpr int flat_lds(int tid, int it) {
    if constexpr (NT % L == 0) {
        return (tid / L) * LP + lds_pad(tid % L) + it * (NT / L) * LP;
    } else if constexpr (L % NT == 0) {
        return ((it * NT) / L) * LP + lds_pad_add<(NT < 16 ? NT : 16)>(tid, (it * NT) % L);
    } else {
        const int e = tid + it * NT;
        const int ce = e / L;
        return ce * LP + lds_pad(e - ce * L);
    }
}

// The same for a pair tile, whose threads take two consecutive positions at a
// time: value 2*it + b is position e % L + b of pair e / L, e = 2*(tid + it*NT)
// (L even, so both positions are on one side of every padding slot).
template <int L, int NT, int LP>
RK_HD constexpr int flat_pair_lds(int tid, int it, int b) {
    if constexpr ((2 * NT) % L == 0) {
        return ((2 * tid) / L) * LP + lds_pad((2 * tid) % L) + it * ((2 * NT) / L) * LP + b;
    } else if constexpr (L % (2 * NT) == 0) {
        return ((it * 2 * NT) / L) * LP + lds_pad_add<(2 * NT < 16 ? 2 * NT : 16)>(2 * tid, (it * 2 * NT) % L) + b;
    } else {
        const int e = 2 * (tid + it * NT);
        const int ce = e / L;
        return ce * LP + lds_pad(e - ce * L) + b;
    }
}

// Padded LDS position of element it of a thread at position ps < T of an
// instance on a staged COLUMN / ROW side: ps + it*T.
template <int T> RK_HD constexpr int col_lds(int ps, int it) { return lds_pad_add<(T < 16 ? T : 16)>(ps, it * T); }

// LOWER: the upper half of the first stage's inputs is zero (lower_in).
// LEAD0: the first exchange is not the tile's first use of LDS.
template <int L, int S, bool SPLIT, int VM, bool WAVE = false, bool LOWER = false, bool LEAD0 = true, class X>
__device__ __forceinline__ void run_stages(X (&v)[VM], void* my, int t, const scalar_t<X>* twl) {
    using P = Plan<L>;
    constexpr int R = P::radix(S);
    constexpr int NS = P::ns(S);
    constexpr int Q = P::q(S);
    constexpr int T = P::T;
    if constexpr (S > 0) {
        // stage twiddles W_{NS*R}^{r*(j%NS)} from the FP64-rounded W_L table
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const int j = t + q * T;
            if (stage_valid<L, S>(t, q)) {
                const int m = j % NS;
                // byte offset of W_L^{r*m*L/(NS*R)}, one add per r
                const rk_u32 step = (rk_u32)m * (L / (NS * R)) * (rk_u32)sizeof(scalar_t<X>);
                rk_u32 off = 0;
#pragma unroll
                for (int r = 1; r < R; ++r) {
                    off = step_off(off, step);
                    v[q * R + r] = c_mul(v[q * R + r], *reinterpret_cast<const scalar_t<X>*>(
                                                           reinterpret_cast<const char*>(twl) + off));
                }
            }
        }
    }
#pragma unroll
    for (int q = 0; q < Q; ++q)
        if (stage_valid<L, S>(t, q)) {
            if constexpr (LOWER && S == 0) dft_lower<R>(&v[q * R]);
            else dft<R>(&v[q * R]);
        }
    if constexpr (S + 1 < P::NSTAGE) {
        constexpr int R1 = P::radix(S + 1);
        constexpr int Q1 = P::q(S + 1);
        lds_exchange<SPLIT, Q * R, Q1 * R1, WAVE, (LEAD0 || S > 0)>(
            my, v, v,
            [&](int i) { return stage_valid<L, S>(t, i / R) ? stage_out_lds<L, S>(t, i) : -1; },
            [&](int i) { return stage_valid<L, S + 1>(t, i / R1) ? stage_in_lds<L, S + 1>(t, i) : -1; });
        run_stages<L, S + 1, SPLIT, VM, WAVE>(v, my, t, twl);
    }
}

// ------------------------------------------------------------------------
// the pass kernel body
// ------------------------------------------------------------------------
// Tile of this work-group.  The dispatcher hands work-group b to XCD
// b % n_xcd; with groups of G > 1 the G tiles of each group of consecutive
// tiles go to work-groups on one XCD, so tiles that share cache lines (narrow
// column tiles) share that XCD's L2 instead of each fetching whole lines.
// Both counts are powers of two: scalar shifts, where four divisions cost
// about 80 vector instructions per wave.
__device__ __forceinline__ rk_u64 xcd_tile(const rk_pass_args& a) {
    const rk_u32 b = blockIdx.x;
    const rk_u32 g = a.xcd_group_lg, nx = a.n_xcd_lg;
    if (g == 0) return b;
    const rk_u32 full = (gridDim.x >> (g + nx)) << (g + nx);
    if (b >= full) return b;
    const rk_u32 x = b & ((1u << nx) - 1), k = b >> nx;
    return ((rk_u64)(k >> g) << (g + nx)) + (x << g) + (k & ((1u << g) - 1));
}

// LDS bytes of a tile and whether its exchanges are split into halves.
// HALF forces the split exchange on a tile that would fit whole (half the LDS,
// twice the resident work-groups).
template <int L, int C, bool HALF = false, int ES = 8> __host__ __device__ constexpr bool tile_split() {
    return HALF || lds_split(L, C, ES);
}
template <int L, int C, bool HALF = false, int ES = 8> __host__ __device__ constexpr int tile_pitch() {
    return lds_pitch_for(L, C, Plan<L>::T, HALF, ES);
}
template <int L, int C, bool HALF = false, int ES = 8> __host__ __device__ constexpr int tile_lds_bytes() {
    return C * tile_pitch<L, C, HALF, ES>() * (tile_split<L, C, HALF, ES>() ? ES / 2 : ES);
}

// The same of a pass's value type.  A pair tile of C instances has C/2 pairs
// and exchanges real parts, then imaginary parts, of both instances of a pair
// as 64-bit values: its LDS is that of a whole (unsplit) tile of C/2 instances.
template <int L, int C, bool HALF, class X> __host__ __device__ constexpr bool tile_split_x() {
    return pair_width<X>() == 2 || tile_split<L, C, HALF, (int)sizeof(scalar_t<X>)>();
}
template <int L, int C, bool HALF, class X> __host__ __device__ constexpr int tile_pitch_x() {
    if (pair_width<X>() == 2) return lds_pitch_pair(L, C, Plan<L>::T);
    return tile_pitch<L, C, HALF, (int)sizeof(scalar_t<X>)>();
}
template <int L, int C, bool HALF, class X> __host__ __device__ constexpr int tile_lds_bytes_x() {
    if (pair_width<X>() == 2) return pair_lds_bytes(L, C, Plan<L>::T);
    return tile_lds_bytes<L, C, HALF, (int)sizeof(scalar_t<X>)>();
}

// Instances left from inst0 on, cut to 32 bits (the tile compares them with
// its C).  The high word goes through an empty asm: of a 64-bit compare whose
// result both selects and branches, the compiler (ROCm 7.2) dropped the
// instruction that sets the select's condition, and ragged tiles of short rows
// were stored whole, past the end of the output.
__device__ __forceinline__ rk_u32 instances_left(const rk_pass_args& a, rk_u64 inst0) {
    const rk_u64 left = a.n_inst - inst0;
    rk_u32 hi = (rk_u32)(left >> 32);
    asm("" : "+s"(hi));
    return hi ? 0x7fffffffu : (rk_u32)left;
}

// Elements of a FLAT side of a tile with `left` instances left: C*L, fewer in
// the last tile.
template <int L, int C> __device__ __forceinline__ rk_u32 flat_elements(rk_u32 left) {
    return (left < (rk_u32)C ? left : (rk_u32)C) * (rk_u32)L;
}

// One tile (instances tile*C ... tile*C + C - 1) computed by threads
// tid = 0 ... C*T - 1 with `lds` of at least tile_lds_bytes<L, C, HALF, ES>()
// bytes (ES = sizeof the IO policy's element type).
// Every value a thread computes and every address it writes is a function of
// (a, tile, tid) alone, so a caller with more threads than C*T may give the
// surplus threads tid = C*T - 1: they repeat that thread's work, writing the
// same values to the same addresses, and take part in every barrier.
// With PRE, the tile's DIRECT loads were issued earlier (raw values in
// `pre`, see direct_raw_loads): the tile starts from them instead of loading.
template <int L, int C, int V, class IO, int MODES = 0, bool WAVE = false, bool PRE = false, bool HALF = false,
          bool TWLDS = false>
__device__ __forceinline__ void fft_pass_tile(const rk_pass_args& a, const IO& io, typename IO::value_type* lds,
                                              rk_u64 tile, int tid, const typename IO::value_type* pre = nullptr,
                                              scalar_t<typename IO::value_type>* twl_lds = nullptr) {
    using X = typename IO::value_type;
    using F = real_t<X>;
    constexpr int W = pair_width<X>();   // instances per thread
    constexpr int CT = C / W;
    static_assert(W == 1 || (C % 2 == 0 && MODES && (MODES & 3) == RK_MODE_DIRECT && !WAVE && !PRE && !HALF &&
                             !Variant<V>::BLUE && !pad_in<V>() && Variant<V>::POST == RK_VAR_POST_NONE && ((MODES >> 2) & 3) != RK_MODE_ROW),
                  "pairs of instances: column tiles with DIRECT loads and DIRECT or FLAT stores");
    using P = Plan<L>;
    static_assert(!WAVE || (64 % P::T == 0), "wave-local stages need whole instances per wave");
    constexpr int T = P::T;
    constexpr int NT = CT * T;
    constexpr int R0 = P::R0;
    constexpr int LP = tile_pitch_x<L, C, HALF, X>();
    constexpr int VM = P::vmax();
    constexpr int SL = P::NSTAGE - 1;
    constexpr int RL = P::radix(SL);
    constexpr int QL = P::q(SL);
    constexpr bool BLUE = Variant<V>::BLUE;
    constexpr bool TWID = Variant<V>::PRE == RK_VAR_PRE_TWIDDLE;
    constexpr bool SPLIT = tile_split_x<L, C, HALF, X>();
    constexpr bool LOW = lower_in<V>(R0);
    constexpr int NL = LOW ? R0 / 2 : R0;   // first-stage inputs of a thread that may be nonzero
    const rk_u64 inst0 = tile * (rk_u64)C;
    const rk_u32 load_mode = MODES ? (rk_u32)(MODES & 3) : a.load_mode;
    const rk_u32 store_mode = MODES ? (rk_u32)((MODES >> 2) & 3) : a.store_mode;

    // compute mapping (see fft_args.h): lanes along an instance or across
    // instances (WAVE: the row mapping, compiled in)
    const bool colmap = WAVE ? false : W == 2 ? true : a.cmap != 0;
    const int c = colmap ? (tid % CT) : (tid / T);
    int t = colmap ? (tid / CT) : (tid % T);
    const int cbase = c * LP;
    // the other mapping, for a side staged through LDS
    const int cs = colmap ? (tid / T) : (tid % CT);
    const int ps = colmap ? (tid % T) : (tid / CT);

    X v[VM];
    X g[R0];   // staging registers (global side of a staged load/store)

    // With TWLDS the tile copies the stage twiddles W_L^e into twl_lds.  Their
    // loads are issued before the tile's own and written to LDS once those are
    // on their way too (the first exchange's barrier publishes them), so the
    // tile waits for memory once, not twice; the scheduling barrier keeps the
    // first use of a loaded value behind the last load.  A tile that is one
    // round of latencies shows it most: with both, 4096 x 1000 16.9 -> 15.4
    // us, 2048 x 2048 16.9 -> 14.7, 16384 x 256 13.0 -> 11.9, 4096 x 997 35.2
    // -> 32.3, 8192 x 1024 29.7 -> 27.9.
    constexpr int NTW = TWLDS ? (L + NT - 1) / NT : 1;
    scalar_t<X> tw[NTW];
    if constexpr (TWLDS) {
        const scalar_t<X>* tab = table<X>(a.twl);
#pragma unroll
        for (int k = 0; k < NTW; ++k) tw[k] = tab[L % NT == 0 || tid + k * NT < L ? tid + k * NT : 0];
    }
    auto loads_issued = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (TWLDS) {
#pragma unroll
            for (int k = 0; k < NTW; ++k)
                if (L % NT == 0 || tid + k * NT < L) twl_lds[tid + k * NT] = tw[k];
        }
    };

    // ---- stage-0 inputs: element p = t + r*T of instance c ----
    const Inst ic = decompose<L>(a, inst0 + c * W);
    auto own_pos = [&](int i) { return cbase + stage_in_lds<L, 0>(t, i); };
    if (PRE || load_mode == RK_MODE_DIRECT) {
        const Walk w = in_walk(a, ic, t);
        if constexpr (PRE) {
#pragma unroll
            for (int r = 0; r < NL; ++r) v[r] = pre[r];
        } else {
            load_run<V, NL, T, R0 / 4>(a, io, ic, w, v);
        }
        loads_issued();
        pre_ops<V, NL, T>(a, w, v);
        if constexpr (TWID) apply_pass_twiddles<R0>(a, ic.l, t, T, v);
    } else if constexpr (W == 2) {
        // pairs load DIRECT
    } else if (load_mode == RK_MODE_FLAT) {
        // instance-linear block of C*L elements, no pre-ops
        const rk_i64 base = a.in_off + (rk_i64)inst0 * L;
        const rk_u32 left = instances_left(a, inst0), last = flat_elements<L, C>(left) - 1;
#pragma unroll
        for (int it = 0; it < R0; ++it) {
            // a lane past the last instance loads another element (the last, or
            // a transformation's first); its results are never stored.  The
            // bound on the element keeps the address a 32-bit offset from one
            // uniform base: with a select of the tile's first element all 16
            // held 64-bit addresses at once, the 48-point tile 145 VGPRs (now
            // 114) and three work-groups per CU instead of four: 87381 x 48
            // 15.1 -> 13.1 us, 37449 x 112 17.2 -> 15.1, 174762 x 24 12.7 ->
            // 11.6.
            const int e = tid + it * NT;
            const int ce = e / L, p = e - ce * L;
            const bool ok = (rk_u32)ce < left;
            if constexpr (HasPtr<IO>::value) {
                const rk_u32 n = (rk_u32)e < last ? (rk_u32)e : last;
                g[it] = io.load_p(reinterpret_cast<rk_u64>(table<X>(a.in) + base) + n * (rk_u32)sizeof(X));
            } else if constexpr (IO::kBranchFree) {
                g[it] = io.load(a, ok ? inst0 + ce : inst0, ok ? p : 0, 0, ok ? base + e : base);
            } else {
                g[it] = cx<X>((F)0, (F)0);
                if (ok) g[it] = io.load(a, inst0 + ce, p, 0, base + e);
            }
        }
        loads_issued();
        if (a.in_sign < 0.0f) {
            asm volatile("");
#pragma unroll
            for (int it = 0; it < R0; ++it) g[it].y = -g[it].y;
        }
        lds_exchange<SPLIT, R0, R0, false, PRE>(
            lds, g, v,
            [&](int it) { return flat_lds<L, NT, LP>(tid, it); }, own_pos);
    } else {
        // COLUMN (under the row mapping) or ROW (under the column mapping)
        const Inst ics = decompose<L>(a, inst0 + cs);
        const Walk w = in_walk(a, ics, ps);
        load_run<V, NL, T, R0 / 4>(a, io, ics, w, g);
        loads_issued();
        pre_ops<V, NL, T>(a, w, g);
        if constexpr (TWID) apply_pass_twiddles<R0>(a, ics.l, ps, T, g);
        lds_exchange<SPLIT, NL, NL, false, PRE>(
            lds, g, v, [&](int it) { return cs * LP + col_lds<T>(ps, it); }, own_pos);
    }

    // LDS of this thread's instance (the stages index it relative to the instance)
    void* my = SPLIT ? (void*)(reinterpret_cast<F*>(lds) + cbase) : (void*)(lds + cbase);
    auto last_out = [&](int i) {
        return stage_valid<L, SL>(t, i / RL) ? cbase + stage_out_lds<L, SL>(t, i) : -1;
    };
    const scalar_t<X>* twl;
    if constexpr (TWLDS) twl = twl_lds;
    else twl = table<X>(a.twl);
    constexpr bool LEAD0 = PRE || !(MODES && (MODES & 3) == RK_MODE_DIRECT);
    run_stages<L, 0, SPLIT, VM, WAVE, LOW, LEAD0>(v, my, t, twl);

    if constexpr (BLUE) {
        // A = FFT(chirp * x): multiply by the kernel spectrum, conjugate, and
        // transform again (the inverse DFT as conj(FFT(conj .))).
#pragma unroll
        for (int i = 0; i < QL * RL; ++i)
            if (stage_valid<L, SL>(t, i / RL)) {
                // position t + (q*T + r*NS): a constant offset from one address
                v[i] = c_conj(c_mul(v[i], (table<X>(a.bspec) + t)[stage_out_pos<L, SL>(0, i)]));
            }
        lds_exchange<SPLIT, QL * RL, R0, WAVE>(lds, v, v, last_out, own_pos);
        // the second transform and the stores recompute what depends on the
        // thread index: the index goes through an empty asm, so the first
        // transform's stage twiddles and the output chirp values are not held
        // in registers across both transforms (the 2048-point tile: 162 -> 124
        // VGPRs, four waves per SIMD instead of two)
        asm volatile("" : "+v"(t));
        if constexpr (TWLDS) run_stages<L, 0, SPLIT, VM, WAVE>(v, my, t, twl_lds);
        else run_stages<L, 0, SPLIT, VM, WAVE>(v, my, t, table<X>(a.twl));
    }

    // ---- store: output element k = stage_out_pos of the last stage ----
    const bool adjust = a.out_sign < 0.0f || a.out_scale != 1.0f;
    if (store_mode == RK_MODE_DIRECT) {
        // last stage: butterfly j = t + q*T < NS
        static_assert(P::nb(SL) == P::ns(SL), "the last Stockham stage writes its outputs at j + r * NS");
        if (ic.valid) {
            // last stage: output k = t + q*T + r*NS
            constexpr int NR = lower_out<V>(RL) ? RL / 2 : RL;
            store_run<V, QL, T, NR, P::ns(SL), RL, RL / 4>(a, io, ic, out_walk(a, ic, t), v, adjust,
                                                           [&](int q) { return stage_valid<L, SL>(t, q); });
        }
    } else if constexpr (W == 2 && ((MODES >> 2) & 3) == RK_MODE_DIRECT) {
        // stored above
    } else if constexpr (W == 2) {
        // FLAT: the tile is C*L contiguous elements; a thread takes two
        // consecutive positions of both instances of a pair (even R0 and L)
        static_assert(R0 % 2 == 0 && L % 2 == 0, "a pair tile stores two positions at a time");
        const rk_i64 base = a.out_off + (rk_i64)inst0 * L;
        const rk_u32 left = instances_left(a, inst0);
        lds_exchange<SPLIT, QL * RL, R0>(lds, v, g, last_out,
                                         [&](int i) { return flat_pair_lds<L, NT, LP>(tid, i / 2, i % 2); });
        adjust_all<R0>(a, g, adjust);
        auto store_all = [&](auto keep) {
#pragma unroll
            for (int it = 0; it < R0 / 2; ++it) {
                const int e = 2 * (tid + it * NT);
                const int ce = e / L, k = e - ce * L;
                if (keep(2 * ce)) {
                    const X y0 = g[2 * it], y1 = g[2 * it + 1];
                    const rk_u64 at = reinterpret_cast<rk_u64>(a.out + base) + (rk_u32)(2 * ce * L + k) * 8u;
                    io.store_run(at, y0.x.x, y0.y.x, y1.x.x, y1.y.x);
                    io.store_run(at + L * 8, y0.x.y, y0.y.y, y1.x.y, y1.y.y);
                }
            }
        };
        if (left >= (rk_u32)C) store_all([](int) { return true; });
        else store_all([&](int ce) { return (rk_u32)ce < left; });
    } else if (store_mode == RK_MODE_FLAT) {
        // no post-ops beyond sign and scale
        lds_exchange<SPLIT, QL * RL, R0>(lds, v, g, last_out, [&](int it) { return flat_lds<L, NT, LP>(tid, it); });
        adjust_all<R0>(a, g, adjust);
        const rk_i64 base = a.out_off + (rk_i64)inst0 * L;
        const rk_u32 left = instances_left(a, inst0), end = flat_elements<L, C>(left);
        auto store_all = [&](auto keep) {
#pragma unroll
            for (int it = 0; it < R0; ++it) {
                const int e = tid + it * NT;
                const int ce = e / L, k = e - ce * L;
                if (keep(e, ce)) {
                    if constexpr (HasPtr<IO>::value)
                        io.store_p(reinterpret_cast<rk_u64>(table<X>(a.out) + base) + (rk_u32)e * (rk_u32)sizeof(X),
                                   g[it]);
                    else
                        io.store(a, inst0 + ce, k, 0, base + e, g[it]);
                }
            }
        };
        // one uniform branch, not one per value
        if (left >= (rk_u32)C) store_all([](int, int) { return true; });
        else store_all([&](int e, int ce) { return HasPtr<IO>::value ? (rk_u32)e < end : (rk_u32)ce < left; });
    } else {
        constexpr int NO = lower_out<V>(R0) ? R0 / 2 : R0;
        lds_exchange<SPLIT, QL * RL, NO>(lds, v, g, last_out, [&](int it) { return cs * LP + col_lds<T>(ps, it); });
        const Inst ics = decompose<L>(a, inst0 + cs);
        if (ics.valid) {
            store_run<V, 1, 0, NO, T, R0, R0 / 4>(a, io, ics, out_walk(a, ics, ps), g, adjust, [](int) { return true; });
        }
    }
}

// Threads per work-group of fft_pass_body<L, C, ...>.
template <int L, int C> __host__ __device__ constexpr int pass_threads() { return C * Plan<L>::T; }
// The same of a catalogue variant number (RK_VAR_PAIR: two instances per thread).
template <int L, int C, int V> __host__ __device__ constexpr int variant_threads() {
    return (V & RK_VAR_PAIR) ? (C / 2) * Plan<L>::T : C * Plan<L>::T;
}
// The work-group size of a kernel's launch bounds: its threads, rounded up to
// whole waves on all four SIMDs above 256.  The compiler raises a kernel's
// registers to what the waves that the LDS admits leave free, counting waves
// over the CU; a work-group of 13 waves, though, needs room for four on one
// SIMD, and a second one then found none (1000-point column tiles of 800
// threads: 72 registers and one work-group per CU, 149 us for 32 x 1000 x
// 1008; with 1024 in the bounds 56 registers and two, 130 us).
RK_HD constexpr int bound_threads(int threads) { return threads > 256 ? (threads + 255) / 256 * 256 : threads; }

// Tiles whose stage twiddles are read from an LDS copy of the W_L table
// instead of global memory (the table loads otherwise take a large share of
// the vector-memory instructions): complex64 tiles with at least one stage
// after the first and exchanges with work-group barriers (no wave-local
// stages), where the extra L entries leave the
// tile's LDS-limited residency per CU unchanged, or cost at most 16 KB and
// leave two work-groups per CU.  Measured on row tiles, whose residency the
// table does lower: 4096 x 1000 20.0 -> 17.6 us, 16384 x 2048 117 -> 102 us,
// 16384 x 1024 50.5 -> 47.7 us, the single-kernel Bluestein 4096 x 997 (both
// of its transforms read the table) 53 -> 44 us; 4096-point rows (a 32 KB
// table, half the residency) 64 -> 70 us, so they keep the global table.
template <int L, int C, int V, bool WAVE, bool HALF, class X> __host__ __device__ constexpr bool twl_in_lds() {
    constexpr int ES = (int)sizeof(scalar_t<X>);
    if (WAVE || ES != 8 || Plan<L>::NSTAGE < 2) return false;
    constexpr int base = tile_lds_bytes_x<L, C, HALF, X>();
    constexpr int with = base + L * ES;
    return (160 * 1024) / with == (160 * 1024) / base || (L * ES <= 16 * 1024 && (160 * 1024) / with >= 2);
}

// One work-group of a pass launch: the tile this work-group owns, with the
// work-group's own LDS.
template <int L, int C, int V, class IO, int MODES = 0, bool WAVE = false, bool HALF = false>
__device__ __forceinline__ void fft_pass_body(const rk_pass_args& a, const IO& io) {
    using X = typename IO::value_type;
    constexpr int LP = tile_pitch_x<L, C, HALF, X>();
    constexpr int CT = C / pair_width<X>();
    __shared__ X lds[tile_split_x<L, C, HALF, X>() ? (CT * LP + 1) / 2 : CT * LP];
    const rk_u64 tile = xcd_tile(a) + a.tile_base;
    if (tile >= a.n_tiles) return;
    if constexpr (twl_in_lds<L, C, V, WAVE, HALF, X>()) {
        __shared__ scalar_t<X> twl_s[L];
        fft_pass_tile<L, C, V, IO, MODES, WAVE, false, HALF, true>(a, io, lds, tile, (int)threadIdx.x, nullptr, twl_s);
    } else {
        fft_pass_tile<L, C, V, IO, MODES, WAVE, false, HALF>(a, io, lds, tile, (int)threadIdx.x);
    }
}

// The raw DIRECT loads of one tile (what fft_pass_tile<..., PRE> starts from).
template <int L, int C, int V, class IO, bool WAVE>
__device__ __forceinline__ void direct_raw_loads(const rk_pass_args& a, const IO& io, rk_u64 tile, int tid,
                                                 typename IO::value_type* raw) {
    using P = Plan<L>;
    constexpr int T = P::T;
    const bool colmap = WAVE ? false : a.cmap != 0;
    const int c = colmap ? (tid % C) : (tid / T);
    const int t = colmap ? (tid / C) : (tid % T);
    const Inst ic = decompose<L>(a, tile * (rk_u64)C + c);
    const Walk w = in_walk(a, ic, t);
    load_run<V, (lower_in<V>(P::R0) ? P::R0 / 2 : P::R0), T, P::R0 / 4>(a, io, ic, w, raw);
}

// Persistent, software-pipelined pass (DIRECT loads only): work-group b runs
// the tiles tile_base + b, + G, + 2G, ... below n_tiles (G = gridDim.x) and
// issues the global loads of its next tile before it computes and stores the
// current one, so one tile's loads are in flight while another is computed.
// The host launches about one work-group per resident slot.
template <int L, int C, int V, class IO, int MODES, bool WAVE, bool HALF>
__device__ __forceinline__ void fft_pass_body_pipe(const rk_pass_args& a, const IO& io) {
    using X = typename IO::value_type;
    constexpr int ES = (int)sizeof(X);
    constexpr int LP = tile_pitch<L, C, HALF, ES>();
    constexpr int R0 = Plan<L>::R0;
    __shared__ X lds[tile_split<L, C, HALF, ES>() ? (C * LP + 1) / 2 : C * LP];
    const int tid0 = (int)threadIdx.x;
    const rk_u64 G = gridDim.x;
    rk_u64 tile = a.tile_base + blockIdx.x;
    if (tile >= a.n_tiles) return;
    X nxt[R0];
    direct_raw_loads<L, C, V, IO, WAVE>(a, io, tile, tid0, nxt);
    for (;;) {
        // everything derived from the thread index (stage twiddle indices and
        // loads, LDS positions) is recomputed per tile instead of being
        // hoisted out of the loop and held in registers across tiles: the
        // empty asm makes the index opaque to the optimiser each iteration
        int tid = tid0;
        asm volatile("" : "+v"(tid));
        X cur[R0];
#pragma unroll
        for (int r = 0; r < R0; ++r) cur[r] = nxt[r];
        const rk_u64 next = tile + G;
        if (next < a.n_tiles) direct_raw_loads<L, C, V, IO, WAVE>(a, io, next, tid, nxt);
        fft_pass_tile<L, C, V, IO, MODES, WAVE, true, HALF>(a, io, lds, tile, tid, cur);
        if (next >= a.n_tiles) break;
        tile = next;
    }
}

// The value type of a variant number: complex128 with RK_VAR_F64, two
// instances' complex64 values with RK_VAR_PAIR.
template <bool F64> struct ElemOf { typedef float2 type; };
template <> struct ElemOf<true> { typedef double2 type; };
template <bool PAIR, bool F64> struct ValueOf { typedef typename ElemOf<F64>::type type; };
template <bool F64> struct ValueOf<true, F64> { typedef cpair2 type; };
template <int V> using elem_t = typename ValueOf<(V & RK_VAR_PAIR) != 0, (V & RK_VAR_F64) != 0>::type;

// The pass kernel of a catalogue variant number V: the low seven bits are the
// compile-time Variant (pre-op, post-op, Bluestein), the higher bits choose the
// IO policy (RK_VAR_STREAM, RK_VAR_NT_LOAD, RK_VAR_NT_STORE), compiled-in
// load/store modes (RK_VAR_MODE_*), wave-local stages (RK_VAR_WAVE) and the
// element type (RK_VAR_F64).  The ahead-of-time catalogue and the run-time
// compiler instantiate this same entry.
template <int L, int C, int V>
__device__ __forceinline__ void fft_pass_entry(const rk_pass_args& a) {
    using X = elem_t<V>;
    constexpr int VB = V & (RK_VAR_STREAM - 1);
    constexpr int M = (V & RK_VAR_MODE_DD) ? RK_MODES(RK_MODE_DIRECT, RK_MODE_DIRECT)
                    : (V & RK_VAR_MODE_DF) ? RK_MODES(RK_MODE_DIRECT, RK_MODE_FLAT)
                    : (V & RK_VAR_MODE_FF) ? RK_MODES(RK_MODE_FLAT, RK_MODE_FLAT) : 0;
    constexpr bool NTL = (V & (RK_VAR_STREAM | RK_VAR_NT_LOAD)) != 0;
    constexpr bool NTS = (V & (RK_VAR_STREAM | RK_VAR_NT_STORE)) != 0;
    constexpr bool WAVE = (V & RK_VAR_WAVE) != 0;
    constexpr bool HALF = (V & RK_VAR_HALF) != 0;
    if constexpr ((V & RK_VAR_PAIR) != 0)
        fft_pass_body<L, C, VB, PairIO<NTL, NTS>, M>(a, PairIO<NTL, NTS>{});
    else if constexpr ((V & RK_VAR_PIPE) != 0)
        fft_pass_body_pipe<L, C, VB, GlobalIO<NTL, NTS, X>, M, WAVE, HALF>(a, GlobalIO<NTL, NTS, X>{});
    else
        fft_pass_body<L, C, VB, GlobalIO<NTL, NTS, X>, M, WAVE, HALF>(a, GlobalIO<NTL, NTS, X>{});
}

// Minimum waves per SIMD of a pass kernel's launch bounds: three for the
// single-kernel Bluestein tiles with DIRECT/DIRECT compiled in of at most 256
// threads (at most 168 VGPRs), else one (the tile's own thread count bounds
// its registers).
// An RK_VAR_OCC kernel asks for the waves per SIMD its LDS allows, so
// registers do not cut the occupancy; a persistent (RK_VAR_PIPE) kernel
// without it for one resident work-group per CU (the registers of its
// prefetched tile then come out of that work-group's share).  A pair kernel
// asks for the work-groups that its LDS and 56 registers beside the two
// instances' values allow (two of the 600-, 1000- and 1024-point tiles; with
// 32 beside them values spill: 64 x 1008000 804 us with the spills, 482
// without).
template <int L, int C, int V> __host__ __device__ constexpr int pass_min_waves() {
    if constexpr ((V & RK_VAR_PAIR) != 0) {
        const int waves = (variant_threads<L, C, V>() + 255) / 256;   // of a work-group, per SIMD
        constexpr int tile = tile_lds_bytes_x<L, C, false, cpair2>();
        constexpr int lds = tile + (twl_in_lds<L, C, V, false, false, cpair2>() ? L * 8 : 0);
        const int by_regs = 512 / (4 * Plan<L>::vmax() + 56) / waves, by_lds = (160 * 1024) / lds;
        const int wgs = by_regs < 1 ? 1 : (by_regs < by_lds ? by_regs : by_lds);
        return wgs * waves;
    }
    if ((V & (RK_VAR_PIPE | RK_VAR_OCC)) != 0) {
        const int waves = (pass_threads<L, C>() + 63) / 64;
        const int slots = (V & RK_VAR_OCC) ? (160 * 1024) / tile_lds_bytes<L, C, (V & RK_VAR_HALF) != 0,
                                                                           (int)sizeof(elem_t<V>)>() : 1;
        const int w = (slots * waves) / 4;
        return w < 1 ? 1 : (w > 8 ? 8 : w);
    }
    return ((V & RK_VAR_MODE_DD) && (V & 16) && pass_threads<L, C>() <= 256) ? 3 : 1;
}

}   // namespace rkfft

#endif
