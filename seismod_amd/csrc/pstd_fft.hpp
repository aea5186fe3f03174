// pstd_fft.hpp -- staggered spectral derivatives by hand-written transforms.
//
// A derivative along an axis of n points is f -> IDFT(H DFT(f)), H(k) the
// whole-spectrum multiplier.  Two real lines (rows along z, columns along x)
// go through one complex transform z = a + i b.  A workgroup keeps P such
// pairs in LDS.
//
// The forward transform runs decimation in frequency: pass q of radix R
// combines the R elements S = m / (R_0 .. R_q) apart inside each block and
// multiplies output t by e^{-2 pi i j t / (S R)}, j the position in the
// block.  Every thread writes what it read, in place, so a pass needs one
// barrier and one LDS buffer, and the spectrum ends in digit-reversed order,
// in which the multiplier is tabulated.  The inverse runs the transposed
// passes (twiddle, then the same radix) on the conjugate, from digit-reversed
// back to natural order.  The first pass reads the field from global memory,
// the last writes the derivative there, and the pass in the middle transforms,
// multiplies and transforms back R contiguous elements in registers: three
// radices cross LDS four times each way and meet five barriers.
//
// What bounds it: the chain of a workgroup's phases (load, five barriers,
// store) in few waves.  Counters, 4 derivatives of 1040^2 FP32: 3 waves a
// SIMD, all of them resident at once and waiting for 53% of their time; the
// vector units busy 48% of the launch (1660 instructions a wave), LDS 16%; 12
// derivatives 46% and 17%, in FP64 20% and 14%.  A launch of 4 derivatives of
// 1040^2 FP32 takes 19.2 us (1.8 TB/s), of 12 derivatives 49 us; the
// out-of-place Stockham passes before, with runtime loops, root tables in LDS
// and two buffers, 37.7 and 91.1 us.  Two passes with radices up to 40 measured
// 29.5 and 54.4 us (195 registers, too few waves), one round per pass instead
// of a loop over items frees the scalar registers of the roots (54.6 -> 49 us).
#pragma once

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <vector>

#include "sm_internal.hpp"

namespace sm {
namespace pstd {

template <typename T>
struct Cx {
    T re, im;
};

// a b + c with one rounding
__device__ __forceinline__ float mad(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double mad(double a, double b, double c) { return __builtin_fma(a, b, c); }

template <typename T>
__device__ __forceinline__ Cx<T> cmul(Cx<T> a, Cx<T> b)
{
    // fused multiply-adds: one rounding less per product (the transforms
    // are held to a tolerance, not to the reference's FFTW bits)
    return {mad(a.re, b.re, -(a.im * b.im)), mad(a.re, b.im, a.im * b.re)};
}
template <typename T>
__device__ __forceinline__ Cx<T> cadd(Cx<T> a, Cx<T> b) { return {a.re + b.re, a.im + b.im}; }
template <typename T>
__device__ __forceinline__ Cx<T> csub(Cx<T> a, Cx<T> b) { return {a.re - b.re, a.im - b.im}; }
// -i a
template <typename T>
__device__ __forceinline__ Cx<T> cmi(Cx<T> a) { return {a.im, -a.re}; }

// cos and sin of 2 pi k / R, k <= R / 2
constexpr double COS3[] = {1.0, -0.5};
constexpr double SIN3[] = {0.0, 0.8660254037844386};
constexpr double COS5[] = {1.0, 0.30901699437494745, -0.8090169943749475};
constexpr double SIN5[] = {0.0, 0.9510565162951535, 0.5877852522924731};
constexpr double COS7[] = {1.0, 0.6234898018587335, -0.2225209339563144, -0.9009688679024191};
constexpr double SIN7[] = {0.0, 0.7818314824680298, 0.9749279121818236, 0.4338837391175581};
constexpr double COS9[] = {1.0, 0.766044443118978, 0.17364817766693036, -0.5, -0.9396926207859084};
constexpr double SIN9[] = {0.0, 0.6427876096865394, 0.984807753012208, 0.8660254037844386, 0.3420201433256687};
constexpr double COS11[] = {1.0, 0.8412535328311812, 0.41541501300188644, -0.14231483827328514, -0.6548607339452851,
    -0.9594929736144974};
constexpr double SIN11[] = {0.0, 0.5406408174555976, 0.9096319953545183, 0.9898214418809327, 0.7557495743542583,
    0.28173255684142967};
constexpr double COS13[] = {1.0, 0.8854560256532099, 0.5680647467311558, 0.12053668025532305, -0.3546048870425356,
    -0.7485107481711011, -0.970941817426052};
constexpr double SIN13[] = {0.0, 0.46472317204376856, 0.8229838658936564, 0.992708874098054, 0.9350162426854148,
    0.6631226582407952, 0.23931566428755777};
constexpr double COS16[] = {1.0, 0.9238795325112867, 0.7071067811865476, 0.3826834323650898, 0.0,
    -0.3826834323650898, -0.7071067811865476, -0.9238795325112867, -1.0};
constexpr double SIN16[] = {0.0, 0.3826834323650898, 0.7071067811865476, 0.9238795325112867, 1.0,
    0.9238795325112867, 0.7071067811865476, 0.3826834323650898, 0.0};
constexpr double root_cos(int R, int k)
{
    k %= R;
    if (2 * k > R) k = R - k;
    switch (R) {
    case 3: return COS3[k];
    case 5: return COS5[k];
    case 7: return COS7[k];
    case 9: return COS9[k];
    case 11: return COS11[k];
    case 13: return COS13[k];
    default: return COS16[k * (16 / R)];
    }
}
constexpr double root_sin(int R, int k)
{
    k %= R;
    const bool neg = 2 * k > R;
    if (neg) k = R - k;
    double v = 0;
    switch (R) {
    case 3: v = SIN3[k]; break;
    case 5: v = SIN5[k]; break;
    case 7: v = SIN7[k]; break;
    case 9: v = SIN9[k]; break;
    case 11: v = SIN11[k]; break;
    case 13: v = SIN13[k]; break;
    default: v = SIN16[k * (16 / R)]; break;
    }
    return neg ? -v : v;
}

// R = A B with coprime A, B (no twiddles between them), 0 if R has none
constexpr int coprime_factor(int R)
{
    int best = 0;
    for (int A = 2; A * A < R; ++A) {
        if (R % A) continue;
        int x = A, y = R / A;
        while (y) { const int t = x % y; x = y; y = t; }
        if (x == 1) best = A;
    }
    return best;
}
constexpr int inverse_mod(int a, int m)
{
    for (int x = 1; x < m; ++x)
        if (a * x % m == 1) return x;
    return 0;
}

// forward DFT of v[0..R) in natural order, in place.  The roots are
// compile-time constants (scalar registers).
template <typename T, int R>
__device__ __forceinline__ void dft(Cx<T> *v)
{
    if constexpr (R == 2) {
        const Cx<T> a = v[0], b = v[1];
        v[0] = cadd(a, b); v[1] = csub(a, b);
    } else if constexpr (R == 4) {
        const Cx<T> a0 = cadd(v[0], v[2]), a1 = csub(v[0], v[2]), a2 = cadd(v[1], v[3]), a3 = csub(v[1], v[3]);
        v[0] = cadd(a0, a2); v[2] = csub(a0, a2);
        v[1] = cadd(a1, cmi(a3)); v[3] = csub(a1, cmi(a3));
    } else if constexpr (coprime_factor(R) != 0) {
        // prime-factor mapping: n = B n1 + A n2, k = k1 B (1/B mod A) + k2 A (1/A mod B)
        constexpr int A = coprime_factor(R), B = R / A;
        constexpr int kB = B * inverse_mod(B % A, A), kA = A * inverse_mod(A % B, B);
        Cx<T> u[B][A];
#pragma unroll
        for (int n2 = 0; n2 < B; ++n2) {
#pragma unroll
            for (int n1 = 0; n1 < A; ++n1) u[n2][n1] = v[(B * n1 + A * n2) % R];
            dft<T, A>(u[n2]);
        }
#pragma unroll
        for (int k1 = 0; k1 < A; ++k1) {
            Cx<T> w[B];
#pragma unroll
            for (int n2 = 0; n2 < B; ++n2) w[n2] = u[n2][k1];
            dft<T, B>(w);
#pragma unroll
            for (int k2 = 0; k2 < B; ++k2) v[(k1 * kB + k2 * kA) % R] = w[k2];
        }
    } else if constexpr (R == 8 || R == 9 || R == 16) {
        // n = B a + i, k = k1 + A l with constant twiddles between the factors
        constexpr int A = R == 9 ? 3 : R == 8 ? 2 : 4, B = R / A;
        Cx<T> u[B][A];
#pragma unroll
        for (int i = 0; i < B; ++i) {
#pragma unroll
            for (int n1 = 0; n1 < A; ++n1) u[i][n1] = v[B * n1 + i];
            dft<T, A>(u[i]);
        }
#pragma unroll
        for (int k1 = 0; k1 < A; ++k1) {
            Cx<T> w[B];
#pragma unroll
            for (int i = 0; i < B; ++i) {
                const Cx<T> y = u[i][k1];
                const int e = i * k1;
                const T c = (T)root_cos(R, e), s = (T)root_sin(R, e);
                if (e == 0) w[i] = y;
                else if (R % 2 == 0 && 4 * e == R) w[i] = cmi(y);
                else if (R % 2 == 0 && 8 * e == R) w[i] = {(y.re + y.im) * c, (y.im - y.re) * c};
                else if (R % 2 == 0 && 8 * e == 3 * R) w[i] = {(y.im - y.re) * s, -((y.re + y.im) * s)};
                else w[i] = {mad(y.re, c, y.im * s), mad(y.im, c, -(y.re * s))};
            }
            dft<T, B>(w);
#pragma unroll
            for (int l = 0; l < B; ++l) v[k1 + A * l] = w[l];
        }
    } else {
        // odd prime R: pair t with R - t; X_s = A_s - i B_s, X_{R-s} = A_s + i B_s
        // with A_s = v0 + sum (v_t + v_{R-t}) cos, B_s = sum (v_t - v_{R-t}) sin
        constexpr int H = (R - 1) / 2;
        Cx<T> sp[H], sm[H];
        const Cx<T> v0 = v[0];
        Cx<T> x0 = v0;
#pragma unroll
        for (int t = 1; t <= H; ++t) {
            sp[t - 1] = cadd(v[t], v[R - t]);
            sm[t - 1] = csub(v[t], v[R - t]);
            x0 = cadd(x0, sp[t - 1]);
        }
        v[0] = x0;
#pragma unroll
        for (int s = 1; s <= H; ++s) {
            Cx<T> A = v0, B = {T(0), T(0)};
#pragma unroll
            for (int t = 1; t <= H; ++t) {
                const T c = (T)root_cos(R, s * t), d = (T)root_sin(R, s * t);
                A.re = mad(sp[t - 1].re, c, A.re); A.im = mad(sp[t - 1].im, c, A.im);
                B.re = t == 1 ? sm[0].re * d : mad(sm[t - 1].re, d, B.re);
                B.im = t == 1 ? sm[0].im * d : mad(sm[t - 1].im, d, B.im);
            }
            v[s] = {A.re + B.im, A.im - B.re};
            v[R - s] = {A.re - B.im, A.im + B.re};
        }
    }
}

// ------------------------------------------------------------------
// transform plans
// ------------------------------------------------------------------
constexpr int FFT_MAXPASS = 6;
constexpr int FFT_MAXRADIX = 16;

// vector operations per element of a radix; 0 if it is not built
constexpr double fft_cost(int R)
{
    switch (R) {
    case 2: return 2;
    case 3: return 5.3;
    case 4: return 4;
    case 5: return 7.2;
    case 7: return 9.4;
    case 8: return 6.5;
    case 9: return 13.3;
    case 11: return 13.6;
    case 13: return 15.7;
    case 16: return 10.5;
    default: break;
    }
    const int A = R <= FFT_MAXRADIX ? coprime_factor(R) : 0;
    if (A == 0) return 0;
    const double a = fft_cost(A), b = fft_cost(R / A);
    return a > 0 && b > 0 ? a + b : 0;
}
// cost per element of a pass itself (LDS both ways, twiddle, addresses)
constexpr double FFT_PASS = 10.0;

struct FftPlan {
    int n = 0, m = 0;               // axis length, transform length
    int nr = 0, R[FFT_MAXPASS] = {};
    int S[FFT_MAXPASS] = {};        // distance of a butterfly's elements
    int toff[FFT_MAXPASS] = {}, tsz = 0;   // twiddles of pass q at toff[q], (t - 1) S + j
    double cost = 0;                // per element
    bool loop = false;              // a pass takes its butterflies in several rounds
};

constexpr int FFT_THREADS = 512;    // largest workgroup: 256 registers a thread

// the cheapest radices of m, none below `least`; false when m has a factor
// above 13, no such radices, or needs fewer than two or more than
// FFT_MAXPASS passes
inline bool fft_radices(int m, int least, FftPlan &p)
{
    p.nr = 0;
    p.cost = 1e30;
    int cur[FFT_MAXPASS];
    auto go = [&](auto &&self, int left, int most, int k, double c) -> void {
        if (left == 1) {
            if (k >= 2 && c < p.cost) {
                p.cost = c;
                p.nr = k;
                for (int q = 0; q < k; ++q) p.R[q] = cur[q];
            }
            return;
        }
        if (k == FFT_MAXPASS) return;
        for (int r = std::min(most, left); r >= least; --r)
            if (left % r == 0) {
                cur[k] = r;
                self(self, left / r, r, k + 1, c + fft_cost(r) + FFT_PASS);
            }
    };
    go(go, m, FFT_MAXRADIX, 0, 0.0);
    if (p.nr == 0) return false;
    // an odd radix last: the middle pass reads R contiguous elements per
    // thread, and an odd stride between lanes spreads them over the banks
    // without padding.  The rest in falling order, so that the later
    // passes' blocks are long runs.
    std::sort(p.R, p.R + p.nr, [](int a, int b) { return (a % 2) != (b % 2) ? a % 2 == 0 : a % 2 ? a < b : a > b; });
    return true;
}

inline void fft_layout(FftPlan &p)
{
    int B = p.m;
    p.tsz = 0;
    for (int q = 0; q < p.nr; ++q) {
        p.S[q] = B / p.R[q];
        p.toff[q] = p.tsz;
        if (p.S[q] > 1) p.tsz += (p.R[q] - 1) * p.S[q];
        B = p.S[q];
    }
}

// threads of a workgroup: every pass takes its butterflies in one round
// unless the plan loops
inline int fft_threads(const FftPlan &p, int P)
{
    int most = 0;
    for (int q = 0; q < p.nr; ++q) most = std::max(most, P * (p.m / p.R[q]));
    if (p.loop) most = std::min(most, FFT_THREADS);
    return (most + 63) / 64 * 64;
}

// plan of the derivative of n points in values of elt bytes; false when no
// hand-written transform takes this length.
//
// First choice are the cheapest radices with which FFT_THREADS threads take
// every pass in one round: of 2000 points, none below 4.  (Lines above
// FFT_FEWER bytes only if no radices are cheaper: with dearer ones hipFFT's
// long rows are faster along z, FP64 256 x 2376 322 and 414 us a step, but
// 256 x 2592 402 and 375, 256 x 3430 497 and 412.)  A line of at most
// FFT_LOOP bytes that has none takes the cheapest of all and loops (1617 to
// 3402 points in FP32, 1617 in FP64).  A step of the SH solver, FP32, this
// loop against hipFFT: 256 x 3000 177 and 301 us, 3000 x 256 183 and 425,
// 256 x 2662 184 and 297, 3000^2 1531 and 3556.  Longer lines stay with
// hipFFT: 256 x 4000 343 us, 391 in one round of 1024 threads.
//
// The derivative is a circular convolution with a real kernel of n points, so
// a length with other factors runs as a linear one:
// lines padded with zeros to any m >= 2 n - 1 that the radices make, and the
// kernel's spectrum over m points as the multiplier: twice the work of a
// length that the radices make (1039^2 against 1040^2, 8 FP32 derivatives:
// 77.6 and 36.2 us), a quarter of hipFFT's chirp transforms and their copy
// passes (469 x 363, FP64, a P-SV stage: 45 against 230 us).  One round of
// FFT_THREADS threads takes m up to 4096, n up to 2048.
constexpr size_t FFT_LOOP = 28 * 1024, FFT_FEWER = 40 * 1024;
inline bool fft_plan(int n, size_t elt, FftPlan &p)
{
    auto one_round = [](int m) { return std::max(2, (m + FFT_THREADS - 1) / FFT_THREADS); };
    p = FftPlan();
    if (n < 2) return false;
    p.m = n;
    const size_t bytes = 2 * (size_t)n * elt;
    bool ok = bytes <= FFT_FEWER ? fft_radices(n, one_round(n), p)
                                 : fft_radices(n, 2, p) && fft_threads(p, 1) <= FFT_THREADS;
    if (!ok && bytes <= FFT_LOOP) ok = p.loop = fft_radices(n, 2, p);
    if (!ok) {
        double cost = 1e30;
        for (int m = 2 * n - 1; m <= 2 * n + n / 4 + 16; ++m) {
            FftPlan f;
            if (!fft_radices(m, one_round(m), f) || f.cost * m >= cost) continue;
            ok = true;
            cost = f.cost * m;
            p = f;
            p.m = m;
        }
    }
    p.n = n;
    if (ok) fft_layout(p);
    return ok;
}
// rounds of the longest pass of one group of lines
inline int fft_rounds(const FftPlan &p)
{
    int most = 0;
    for (int q = 0; q < p.nr; ++q) most = std::max(most, p.m / p.R[q]);
    return (most + FFT_THREADS - 1) / FFT_THREADS;
}

// whole-spectrum multiplier of the forward (sgn 1) or backward (-1)
// derivative of n points of spacing d, 1 / n of the inverse included: the
// Nyquist bin real, as a complex-to-real inverse takes it
inline void fft_multiplier(int n, double d, double sgn, int k, double &re, double &im)
{
    const double two_pi = 8.0 * std::atan(1.0);
    const int q = 2 * k <= n ? k : n - k;
    const double w = q * (two_pi / (d * n * n)), ph = sgn * 0.5 * w * d * n;
    re = -w * std::sin(ph);
    im = 2 * k == n ? 0.0 : (2 * k < n ? 1.0 : -1.0) * w * std::cos(ph);
}

// the multiplier over the m points of plan p, in natural order
inline std::vector<double> fft_spectrum(const FftPlan &p, double d, double sgn)
{
    const int n = p.n, m = p.m;
    std::vector<double> out(2 * (size_t)m);
    if (m == n) {
        for (int k = 0; k < n; ++k) fft_multiplier(n, d, sgn, k, out[2 * k], out[2 * k + 1]);
        return out;
    }
    // (sums in extended precision: their rounding would be the largest error
    // of an FP64 derivative)
    typedef long double L;
    const L two_pi = 8.0L * std::atan(1.0L);
    auto roots = [&](int len) {
        std::vector<L> w(2 * (size_t)len);
        for (int q = 0; q < len; ++q) {
            w[2 * q] = std::cos(two_pi * q / len);
            w[2 * q + 1] = std::sin(two_pi * q / len);
        }
        return w;
    };
    // kernel c[j] = sum_k H(k) e^{2 pi i j k / n}; H(n - k) = conj H(k)
    std::vector<L> c(n, 0.0L), w = roots(n);
    std::vector<L> h(n + 2);
    for (int k = 0; 2 * k <= n; ++k) {
        const L wk = k * (two_pi / ((L)d * n * n)), ph = sgn * 0.5L * wk * d * n;
        h[2 * k] = -wk * std::sin(ph);
        h[2 * k + 1] = 2 * k == n ? 0.0L : wk * std::cos(ph);
    }
    for (int j = 0; j < n; ++j)
        for (int k = 1; 2 * k <= n; ++k) {
            const size_t q = (size_t)((int64_t)j * k % n);
            c[j] += (2 * k == n ? 1.0L : 2.0L) * (h[2 * k] * w[2 * q] - h[2 * k + 1] * w[2 * q + 1]);
        }
    // its spectrum: kernel positions -(n - 1) .. n - 1 of the m points
    w = roots(m);
    for (int k = 0; 2 * k <= m; ++k) {
        L re = 0.0L, im = 0.0L;
        size_t q = (size_t)(((int64_t)(1 - n) * k) % m + m) % m;
        for (int j = 1 - n; j < n; ++j) {
            const L v = c[j < 0 ? j + n : j];
            re += v * w[2 * q];
            im -= v * w[2 * q + 1];
            q += k;
            if (q >= (size_t)m) q -= m;
        }
        const size_t r = (size_t)((m - k) % m);
        out[2 * k] = out[2 * r] = (double)(re / m);
        out[2 * k + 1] = (double)(im / m);
        if (r != (size_t)k) out[2 * r + 1] = (double)(-im / m);
    }
    return out;
}

// twiddles of every pass, (re, im) pairs
inline std::vector<double> fft_twiddles(const FftPlan &p)
{
    const double two_pi = 8.0 * std::atan(1.0);
    std::vector<double> tw;
    tw.reserve(2 * p.tsz);
    for (int q = 0; q < p.nr; ++q)
        for (int t = 1; t < p.R[q] && p.S[q] > 1; ++t)
            for (int j = 0; j < p.S[q]; ++j) {
                const double th = two_pi * ((double)j * t) / ((double)p.S[q] * p.R[q]);
                tw.push_back(std::cos(th)); tw.push_back(-std::sin(th));
            }
    return tw;
}

// frequency of element t of the middle pass's butterfly b: the digits of
// the position, first pass fastest
inline int fft_freq(const FftPlan &p, int b, int t)
{
    int e = b * p.R[p.nr - 1] + t, k = 0, w = 1;
    for (int q = 0; q < p.nr; ++q) {
        k += w * (e / p.S[q]);
        e %= p.S[q];
        w *= p.R[q];
    }
    return k;
}

// up to 8 derivatives of one stage along one axis: job j differentiates
// field ((fields >> 4j) & 15) of x into d + ((slots >> 4j) & 15) N, with
// the forward multiplier if bit j of fwd is set
template <typename T>
struct DfftArgs {
    const T *x;
    T *d;
    unsigned N;
    uint32_t fields, slots, fwd;
    const Cx<T> *tw, *mul_f, *mul_b;
    int n, m, nr, tsz;
    uint32_t radix[FFT_MAXPASS], S[FFT_MAXPASS], nb[FFT_MAXPASS], toff[FFT_MAXPASS];
    uint32_t mS[FFT_MAXPASS], mN[FFT_MAXPASS];   // ceil(2^32 / S), ceil(2^32 / nb)
    uint32_t mL, pad;               // ceil(2^32 / R) of the last radix; 1 if its blocks are padded to R + 1
    int ls;                         // LDS elements per pair
    int nz2, lim;                   // row pitch, lines of the other axis
    int P, lP, ntiles, nblocks;
    int vec;                        // x: the two columns of a pair in one load
};

extern __shared__ __align__(16) unsigned char pstd_lds[];

// l / d for l < 2^16, m = ceil(2^32 / d) (d = 1: m = 0)
__device__ __forceinline__ uint32_t divm(uint32_t l, uint32_t m) { return m ? __umulhi(l, m) : l; }

// a group of V pairs at one position: one thread takes all of them, so that
// addresses, twiddles, multipliers and roots serve V transforms
template <typename T, int V>
struct __align__(V * 2 * sizeof(T) < 16 ? V * 2 * sizeof(T) : 16) Elem {
    Cx<T> c[V];
};

template <typename T, int V>
struct FftIO {
    const T *f;
    T *out;
    int r0;                         // first line of the tile
    Elem<T, V> *A;
    Cx<T> *tw;
};

// LDS position of element e of a line
template <typename T>
__device__ __forceinline__ uint32_t lds_at(const DfftArgs<T> &a, uint32_t e) { return e + a.pad * divm(e, a.mL); }

template <typename T, int AX>
__device__ __forceinline__ void outer_item(const DfftArgs<T> &a, uint32_t l, uint32_t &p, uint32_t &j)
{
    // along x the groups run fastest: 2 V P adjacent values of a row per
    // lanes at one position
    if (AX == 0) { p = l & (a.P - 1); j = l >> a.lP; }
    else { p = divm(l, a.mN[0]); j = l - p * a.nb[0]; }
}

// v[g][t] <- elements j + t S of group g's pair of lines
template <typename T, int V, int R, int AX, bool PAD>
__device__ __forceinline__ void load_lines(const DfftArgs<T> &a, const FftIO<T, V> &io, int p, uint32_t j,
                                           Cx<T> (&v)[V][R])
{
    const uint32_t S = a.S[0];
    // elements from n on (a padded line) are 0 and have no derivative
    auto in = [&](int t) { return !PAD || j + t * S < (uint32_t)a.n; };
    const int r0 = io.r0 + 2 * V * p;
    if (AX == 0) {
        const T *f = io.f + (size_t)j * a.nz2 + r0;
        const size_t st = (size_t)S * a.nz2;
        if (a.vec == 2 * V && r0 + 2 * V <= a.lim) {
#pragma unroll
            for (int t = 0; t < R; ++t) {
                if (!in(t)) continue;
                const Elem<T, V> e = *(const Elem<T, V> *)(f + t * st);
#pragma unroll
                for (int g = 0; g < V; ++g) v[g][t] = e.c[g];
            }
            return;
        }
#pragma unroll
        for (int g = 0; g < V; ++g) {
            const int r = r0 + 2 * g;
            if (a.vec) {
                if (r < a.lim) {
#pragma unroll
                    for (int t = 0; t < R; ++t) if (in(t)) v[g][t] = *(const Cx<T> *)(f + 2 * g + t * st);
                }
            } else {
                if (r < a.lim) {
#pragma unroll
                    for (int t = 0; t < R; ++t) if (in(t)) v[g][t].re = f[2 * g + t * st];
                }
                if (r + 1 < a.lim) {
#pragma unroll
                    for (int t = 0; t < R; ++t) if (in(t)) v[g][t].im = f[2 * g + t * st + 1];
                }
            }
        }
    } else {
#pragma unroll
        for (int g = 0; g < V; ++g) {
            const int r = r0 + 2 * g;
            const T *f = io.f + (size_t)r * a.nz2 + j;
            if (r < a.lim) {
#pragma unroll
                for (int t = 0; t < R; ++t) if (in(t)) v[g][t].re = f[t * S];
            }
            if (r + 1 < a.lim) {
#pragma unroll
                for (int t = 0; t < R; ++t) if (in(t)) v[g][t].im = f[a.nz2 + t * S];
            }
        }
    }
}

// the conjugates of v[g][t] -> elements j + t S of the derivatives
template <typename T, int V, int R, int AX, bool PAD>
__device__ __forceinline__ void store_lines(const DfftArgs<T> &a, const FftIO<T, V> &io, int p, uint32_t j,
                                            const Cx<T> (&v)[V][R])
{
    const uint32_t S = a.S[0];
    // elements from n on (a padded line) are 0 and have no derivative
    auto in = [&](int t) { return !PAD || j + t * S < (uint32_t)a.n; };
    const int r0 = io.r0 + 2 * V * p;
    if (AX == 0) {
        T *o = io.out + (size_t)j * a.nz2 + r0;
        const size_t st = (size_t)S * a.nz2;
        if (a.vec == 2 * V && r0 + 2 * V <= a.lim) {
#pragma unroll
            for (int t = 0; t < R; ++t) {
                if (!in(t)) continue;
                Elem<T, V> e;
#pragma unroll
                for (int g = 0; g < V; ++g) e.c[g] = {v[g][t].re, -v[g][t].im};
                *(Elem<T, V> *)(o + t * st) = e;
            }
            return;
        }
#pragma unroll
        for (int g = 0; g < V; ++g) {
            const int r = r0 + 2 * g;
            if (a.vec) {
                if (r < a.lim) {
#pragma unroll
                    for (int t = 0; t < R; ++t) if (in(t)) *(Cx<T> *)(o + 2 * g + t * st) = {v[g][t].re, -v[g][t].im};
                }
            } else {
                if (r < a.lim) {
#pragma unroll
                    for (int t = 0; t < R; ++t) if (in(t)) o[2 * g + t * st] = v[g][t].re;
                }
                if (r + 1 < a.lim) {
#pragma unroll
                    for (int t = 0; t < R; ++t) if (in(t)) o[2 * g + t * st + 1] = -v[g][t].im;
                }
            }
        }
    } else {
#pragma unroll
        for (int g = 0; g < V; ++g) {
            const int r = r0 + 2 * g;
            T *o = io.out + (size_t)r * a.nz2 + j;
            if (r < a.lim) {
#pragma unroll
                for (int t = 0; t < R; ++t) if (in(t)) o[t * S] = v[g][t].re;
            }
            if (r + 1 < a.lim) {
#pragma unroll
                for (int t = 0; t < R; ++t) if (in(t)) o[a.nz2 + t * S] = -v[g][t].im;
            }
        }
    }
}

template <typename T, int V, int R>
__device__ __forceinline__ void lds_load(const Elem<T, V> *s, uint32_t st, Cx<T> (&v)[V][R])
{
#pragma unroll
    for (int t = 0; t < R; ++t) {
        const Elem<T, V> e = s[t * st];
#pragma unroll
        for (int g = 0; g < V; ++g) v[g][t] = e.c[g];
    }
}
template <typename T, int V, int R>
__device__ __forceinline__ void lds_store(Elem<T, V> *s, uint32_t st, const Cx<T> (&v)[V][R])
{
#pragma unroll
    for (int t = 0; t < R; ++t) {
        Elem<T, V> e;
#pragma unroll
        for (int g = 0; g < V; ++g) e.c[g] = v[g][t];
        s[t * st] = e;
    }
}
template <typename T, int V, int R>
__device__ __forceinline__ void twiddle(const Cx<T> *tw, uint32_t S, Cx<T> (&v)[V][R])
{
#pragma unroll
    for (int t = 1; t < R; ++t) {
        const Cx<T> w = tw[(t - 1) * S];
#pragma unroll
        for (int g = 0; g < V; ++g) v[g][t] = cmul(v[g][t], w);
    }
}
template <typename T, int V, int R>
__device__ __forceinline__ void dft_group(Cx<T> (&v)[V][R])
{
#pragma unroll
    for (int g = 0; g < V; ++g) dft<T, R>(v[g]);
}

#define PSTD_RADIX(r, CALL)                                                                         \
    switch (r) {                                                                                    \
    case 2: { constexpr int R = 2; CALL; break; }                                                   \
    case 3: { constexpr int R = 3; CALL; break; }                                                   \
    case 4: { constexpr int R = 4; CALL; break; }                                                   \
    case 5: { constexpr int R = 5; CALL; break; }                                                   \
    case 6: { constexpr int R = 6; CALL; break; }                                                   \
    case 7: { constexpr int R = 7; CALL; break; }                                                   \
    case 8: { constexpr int R = 8; CALL; break; }                                                   \
    case 9: { constexpr int R = 9; CALL; break; }                                                   \
    case 10: { constexpr int R = 10; CALL; break; }                                                 \
    case 11: { constexpr int R = 11; CALL; break; }                                                 \
    case 12: { constexpr int R = 12; CALL; break; }                                                 \
    case 13: { constexpr int R = 13; CALL; break; }                                                 \
    case 14: { constexpr int R = 14; CALL; break; }                                                 \
    case 15: { constexpr int R = 15; CALL; break; }                                                 \
    default: { constexpr int R = 16; CALL; break; }                                                 \
    }

// The passes and the kernel: one item a thread, or, for pstd_rounds.hip, loops
// over the items of a pass.  (Two texts of one source in two translation
// units and not a template: any form of loop in the one-round kernels, even
// one the compiler removes, and the loop kernels' code between theirs moved
// their steps by up to 5%: 256 x 1296 FP64 156 and 165 us.)
#ifdef PSTD_ROUNDS
#define PSTD_ITEMS for (uint32_t l = threadIdx.x; l < items; l += blockDim.x)
namespace rounds {
#else
#define PSTD_ITEMS const uint32_t l = threadIdx.x; if (l < items)
#endif

// first pass: global memory -> LDS
template <typename T, int V, int R, int AX, bool PAD>
__device__ __forceinline__ void pass_first(const DfftArgs<T> &a, const FftIO<T, V> &io)
{
    const uint32_t S = a.S[0], items = a.nb[0] << a.lP;
    const uint32_t lst = S + a.pad * divm(S, a.mL);
#ifdef PSTD_ROUNDS
    for (int q = threadIdx.x; q < a.tsz; q += blockDim.x) io.tw[q] = a.tw[q];
    __syncthreads();
    PSTD_ITEMS {
        uint32_t p, j;
        outer_item<T, AX>(a, l, p, j);
        Cx<T> v[V][R];
#pragma unroll
        for (int g = 0; g < V; ++g)
#pragma unroll
            for (int t = 0; t < R; ++t) v[g][t] = {T(0), T(0)};
        load_lines<T, V, R, AX, PAD>(a, io, (int)p, j, v);
        dft_group<T, V, R>(v);
        twiddle<T, V, R>(io.tw + j, S, v);
        lds_store<T, V, R>(io.A + p * a.ls + lds_at(a, j), lst, v);
    }
#else
    const uint32_t l = threadIdx.x;
    uint32_t p = 0, j = 0;
    Cx<T> v[V][R];
#pragma unroll
    for (int g = 0; g < V; ++g)
#pragma unroll
        for (int t = 0; t < R; ++t) v[g][t] = {T(0), T(0)};
    if (l < items) {
        outer_item<T, AX>(a, l, p, j);
        load_lines<T, V, R, AX, PAD>(a, io, (int)p, j, v);
    }
    // the twiddle table, while the lines are on their way
    for (int q = threadIdx.x; q < a.tsz; q += blockDim.x) io.tw[q] = a.tw[q];
    __syncthreads();
    if (l < items) {
        dft_group<T, V, R>(v);
        twiddle<T, V, R>(io.tw + j, S, v);
        lds_store<T, V, R>(io.A + p * a.ls + lds_at(a, j), lst, v);
    }
#endif
}

// a pass between the first and the middle one, forward or transposed
template <typename T, int V, int R>
__device__ __forceinline__ void pass_inner(const DfftArgs<T> &a, const FftIO<T, V> &io, int q, bool inv)
{
    const uint32_t S = a.S[q], nb = a.nb[q], items = nb << a.lP;
    const uint32_t lst = S + a.pad * divm(S, a.mL);
    PSTD_ITEMS {
        const uint32_t p = divm(l, a.mN[q]), b = l - p * nb;
        const uint32_t blk = divm(b, a.mS[q]), j = b - blk * S;
        Elem<T, V> *s = io.A + p * a.ls + lds_at(a, blk * S * R + j);
        const Cx<T> *tw = io.tw + a.toff[q] + j;
        Cx<T> v[V][R];
        lds_load<T, V, R>(s, lst, v);
        if (inv) twiddle<T, V, R>(tw, S, v);
        dft_group<T, V, R>(v);
        if (!inv) twiddle<T, V, R>(tw, S, v);
        lds_store<T, V, R>(s, lst, v);
    }
}

// the middle: last forward pass, multiplier, first inverse pass
template <typename T, int V, int R>
__device__ __forceinline__ void pass_mid(const DfftArgs<T> &a, const FftIO<T, V> &io, const Cx<T> *mul)
{
    const int q = a.nr - 1;
    const uint32_t nb = a.nb[q], items = nb << a.lP;
    PSTD_ITEMS {
        const uint32_t p = divm(l, a.mN[q]), b = l - p * nb;
        Cx<T> h[R], v[V][R];
#pragma unroll
        for (int t = 0; t < R; ++t) h[t] = mul[t * nb + b];
        Elem<T, V> *s = io.A + p * a.ls + b * (R | 1);
        lds_load<T, V, R>(s, 1, v);
        dft_group<T, V, R>(v);
#pragma unroll
        for (int t = 0; t < R; ++t)
#pragma unroll
            for (int g = 0; g < V; ++g) {
                const Cx<T> z = cmul(v[g][t], h[t]);
                v[g][t] = {z.re, -z.im};
            }
        dft_group<T, V, R>(v);
        lds_store<T, V, R>(s, 1, v);
    }
}

// last pass: LDS -> global memory
template <typename T, int V, int R, int AX, bool PAD>
__device__ __forceinline__ void pass_last(const DfftArgs<T> &a, const FftIO<T, V> &io)
{
    const uint32_t S = a.S[0], items = a.nb[0] << a.lP;
    const uint32_t lst = S + a.pad * divm(S, a.mL);
    PSTD_ITEMS {
        uint32_t p, j;
        outer_item<T, AX>(a, l, p, j);
        Cx<T> v[V][R];
        lds_load<T, V, R>(io.A + p * a.ls + lds_at(a, j), lst, v);
        twiddle<T, V, R>(io.tw + j, S, v);
        dft_group<T, V, R>(v);
        store_lines<T, V, R, AX, PAD>(a, io, (int)p, j, v);
    }
}

// the derivative of the lines of tile b: AX 1 z (unit stride, row pairs
// r, r + 1), AX 0 x (stride nz2, column pairs c, c + 1); a missing partner
// reads as 0 and is not written
template <typename T, int V, int AX, bool PAD>
__device__ __forceinline__ void dfft_body(const DfftArgs<T> &a, int b)
{
    const int jb = b / a.ntiles, tile = b - jb * a.ntiles;
    FftIO<T, V> io;
    io.f = a.x + (size_t)((a.fields >> (4 * jb)) & 15) * a.N;
    io.out = a.d + (size_t)((a.slots >> (4 * jb)) & 15) * a.N;
    io.r0 = 2 * V * tile * a.P;
    io.A = (Elem<T, V> *)pstd_lds;
    io.tw = (Cx<T> *)(io.A + a.P * a.ls);
    const Cx<T> *mul = ((a.fwd >> jb) & 1) ? a.mul_f : a.mul_b;
    PSTD_RADIX(a.radix[0], (pass_first<T, V, R, AX, PAD>(a, io)))
    __syncthreads();
    // the inner passes forward, the middle, the inner passes back
    const int inner = a.nr - 2;
    for (int k = 0; k < 2 * inner + 1; ++k) {
        if (k == inner) {
            PSTD_RADIX(a.radix[a.nr - 1], (pass_mid<T, V, R>(a, io, mul)))
        } else {
            const int q = k < inner ? k + 1 : 2 * inner - k + 1;
            PSTD_RADIX(a.radix[q], (pass_inner<T, V, R>(a, io, q, k > inner)))
        }
        __syncthreads();
    }
    PSTD_RADIX(a.radix[0], (pass_last<T, V, R, AX, PAD>(a, io)))
}

// the derivatives of a stage along x (ax) and z (az) in one grid (either may
// have none); PAD: a line is shorter than its transform.  Every XCD takes a
// range of consecutive x tiles (adjacent columns share cache lines) and then a range of z tiles: the x tiles move
// more cache lines and take longer, so giving half of the XCDs only x tiles
// would leave the others waiting.
template <typename T, int V, bool PAD>
__global__ __launch_bounds__(FFT_THREADS) void pstd_dfft(const DfftArgs<T> ax, const DfftArgs<T> az)
{
    const int px = (ax.nblocks + 7) / 8, pz = (az.nblocks + 7) / 8;
    const int xcd = blockIdx.x % 8, i = blockIdx.x / 8;
    if (i < px) {
        if (xcd * px + i < ax.nblocks) dfft_body<T, V, 0, PAD>(ax, xcd * px + i);
    } else {
        if (xcd * pz + i - px < az.nblocks) dfft_body<T, V, 1, PAD>(az, xcd * pz + i - px);
    }
}

#undef PSTD_ITEMS
#ifdef PSTD_ROUNDS
}  // namespace rounds
#endif

// LDS elements of one group of pairs: the padded line, spread so that the P
// groups that lanes touch at one position lie on different banks (a row of
// banks holds 256 bytes)
inline int fft_line(const FftPlan &p, int V, int P, size_t elt)
{
    const int RL = p.R[p.nr - 1], row = std::max<int>(1, 256 / (V * 2 * elt));
    int ls = p.m / RL * (RL | 1);
    const int want = row / std::min(P, row);
    while (ls % row != want % row) ++ls;
    return ls;
}
inline size_t fft_lds(const FftPlan &p, int V, int P, size_t elt)
{
    return ((size_t)P * fft_line(p, V, P, elt) * V + (size_t)p.tsz) * 2 * elt;
}

}  // namespace pstd
}  // namespace sm
