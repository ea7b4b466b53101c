// Line-transform passes of the 3D fine-grid FFT (see fft_lines.hpp).
//
// A workgroup takes `lines` lines of one axis into LDS (element k of line c
// at LDS index c n + k when the axis is the contiguous one, k lines + c
// otherwise, so both loads are coalesced: whole lines, or rows of adjacent
// columns), runs the Stockham passes of its radix plan in place (every
// thread reads its butterflies into registers, the workgroup waits, every
// thread writes them), and stores the lines back.  Pass (radix R, p =
// product of the earlier radices), butterfly i of a line:
//
//   k = i mod p;  u_t = x[i + t n/R] w_n^{t k n/(p R)};  u = DFT_R(u);
//   x'[(i - k) R + k + t p] = u_t,   t = 0 .. R-1,
//
// which leaves the transform in natural order after the last pass.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>
#include <vector>

#include "fft_lines.hpp"

namespace mnufft {

namespace {

constexpr int kThreads = 512;
constexpr int kMaxGroupLines = 128;
constexpr int kMaxRowWords = 4864 / 32;  // bits of the longest axis

// Dynamic LDS per workgroup: lines + twiddles, at most 80 KB (two
// workgroups per CU) where the device allows it, else 64 KB; the static
// register arrays are sized for the largest.  Strided axes take `columns`
// adjacent columns (128-byte rows) when they fit.
template <typename T>
struct LdsElems;
template <>
struct LdsElems<float> {
    static constexpr int value = 9728;  // 80 KB less the per-line arrays
    static constexpr int base = 7680;   // 64 KB less the per-line arrays
    static constexpr int group = 18 * kThreads;  // elements of a workgroup's lines
    static constexpr int columns = 16;
};
template <>
struct LdsElems<double> {
    static constexpr int value = 4864;
    static constexpr int base = 3840;
    static constexpr int group = 9 * kThreads;
    static constexpr int columns = 8;
};
// static LDS: line bases, mode rows and two factors per line
constexpr size_t kLineLds = kMaxGroupLines * (2 * sizeof(int64_t) + 2 * sizeof(double));
constexpr size_t kLdsWide = 80 * 1024 - kLineLds;

template <typename T>
struct Cx {
    T re, im;
};

template <typename T>
__device__ inline Cx<T> cmul(Cx<T> a, Cx<T> b)
{
    return Cx<T>{a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
}
template <typename T>
__device__ inline Cx<T> cadd(Cx<T> a, Cx<T> b)
{
    return Cx<T>{a.re + b.re, a.im + b.im};
}
template <typename T>
__device__ inline Cx<T> csub(Cx<T> a, Cx<T> b)
{
    return Cx<T>{a.re - b.re, a.im - b.im};
}
// i s a for real s
template <typename T>
__device__ inline Cx<T> irot(Cx<T> a, T s)
{
    return Cx<T>{-s * a.im, s * a.re};
}

// q = a / b, r = a mod b for 0 <= a < 2^20, from a float reciprocal with
// one correction step.
__device__ inline void divmod_small(int a, int b, float inv_b, int &q, int &r)
{
    q = (int)((float)a * inv_b);
    r = a - q * b;
    if (r < 0) {
        --q;
        r += b;
    } else if (r >= b) {
        ++q;
        r -= b;
    }
}

// Small DFTs, X_s = sum_t u_t exp(2 pi i s t / R).  The other sign is the same
// transform with real and imaginary parts exchanged on the way in and out.
template <typename T>
__device__ __forceinline__ void dft2(Cx<T> *u)
{
    const Cx<T> a = u[0], b = u[1];
    u[0] = cadd(a, b);
    u[1] = csub(a, b);
}

template <typename T>
__device__ __forceinline__ void dft3(Cx<T> *u)
{
    const T s = (T)0.86602540378443864676;  // sin(2 pi / 3)
    const Cx<T> t1 = cadd(u[1], u[2]);
    const Cx<T> d = irot(csub(u[1], u[2]), s);
    const Cx<T> m = Cx<T>{u[0].re - (T)0.5 * t1.re, u[0].im - (T)0.5 * t1.im};
    u[0] = cadd(u[0], t1);
    u[1] = cadd(m, d);
    u[2] = csub(m, d);
}

template <typename T>
__device__ __forceinline__ void dft4(Cx<T> *u)
{
    const Cx<T> a = cadd(u[0], u[2]), b = csub(u[0], u[2]);
    const Cx<T> c = cadd(u[1], u[3]);
    const Cx<T> d = irot(csub(u[1], u[3]), (T)1);
    u[0] = cadd(a, c);
    u[2] = csub(a, c);
    u[1] = cadd(b, d);
    u[3] = csub(b, d);
}

template <typename T>
__device__ __forceinline__ void dft5(Cx<T> *u)
{
    const T c1 = (T)0.30901699437494742410;           // cos(2 pi / 5)
    const T c2 = (T)-0.80901699437494742410;          // cos(4 pi / 5)
    const T s1 = (T)0.95105651629515357212;  // sin(2 pi / 5)
    const T s2 = (T)0.58778525229247312917;  // sin(4 pi / 5)
    const Cx<T> a1 = cadd(u[1], u[4]), b1 = csub(u[1], u[4]);
    const Cx<T> a2 = cadd(u[2], u[3]), b2 = csub(u[2], u[3]);
    const Cx<T> u0 = u[0];
    const Cx<T> m1 = Cx<T>{u0.re + c1 * a1.re + c2 * a2.re, u0.im + c1 * a1.im + c2 * a2.im};
    const Cx<T> m2 = Cx<T>{u0.re + c2 * a1.re + c1 * a2.re, u0.im + c2 * a1.im + c1 * a2.im};
    // i (s1 b1 + s2 b2) and i (s2 b1 - s1 b2)
    const Cx<T> e1 = Cx<T>{-(s1 * b1.im + s2 * b2.im), s1 * b1.re + s2 * b2.re};
    const Cx<T> e2 = Cx<T>{-(s2 * b1.im - s1 * b2.im), s2 * b1.re - s1 * b2.re};
    u[0] = Cx<T>{u0.re + a1.re + a2.re, u0.im + a1.im + a2.im};
    u[1] = cadd(m1, e1);
    u[4] = csub(m1, e1);
    u[2] = cadd(m2, e2);
    u[3] = csub(m2, e2);
}

// Even and odd halves as two DFT4s, the odd half turned by w^s, w = exp(2 pi i / 8).
template <typename T>
__device__ __forceinline__ void dft8(Cx<T> *u)
{
    const T h = (T)0.70710678118654752440;  // cos(pi / 4)
    const T d = (T)1;
    Cx<T> e[4] = {u[0], u[2], u[4], u[6]};
    Cx<T> o[4] = {u[1], u[3], u[5], u[7]};
    dft4<T>(e);
    dft4<T>(o);
    const Cx<T> o1 = Cx<T>{h * (o[1].re - d * o[1].im), h * (o[1].im + d * o[1].re)};
    const Cx<T> o2 = irot(o[2], d);
    const Cx<T> o3 = Cx<T>{h * (-o[3].re - d * o[3].im), h * (-o[3].im + d * o[3].re)};
    u[0] = cadd(e[0], o[0]);
    u[4] = csub(e[0], o[0]);
    u[1] = cadd(e[1], o1);
    u[5] = csub(e[1], o1);
    u[2] = cadd(e[2], o2);
    u[6] = csub(e[2], o2);
    u[3] = cadd(e[3], o3);
    u[7] = csub(e[3], o3);
}

// cos and sin of 2 pi k / R, k = 1 .. (R - 1) / 2, for the prime radices 7, 11, 13.
__host__ __device__ constexpr double prime_cos(int R, int k)
{
    constexpr double c7[3] = {0.6234898018587336, -0.22252093395631434, -0.900968867902419};
    constexpr double c11[5] = {0.8412535328311812, 0.41541501300188644, -0.142314838273285,
                               -0.654860733945285, -0.9594929736144974};
    constexpr double c13[6] = {0.8854560256532099, 0.5680647467311559, 0.120536680255323,
                               -0.35460488704253545, -0.7485107481711012, -0.970941817426052};
    return R == 7 ? c7[k - 1] : (R == 11 ? c11[k - 1] : c13[k - 1]);
}
__host__ __device__ constexpr double prime_sin(int R, int k)
{
    constexpr double s7[3] = {0.7818314824680298, 0.9749279121818236, 0.43388373911755823};
    constexpr double s11[5] = {0.5406408174555976, 0.9096319953545183, 0.9898214418809328,
                               0.7557495743542583, 0.28173255684142967};
    constexpr double s13[6] = {0.4647231720437685, 0.8229838658936564, 0.992708874098054,
                               0.9350162426854148, 0.6631226582407952, 0.23931566428755768};
    return R == 7 ? s7[k - 1] : (R == 11 ? s11[k - 1] : s13[k - 1]);
}

// Odd prime R from the pairs t, R - t:
//   X_s = u_0 + sum_t (u_t + u_{R-t}) cos(2 pi s t / R) + i (u_t - u_{R-t}) sin(2 pi s t / R),
// t = 1 .. (R - 1) / 2, and X_{R-s} with the sine terms negated.
template <typename T, int R>
__device__ __forceinline__ void dft_prime(Cx<T> *u)
{
    constexpr int H = (R - 1) / 2;
    Cx<T> a[H], b[H];
#pragma unroll
    for (int t = 1; t <= H; ++t) {
        a[t - 1] = cadd(u[t], u[R - t]);
        b[t - 1] = csub(u[t], u[R - t]);
    }
    Cx<T> out[R];
    out[0] = u[0];
#pragma unroll
    for (int t = 0; t < H; ++t) out[0] = cadd(out[0], a[t]);
#pragma unroll
    for (int s = 1; s <= H; ++s) {
        Cx<T> m = u[0], e = Cx<T>{(T)0, (T)0};
#pragma unroll
        for (int t = 1; t <= H; ++t) {
            const int idx = (s * t) % R;
            const T c = (T)(idx <= H ? prime_cos(R, idx) : prime_cos(R, R - idx));
            const T sn = (T)(idx <= H ? prime_sin(R, idx) : -prime_sin(R, R - idx));
            m = Cx<T>{m.re + c * a[t - 1].re, m.im + c * a[t - 1].im};
            e = Cx<T>{e.re + sn * b[t - 1].re, e.im + sn * b[t - 1].im};
        }
        const Cx<T> ie = Cx<T>{-e.im, e.re};
        out[s] = cadd(m, ie);
        out[R - s] = csub(m, ie);
    }
#pragma unroll
    for (int t = 0; t < R; ++t) u[t] = out[t];
}

// cos(2 pi k / n) and sin(2 pi k / n) at compile time: the angle folded to
// the first octant on the integers, then the Taylor series.
constexpr double octant_series(double x, bool sine)
{
    double term = sine ? x : 1.0, sum = term;
    for (int i = sine ? 2 : 1; i < 28; i += 2) {
        term *= -x * x / (i * (i + 1.0));
        sum += term;
    }
    return sum;
}
constexpr double unit_cos(int k, int n)
{
    k = ((k % n) + n) % n;
    if (2 * k > n) k = n - k;                      // cos(-x) = cos x
    if (4 * k > n) return -unit_cos(n - 2 * k, 2 * n);  // cos(pi - x) = -cos x
    constexpr double tau = 6.28318530717958647692;
    return 8 * k <= n ? octant_series(tau * k / n, false)
                      : octant_series(tau * (n - 4.0 * k) / (4.0 * n), true);
}
template <int R>
struct UnitRoots {
    double c[R], s[R];
    constexpr UnitRoots() : c(), s()
    {
        for (int k = 0; k < R; ++k) {
            c[k] = unit_cos(k, R);
            s[k] = unit_cos(4 * k - R, 4 * R);  // sin x = cos(x - pi / 2)
        }
    }
};

template <typename T, int R>
__device__ __forceinline__ void dft(Cx<T> *u);

// R = A B with A and B coprime (prime-factor mapping, no twiddles): element
// (B a + A b) mod R, frequency k from (k mod A, k mod B).
template <typename T, int A, int B>
__device__ __forceinline__ void dft_coprime(Cx<T> *u)
{
    constexpr int R = A * B;
    Cx<T> y[B][A];
#pragma unroll
    for (int b = 0; b < B; ++b) {
#pragma unroll
        for (int a = 0; a < A; ++a) y[b][a] = u[(B * a + A * b) % R];
        dft<T, A>(y[b]);
    }
#pragma unroll
    for (int a = 0; a < A; ++a) {
        Cx<T> v[B];
#pragma unroll
        for (int b = 0; b < B; ++b) v[b] = y[b][a];
        dft<T, B>(v);
#pragma unroll
        for (int k = 0; k < R; ++k)
            if (k % A == a) u[k] = v[k % B];
    }
}

// R = Q Q: elements Q a + b, DFT_Q over a, twiddles w_R^{b k}, DFT_Q over b.
template <typename T, int Q>
__device__ __forceinline__ void dft_square(Cx<T> *u)
{
    constexpr int R = Q * Q;
    constexpr UnitRoots<R> w;
    Cx<T> y[Q][Q];
#pragma unroll
    for (int b = 0; b < Q; ++b) {
#pragma unroll
        for (int a = 0; a < Q; ++a) y[b][a] = u[Q * a + b];
        dft<T, Q>(y[b]);
#pragma unroll
        for (int k = 1; k < Q; ++k)
            if (b > 0)
                y[b][k] = cmul(y[b][k], Cx<T>{(T)w.c[b * k], (T)w.s[b * k]});
    }
#pragma unroll
    for (int k = 0; k < Q; ++k) {
        Cx<T> v[Q];
#pragma unroll
        for (int b = 0; b < Q; ++b) v[b] = y[b][k];
        dft<T, Q>(v);
#pragma unroll
        for (int m = 0; m < Q; ++m) u[k + Q * m] = v[m];
    }
}

template <typename T, int R>
__device__ __forceinline__ void dft(Cx<T> *u)
{
    if constexpr (R == 7 || R == 11 || R == 13) dft_prime<T, R>(u);
    if constexpr (R == 2) dft2<T>(u);
    if constexpr (R == 3) dft3<T>(u);
    if constexpr (R == 4) dft4<T>(u);
    if constexpr (R == 5) dft5<T>(u);
    if constexpr (R == 6) dft_coprime<T, 2, 3>(u);
    if constexpr (R == 8) dft8<T>(u);
    if constexpr (R == 9) dft_square<T, 3>(u);
    if constexpr (R == 10) dft_coprime<T, 2, 5>(u);
    if constexpr (R == 12) dft_coprime<T, 4, 3>(u);
    if constexpr (R == 15) dft_coprime<T, 3, 5>(u);
    if constexpr (R == 16) dft_square<T, 4>(u);
}

// Per-line data of a workgroup in LDS: grid base, mode row and the line's
// deconvolution factors (type 2: the u and v axes' 1/phi_hat; type 1: their
// product in axis order).
struct LineData {
    int64_t *base, *mrow = nullptr;
    double *f1 = nullptr, *f2 = nullptr;
    void *modes = nullptr;  // this vector's modes (IO 1, 2)
    uint32_t *rows = nullptr;  // the elements to write, as bits (IO 3)
};

// Mode storage index of signed frequency m on an axis of N modes.
__device__ inline int64_t mode_slot(int64_t m, int64_t N, int centered)
{
    return centered ? m + N / 2 : (m >= 0 ? m : m + N);
}

// A butterfly of the first pass reads, and one of the last pass writes, the
// elements e = i + t nb, t = 0 .. R - 1.  visit(t, kept): whether the lane's
// element lies in the kept window [0, hi) and [n - lo, n) (for most t the
// same for every lane: scalar branches on the masks).
template <int R, typename Visit>
__device__ __forceinline__ void for_kept(const LineFftKept &m, int i, int nb, int n, int hi, int lo,
                                         Visit visit)
{
#pragma unroll
    for (int t = 0; t < R; ++t) {
        if ((m.all >> t) & 1u) {
            visit(t, true);
        } else if ((m.some >> t) & 1u) {
            const int e = i + t * nb;
            visit(t, e < hi || e >= n - lo);
        } else {
            visit(t, false);
        }
    }
}

// IO (the launch's mode reads or writes): 0 grid only; 1 the first pass
// reads the modes and predeconvolves them (type 2); 2 the last pass writes
// the deconvolved modes (type 1); 3 the last pass writes the elements whose
// bit is set (a sparse type 2, whose points reach few cells).
//
// What bounds the passes: HBM for FP32 (512^3, 4 vectors: x 1.55 ms, y 0.75
// ms, 4.1 and 4.3 TB/s where a copy reaches 4.6), HBM latency on the short
// rows of long FP64 axes (900^3: x 1.5, y 2.2 ms, z 5.8 ms for every row, 3.7
// ms for the marked ones of a sparse type 2).  The vector ALU bounded them
// before (x 2.1, y 1.0 ms; 900^3 1.8, 2.7, 7.1 ms): an address product, a
// window test and index divisions for every element, divisions of the pass
// constants in every thread and five small radices at 900 took 124 (FP32) and
// 156 (FP64) instructions an element; now one 64-bit pointer a butterfly
// stepped by a uniform stride, windows as masks over t, constants from the
// host and the largest radices: 56 and 77.

// One butterfly index of the workgroup: line c, butterfly i of the line.
template <typename T>
__device__ inline void butterfly(const LineFftAxis &P, const LineFftPass &ps, int b, int *c, int *i)
{
    if (P.line_major) {
        divmod_small(b, ps.nb, ps.inv_nb, *c, *i);
    } else {
        *i = b >> P.log_lines;
        *c = b & (P.lines - 1);
    }
}

template <typename T, int R>
__device__ __forceinline__ void exchange(Cx<T> (&u)[R])
{
#pragma unroll
    for (int t = 0; t < R; ++t) u[t] = Cx<T>{u[t].im, u[t].re};
}

// u_t times w^(t k), the pass's twiddles.
template <typename T, int R>
__device__ __forceinline__ void turn(Cx<T> (&u)[R], const Cx<T> *tw, int wstep)
{
#pragma unroll
    for (int t = 1; t < R; ++t) {
        tw += wstep;
        u[t] = cmul(u[t], *tw);
    }
}

// The first pass (p = 1, no twiddles): butterflies from the grid or the
// modes into LDS.
template <typename T, int R, int IO>
__device__ __forceinline__ void pass_in(Cx<T> *X, const LineFftAxis &P, const LineFftPass &ps,
                                        const Cx<T> *__restrict__ grid, const LineData &ld)
{
    const int threads = (int)blockDim.x;
    const int n = P.n, nb = ps.nb, total = P.lines * nb;
    const int ks = P.line_major ? 1 : P.lines, cs = P.line_major ? n : 1;
    const int64_t tstep = (int64_t)nb * P.estride;  // elements between a butterfly's
    // mode slot of element e: e + half at the window's low end, e + back at
    // its high end
    const int half = P.centered ? (int)(P.eN / 2) : 0;
    const int back = P.centered ? half - n : (int)P.eN - n;
    for (int b = (int)threadIdx.x; b < total; b += threads) {
        int c, i;
        butterfly<T>(P, ps, b, &c, &i);
        Cx<T> u[R];
        const int64_t bc = ld.base[c];
        if (bc < 0) {
#pragma unroll
            for (int t = 0; t < R; ++t) u[t] = Cx<T>{(T)0, (T)0};
        } else if constexpr (IO == 1) {
            // the predeconvolution: mode times (1/phi_hat) in axis order
            const Cx<T> *row = (const Cx<T> *)ld.modes + ld.mrow[c];
            const double g1 = ld.f1[c], g2 = ld.f2[c];
            const double *phi = P.inv_phihat + P.eph;
            for_kept<R>(P.in, i, nb, n, P.in_hi, P.in_lo, [&](int t, bool in) {
                u[t] = Cx<T>{(T)0, (T)0};
                if (in) {
                    const int e = i + t * nb;
                    const bool low = e < P.in_hi;
                    double amp = 1.0;
                    amp *= phi[low ? e : n - e];
                    amp *= g1;
                    amp *= g2;
                    const Cx<T> src = row[(int64_t)(e + (low ? half : back)) * P.ems];
                    const T ta = (T)amp;
                    u[t] = Cx<T>{src.re * ta, src.im * ta};
                }
            });
        } else {
            const Cx<T> *src = grid + bc + (int64_t)i * P.estride;
            for_kept<R>(P.in, i, nb, n, P.in_hi, P.in_lo, [&](int t, bool in) {
                u[t] = Cx<T>{(T)0, (T)0};
                if (in) u[t] = src[t * tstep];
            });
        }
        if (P.exchange) exchange<T, R>(u);
        dft<T, R>(u);
        Cx<T> *out = X + i * R * ks + c * cs;
#pragma unroll
        for (int t = 0; t < R; ++t) out[t * ks] = u[t];
    }
    __syncthreads();
}

// (MAXB butterflies a thread cover the largest group at kThreads threads; a
// smaller workgroup has a thread for every butterfly of every pass.)
//
// A middle pass, in place in LDS: every thread reads its butterflies into
// registers, the workgroup waits, every thread writes them.
template <typename T, int R>
__device__ __forceinline__ void pass_mid(Cx<T> *X, const Cx<T> *tw, const LineFftAxis &P,
                                         const LineFftPass &ps)
{
    constexpr int MAXB = (LdsElems<T>::group / R + kThreads - 1) / kThreads;
    const int threads = (int)blockDim.x;
    const int n = P.n, nb = ps.nb, total = P.lines * nb;
    const int ks = P.line_major ? 1 : P.lines, cs = P.line_major ? n : 1;
    const int in_step = nb * ks, out_step = ps.p * ks;
    Cx<T> u[MAXB][R];
    int at[MAXB];
#pragma unroll
    for (int s = 0; s < MAXB; ++s) {
        const int b = (int)threadIdx.x + s * threads;
        at[s] = -1;
        if (b < total) {
            int c, i, q, k;
            butterfly<T>(P, ps, b, &c, &i);
            divmod_small(i, ps.p, ps.inv_p, q, k);
            const Cx<T> *src = X + i * ks + c * cs;
#pragma unroll
            for (int t = 0; t < R; ++t) u[s][t] = src[t * in_step];
            turn<T, R>(u[s], tw, k * ps.tw_step);
            dft<T, R>(u[s]);
            at[s] = (q * ps.p * R + k) * ks + c * cs;
        }
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < MAXB; ++s) {
        if (at[s] < 0) continue;
        Cx<T> *out = X + at[s];
#pragma unroll
        for (int t = 0; t < R; ++t) out[t * out_step] = u[s][t];
    }
    __syncthreads();
}

// The last pass (p R = n): butterflies from LDS to the grid or the modes.
// Radix 1 only writes (an axis of one pass).
template <typename T, int R, int IO>
__device__ __forceinline__ void pass_out(const Cx<T> *X, const Cx<T> *tw, const LineFftAxis &P,
                                         const LineFftPass &ps, Cx<T> *__restrict__ grid,
                                         const LineData &ld)
{
    const int threads = (int)blockDim.x;
    const int n = P.n, nb = ps.nb, total = P.lines * nb;
    const int ks = P.line_major ? 1 : P.lines, cs = P.line_major ? n : 1;
    const int in_step = nb * ks;
    const int64_t tstep = (int64_t)nb * P.estride;
    const int half = P.centered ? (int)(P.eN / 2) : 0;
    const int back = P.centered ? half - n : (int)P.eN - n;
    for (int b = (int)threadIdx.x; b < total; b += threads) {
        int c, i;
        butterfly<T>(P, ps, b, &c, &i);
        const int64_t bc = ld.base[c];
        if (bc < 0) continue;
        Cx<T> u[R];
        const Cx<T> *src = X + i * ks + c * cs;
#pragma unroll
        for (int t = 0; t < R; ++t) u[t] = src[t * in_step];
        if constexpr (R > 1) {
            turn<T, R>(u, tw, i * ps.tw_step);
            dft<T, R>(u);
        }
        if (P.exchange) exchange<T, R>(u);
        if constexpr (IO == 2) {
            // the deconvolution: cell times (1/phi_hat) in axis order
            Cx<T> *row = (Cx<T> *)ld.modes + ld.mrow[c];
            const double g = ld.f1[c];
            const double *phi = P.inv_phihat + P.eph;
            for_kept<R>(P.out, i, nb, n, P.out_hi, P.out_lo, [&](int t, bool in) {
                if (in) {
                    const int e = i + t * nb;
                    const bool low = e < P.out_hi;
                    double amp = g;
                    amp *= phi[low ? e : n - e];
                    const T ta = (T)amp;
                    row[(int64_t)(e + (low ? half : back)) * P.ems] =
                        Cx<T>{u[t].re * ta, u[t].im * ta};
                }
            });
        } else {
            Cx<T> *out = grid + bc + (int64_t)i * P.estride;
            for_kept<R>(P.out, i, nb, n, P.out_hi, P.out_lo, [&](int t, bool in) {
                if constexpr (IO == 3) {
                    const int e = i + t * nb;
                    in = in && ((ld.rows[e >> 5] >> (e & 31)) & 1u);
                }
                if (in) out[t * tstep] = u[t];
            });
        }
    }
}

#define MNUFFT_RADICES(X) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11) X(12) X(13) X(15) X(16)

// The transform of workgroup `group`'s lines of one axis pass (P) of the
// grid `grid` (one vector), X: (lines + 1) n elements of LDS.
template <typename T, int IO>
__device__ __forceinline__ void fft_lines_body(const LineFftAxis &P, Cx<T> *__restrict__ grid,
                                               const Cx<T> *__restrict__ tw_global,
                                               int64_t group, Cx<T> *X, const LineData &ld)
{
    int64_t *base = ld.base;
    Cx<T> *tw = X + P.lines * P.n;
    const int n = P.n;
    for (int m = threadIdx.x; m < n; m += (int)blockDim.x) tw[m] = tw_global[m];
    // (line numbers are below 2^32: at most 65536 per axis)
    const uint32_t nu = (uint32_t)P.nu, nlines = (uint32_t)(P.nu * P.nv);
    const uint32_t line0 = (uint32_t)group * (uint32_t)P.lines;
    for (int c = threadIdx.x; c < P.lines; c += (int)blockDim.x) {
        const uint32_t L = line0 + (uint32_t)c;
        int64_t b = -1;
        if (L < nlines) {
            const int64_t w = L / nu, u = L - (uint32_t)w * nu;
            const int64_t uu = u < P.u_hi ? u : u + P.u_gap;
            const int64_t vv = w < P.v_hi ? w : w + P.v_gap;
            b = uu * P.su + vv * P.sv;
            if constexpr (IO == 1 || IO == 2) {
                // the line's mode row and factors (u, v: fine indices of the
                // kept windows of their axes)
                int64_t mr = 0;
                double fu = 1.0, fv = 1.0;
                if (P.has_u) {
                    const int64_t m = uu < (P.uN + 1) / 2 ? uu : uu - P.un;
                    mr += mode_slot(m, P.uN, P.centered) * P.ums;
                    fu = P.inv_phihat[P.uph + (m < 0 ? -m : m)];
                }
                if (P.has_v) {
                    const int64_t m = vv < (P.vN + 1) / 2 ? vv : vv - P.vn;
                    mr += mode_slot(m, P.vN, P.centered) * P.vms;
                    fv = P.inv_phihat[P.vph + (m < 0 ? -m : m)];
                }
                ld.mrow[c] = mr;
                if constexpr (IO == 1) {
                    ld.f1[c] = fu;
                    ld.f2[c] = fv;
                } else {
                    double amp = 1.0;
                    amp *= fu;
                    if (P.has_v) amp *= fv;
                    ld.f1[c] = amp;
                }
            }
        }
        base[c] = b;
    }
    __syncthreads();
    if (P.npass < 2) return;  // one cell
#define MNUFFT_IN(R)                                              \
    case R: pass_in<T, R, IO == 1 ? 1 : 0>(X, P, P.pass[0], grid, ld); break;
    switch (P.pass[0].radix) { MNUFFT_RADICES(MNUFFT_IN) }
#undef MNUFFT_IN
    const int last = P.npass - 1;
    for (int s = 1; s < last; ++s) {
#define MNUFFT_MID(R) \
    case R: pass_mid<T, R>(X, tw, P, P.pass[s]); break;
        switch (P.pass[s].radix) { MNUFFT_RADICES(MNUFFT_MID) }
#undef MNUFFT_MID
    }
#define MNUFFT_OUT(R)                                             \
    case R: pass_out<T, R, IO == 1 ? 0 : IO>(X, tw, P, P.pass[last], grid, ld); break;
    switch (P.pass[last].radix) { MNUFFT_RADICES(MNUFFT_OUT) MNUFFT_OUT(1) }
#undef MNUFFT_OUT
}

// Workgroups go round the eight XCDs in turn; neighbouring groups of a
// strided pass share cache lines, DRAM pages and page translations, so each
// XCD takes a contiguous run of groups.
__device__ inline int64_t xcd_group(uint32_t block, uint32_t blocks)
{
    const uint32_t x = block & 7u, per = blocks >> 3, rest = blocks & 7u;
    return (int64_t)x * per + (x < rest ? x : rest) + (block >> 3);
}

// One plan's axis pass: workgroup (group, vector); IO / modes_all: this
// launch's mode reads or writes (all vectors' modes).
template <typename T, int IO>
__global__ __launch_bounds__(kThreads, 4) void k_fft_lines(const LineFftAxis *__restrict__ ax,
                                                           void *modes_all, T *__restrict__ data,
                                                           const Cx<T> *__restrict__ tw_global,
                                                           const uint32_t *__restrict__ rows_all)
{
    const LineFftAxis &P = *ax;
    extern __shared__ __align__(16) unsigned char lds_raw[];
    Cx<T> *grid = (Cx<T> *)data + (int64_t)blockIdx.y * P.vec_stride;
    const int64_t group = P.line_major ? (int64_t)blockIdx.x : xcd_group(blockIdx.x, gridDim.x);
    __shared__ int64_t base[kMaxGroupLines];
    if constexpr (IO == 0) {
        fft_lines_body<T, 0>(P, grid, tw_global, group, (Cx<T> *)lds_raw, LineData{base});
    } else if constexpr (IO == 3) {
        __shared__ uint32_t rows[kMaxRowWords];
        const int words = (P.n + 31) / 32;
        for (int w = threadIdx.x; w < words; w += (int)blockDim.x) rows[w] = rows_all[group * words + w];
        fft_lines_body<T, 3>(P, grid, tw_global, group, (Cx<T> *)lds_raw,
                             LineData{base, nullptr, nullptr, nullptr, nullptr, rows});
    } else {
        __shared__ int64_t mrow[kMaxGroupLines];
        __shared__ double f1[kMaxGroupLines], f2[kMaxGroupLines];
        Cx<T> *modes = (Cx<T> *)modes_all + (int64_t)blockIdx.y * P.mode_total;
        fft_lines_body<T, IO>(P, grid, tw_global, group, (Cx<T> *)lds_raw,
                              LineData{base, mrow, f1, f2, modes});
    }
}

// The same axis pass of many plans (one vector each) in one launch: job q
// takes workgroups [group0[q], group0[q + 1]).
template <typename T>
__global__ __launch_bounds__(kThreads, 4) void k_fft_lines_many(const LineFftJob *__restrict__ jobs,
                                                                int njobs)
{
    extern __shared__ __align__(16) unsigned char lds_raw[];
    __shared__ int64_t base[kMaxGroupLines];
    const int64_t b = blockIdx.x;
    int lo = 0, hi = njobs - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (jobs[mid].group0 <= b)
            lo = mid;
        else
            hi = mid - 1;
    }
    // the job is the workgroup's: its fields in scalar registers
    const LineFftJob &J = jobs[__builtin_amdgcn_readfirstlane(lo)];
    fft_lines_body<T, 0>(*J.ax, (Cx<T> *)J.grid, (const Cx<T> *)J.tw, b - J.group0,
                         (Cx<T> *)lds_raw, LineData{base});
}

// Radix plan: the fewest passes of radix 2 .. 16 (each costs an LDS round
// trip of every element, two barriers and the twiddles), of those the one
// with the smallest largest radix (its registers, its idle lanes), larger
// radices first (the first pass's reads are in flight together); false for
// prime factors beyond 13.  At 900 cells 10 x 10 x 9 instead of 5 x 5 x 3 x 3
// x 4, at 256 16 x 16 instead of 8 x 8 x 4.
bool radix_plan(int n, LineFftAxis *ax)
{
    int best[kLineFftMaxPasses], cur[kLineFftMaxPasses], best_count = 0;
    const auto search = [&](const auto &self, int m, int most, int depth) -> void {
        if (m == 1) {
            if (best_count == 0 || depth < best_count ||
                (depth == best_count && cur[0] < best[0])) {
                best_count = depth;
                for (int i = 0; i < depth; ++i) best[i] = cur[i];
            }
            return;
        }
        if (depth == kLineFftMaxPasses || (best_count && depth >= best_count)) return;
        for (int r = std::min(most, m); r >= 2; --r)
            if (m % r == 0 && r != 14) {
                cur[depth] = r;
                self(self, m / r, r, depth + 1);
            }
    };
    if (n < 1) return false;
    search(search, n, 16, 0);
    if (best_count == 0 && n != 1) return false;
    ax->n = n;
    ax->npass = best_count;
    int p = 1;
    for (int i = 0; i < best_count; ++i) {
        const int r = best[i];
        ax->pass[i] = LineFftPass{r, p, n / (p * r), n / r, (float)r / (float)n, 1.0f / (float)p};
        p *= r;
    }
    if (ax->npass == 1)  // the write as a pass of its own
        ax->pass[ax->npass++] = LineFftPass{1, n, 1, n, 1.0f / (float)n, 1.0f / (float)n};
    return true;
}

// Masks of a pass of radix r for the kept window [0, hi) and [n - lo, n).
LineFftKept kept_masks(int r, int n, int hi, int lo)
{
    LineFftKept m{0u, 0u};
    const int nb = n / r;
    for (int t = 0; t < r; ++t) {
        const int e0 = t * nb, e1 = e0 + nb;
        if (e1 <= hi || e0 >= n - lo)
            m.all |= 1u << t;
        else if (e0 < hi || e1 > n - lo)
            m.some |= 1u << t;
    }
    return m;
}

// Whether the line kernels may take the wide LDS budget (set once).
bool wide_lds()
{
    static std::once_flag once;
    static bool ok = false;
    std::call_once(once, [] {
        const void *kernels[] = {
            (const void *)k_fft_lines<float, 0>,  (const void *)k_fft_lines<float, 1>,
            (const void *)k_fft_lines<float, 2>,  (const void *)k_fft_lines<float, 3>,
            (const void *)k_fft_lines<double, 0>, (const void *)k_fft_lines<double, 1>,
            (const void *)k_fft_lines<double, 2>, (const void *)k_fft_lines<double, 3>,
            (const void *)k_fft_lines_many<float>, (const void *)k_fft_lines_many<double>};
        ok = true;
        for (const void *k : kernels)
            ok = ok && hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize,
                                           (int)kLdsWide) == hipSuccess;
        (void)hipGetLastError();
    });
    return ok;
}

// Lines per workgroup: the lines and the twiddle table fit the LDS array
// (`wide`: the 80 KB budget, else 64 KB); along the contiguous axis an element
// per thread at least and few enough groups for about 2048 workgroups (`count`
// lines in all), small groups sharing a CU.
bool group_lines(int n, bool line_major, bool f64, int64_t count, bool wide, LineFftAxis *ax)
{
    const int lds = f64 ? (wide ? LdsElems<double>::value : LdsElems<double>::base)
                        : (wide ? LdsElems<float>::value : LdsElems<float>::base);
    const int most = f64 ? LdsElems<double>::group : LdsElems<float>::group;
    if (2 * n > lds) return false;
    ax->line_major = line_major ? 1 : 0;
    if (line_major) {
        const int64_t fill = std::max<int64_t>((kThreads + n - 1) / n, count / 2048);
        int c = (int)std::min<int64_t>(kMaxGroupLines, fill);
        while (c > 1 && ((c + 1) * n > lds || c * n > most)) --c;
        ax->lines = c;
        ax->log_lines = 0;
    } else {
        int c = f64 ? LdsElems<double>::columns : LdsElems<float>::columns;
        while (c > 1 && ((c + 1) * n > lds || c * n > most)) c /= 2;
        ax->lines = c;
        ax->log_lines = 0;
        while ((1 << ax->log_lines) < c) ++ax->log_lines;
    }
    // a thread for every butterfly of the pass with most of them, at most
    // kThreads, rounded up to whole waves for every SIMD of the CU (7 waves
    // ran 900-cell passes 9% slower than 8).  512 threads for every axis left
    // most waves of short ones idle and fewer workgroups on a CU: 256^3 FP32
    // type 2 x / y / z 44 / 28 / 50 -> 27 / 22 / 37 us, 162 x 128 x 100 FP64
    // 18 / 15 / 28 -> 18 / 11 / 15 us.
    int most_butterflies = 1;
    for (int i = 0; i < ax->npass; ++i)
        most_butterflies = std::max(most_butterflies, ax->lines * ax->pass[i].nb);
    ax->threads = 64;
    while (ax->threads < kThreads && ax->threads < most_butterflies) ax->threads *= 2;
    return ax->lines >= 1;
}

// Keep only the window of N modes of an axis of n cells.
void keep_u(LineFftAxis &a, int64_t n, int64_t N)
{
    a.nu = N;
    a.u_hi = (N + 1) / 2;
    a.u_gap = n - N;
}
void keep_v(LineFftAxis &a, int64_t n, int64_t N)
{
    a.nv = N;
    a.v_hi = (N + 1) / 2;
    a.v_gap = n - N;
}

}  // namespace

bool LineFft::supported(int dim, const int64_t *fine, bool f64)
{
    if (dim != 2 && dim != 3) return false;
    for (int a = 0; a < dim; ++a) {
        LineFftAxis ax;
        if (fine[a] < 1 || fine[a] > 65536 || !radix_plan((int)fine[a], &ax) ||
            !group_lines((int)fine[a], a == 0, f64, 1, wide_lds(), &ax))
            return false;
    }
    return true;
}

int64_t LineFft::row_length_limit(bool f64)
{
    return f64 ? LdsElems<double>::value / 5 : LdsElems<float>::value / 9;
}

LineFft::~LineFft()
{
    if (tables_) (void)hipFree(tables_);
}

bool LineFft::init(int dim, const int64_t *fine, const int64_t *n_modes, int type, bool f64,
                   int isign, const double *inv_phihat, const int64_t *phihat_off,
                   bool centered)
{
    if (!supported(dim, fine, f64)) {
        set_error("line FFT needs a 2D or 3D grid of 2,3,5,7,11,13-smooth lengths within the "
                  "LDS lines");
        return false;
    }
    naxes_ = dim;
    type_ = type;
    f64_ = f64;
    dir_ = isign >= 0 ? 1 : -1;
    const int64_t n0 = fine[0], n1 = fine[1], n2 = dim == 3 ? fine[2] : 1;
    fine_total_ = n0 * n1 * n2;
    const int64_t plane = n0 * n1;
    for (int a = 0; a < dim; ++a) {
        LineFftAxis &x = ax_[a];
        x = LineFftAxis{};
        radix_plan((int)fine[a], &x);
        x.in_hi = x.out_hi = (int)fine[a];
        x.in_lo = x.out_lo = 0;
        x.vec_stride = fine_total_;
    }
    // x: lines (y, z); y: columns (x, z); z: columns (x, y); a 2D grid has no z
    ax_[0].estride = 1;
    ax_[0].nu = ax_[0].u_hi = n1;
    ax_[0].su = n0;
    ax_[0].nv = ax_[0].v_hi = n2;
    ax_[0].sv = plane;
    ax_[1].estride = n0;
    ax_[1].nu = ax_[1].u_hi = n0;
    ax_[1].su = 1;
    ax_[1].nv = ax_[1].v_hi = n2;
    ax_[1].sv = plane;
    if (dim == 3) {
        ax_[2].estride = plane;
        ax_[2].nu = ax_[2].u_hi = n0;
        ax_[2].su = 1;
        ax_[2].nv = ax_[2].v_hi = n1;
        ax_[2].sv = n0;
    }
    const int64_t N0 = n_modes[0], N1 = n_modes[1], N2 = dim == 3 ? n_modes[2] : 1;
    auto window = [](int &hi, int &lo, int64_t N) {
        hi = (int)((N + 1) / 2);
        lo = (int)(N / 2);
    };
    if (type == 2) {
        keep_u(ax_[0], n1, N1);
        window(ax_[0].in_hi, ax_[0].in_lo, N0);
        window(ax_[1].in_hi, ax_[1].in_lo, N1);
        if (dim == 3) {
            keep_v(ax_[0], n2, N2);
            keep_v(ax_[1], n2, N2);
            window(ax_[2].in_hi, ax_[2].in_lo, N2);
        }
    } else {
        window(ax_[0].out_hi, ax_[0].out_lo, N0);
        keep_u(ax_[1], n0, N0);
        window(ax_[1].out_hi, ax_[1].out_lo, N1);
        if (dim == 3) {
            keep_u(ax_[2], n0, N0);
            keep_v(ax_[2], n1, N1);
            window(ax_[2].out_hi, ax_[2].out_lo, N2);
        }
    }
    const bool wide = wide_lds();
    for (int a = 0; a < dim; ++a)
        group_lines((int)fine[a], a == 0, f64, ax_[a].nu * ax_[a].nv, wide, &ax_[a]);
    // the pass that reads (type 2: x) or writes (type 1: the last axis) modes
    LineFftAxis &mx = type == 2 ? ax_[0] : ax_[dim - 1];
    mx.centered = centered ? 1 : 0;
    mx.inv_phihat = inv_phihat;
    int64_t mstride[3] = {1, 1, 1};
    int64_t stride = 1;
    for (int a = 0; a < dim; ++a) {
        mstride[a] = stride;
        stride *= n_modes[a];
    }
    mx.mode_total = stride;
    // type 2: x lines over (y, z); type 1: last-axis lines over (x, y)
    const int ua = type == 2 ? 1 : 0, va = dim == 3 ? (type == 2 ? 2 : 1) : -1;
    const int ea = type == 2 ? 0 : dim - 1;
    mx.has_u = 1;
    mx.uN = n_modes[ua];
    mx.un = fine[ua];
    mx.ums = mstride[ua];
    mx.uph = phihat_off[ua];
    mx.has_v = va >= 0 ? 1 : 0;
    if (va >= 0) {
        mx.vN = n_modes[va];
        mx.vn = fine[va];
        mx.vms = mstride[va];
        mx.vph = phihat_off[va];
    }
    mx.eN = n_modes[ea];
    mx.ems = mstride[ea];
    mx.eph = phihat_off[ea];
    for (int a = 0; a < dim; ++a) {
        LineFftAxis &x = ax_[a];
        if (x.npass == 0) continue;
        x.exchange = dir_ < 0 ? 1 : 0;
        x.in = kept_masks(x.pass[0].radix, x.n, x.in_hi, x.in_lo);
        x.out = kept_masks(x.pass[x.npass - 1].radix, x.n, x.out_hi, x.out_lo);
    }
    // one device allocation: the axes (for batches), then per axis the
    // twiddles w_n^m = exp(2 pi i m / n), from long double
    const size_t eb = f64 ? 2 * sizeof(double) : 2 * sizeof(float);
    size_t at[3], bytes = (sizeof(ax_) + 255) / 256 * 256;
    for (int a = 0; a < dim; ++a) {
        at[a] = bytes;
        bytes += (eb * (size_t)fine[a] + 255) / 256 * 256;
    }
    std::vector<unsigned char> host(bytes, 0);
    std::memcpy(host.data(), ax_, sizeof(ax_));
    for (int a = 0; a < dim; ++a) {
        const int n = (int)fine[a];
        float *hf = (float *)(host.data() + at[a]);
        double *hd = (double *)(host.data() + at[a]);
        for (int m = 0; m < n; ++m) {
            const long double ang =
                2.0L * 3.14159265358979323846264338327950288L * (long double)m / (long double)n;
            const long double c = cosl(ang), s = sinl(ang);
            if (f64) {
                hd[2 * m] = (double)c;
                hd[2 * m + 1] = (double)s;
            } else {
                hf[2 * m] = (float)c;
                hf[2 * m + 1] = (float)s;
            }
        }
    }
    if (tables_) (void)hipFree(tables_);
    tables_ = nullptr;
    if (!hip_ok(hipMalloc(&tables_, bytes), "line FFT tables") ||
        !hip_ok(hipMemcpy(tables_, host.data(), bytes, hipMemcpyHostToDevice),
                "line FFT table upload"))
        return false;
    dev_ax_ = (LineFftAxis *)tables_;
    for (int a = 0; a < dim; ++a) tw_[a] = (char *)tables_ + at[a];
    return true;
}

namespace {

struct JobChunk {
    static constexpr int N = (int)((4096 - 64) / sizeof(LineFftJob));
    LineFftJob j[N];
    int n;
};

__global__ void k_line_jobs(JobChunk chunk, LineFftJob *dst)
{
    for (int i = threadIdx.x; i < chunk.n; i += blockDim.x) dst[i] = chunk.j[i];
}

}  // namespace

bool LineFft::run_many(const std::vector<const LineFft *> &ffts, const std::vector<void *> &grids,
                       LineFftJob **jobs, int64_t *cap, hipStream_t stream)
{
    static_assert(JobChunk::N >= 1 && sizeof(JobChunk) <= 4096, "job chunk");
    if (ffts.empty()) return true;
    const int naxes = ffts[0]->naxes_;
    const bool f64 = ffts[0]->f64_;
    for (const LineFft *f : ffts)
        if (f->naxes_ != naxes || f->f64_ != f64) {
            set_error("batched line FFT: plans of one rank and precision");
            return false;
        }
    // jobs grouped by axis, each group's workgroups numbered from 0
    struct Launch {
        size_t first, count;
        int64_t groups;
        size_t lds;
        int threads;
    };
    std::vector<LineFftJob> all;
    std::vector<Launch> launches;
    for (int a = 0; a < naxes; ++a) {
        Launch L{all.size(), 0, 0, 0, 64};
        for (size_t i = 0; i < ffts.size(); ++i) {
            const LineFft &f = *ffts[i];
            const LineFftAxis &x = f.ax_[a];
            const int64_t g = (x.nu * x.nv + x.lines - 1) / x.lines;
            if (g == 0) continue;
            all.push_back(LineFftJob{f.dev_ax_ + a, grids[i], f.tw_[a], L.groups});
            L.groups += g;
            L.threads = std::max(L.threads, x.threads);
            L.lds = std::max(L.lds, (size_t)(x.lines + 1) * (size_t)x.n * (f64 ? 16 : 8));
        }
        L.count = all.size() - L.first;
        if (L.count) launches.push_back(L);
    }
    const int64_t n = (int64_t)all.size();
    if (n > *cap) {
        if (*jobs) (void)hipFree(*jobs);
        *jobs = nullptr;
        *cap = 0;
        if (!hip_ok(hipMalloc(jobs, sizeof(LineFftJob) * n), "line FFT job table")) return false;
        *cap = n;
    }
    for (int64_t i0 = 0; i0 < n; i0 += JobChunk::N) {
        JobChunk chunk;
        chunk.n = (int)std::min<int64_t>(JobChunk::N, n - i0);
        for (int k = 0; k < chunk.n; ++k) chunk.j[k] = all[(size_t)(i0 + k)];
        k_line_jobs<<<1, 64, 0, stream>>>(chunk, *jobs + i0);
    }
    for (const Launch &L : launches) {
        if (L.groups > 0x7fffffff) {
            set_error("batched line FFT: too many workgroups");
            return false;
        }
        const dim3 g((unsigned)L.groups);
        const LineFftJob *J = *jobs + L.first;
        if (f64)
            k_fft_lines_many<double><<<g, L.threads, L.lds, stream>>>(J, (int)L.count);
        else
            k_fft_lines_many<float><<<g, L.threads, L.lds, stream>>>(J, (int)L.count);
    }
    return hip_ok(hipGetLastError(), "batched line FFT launch");
}

namespace {

template <typename T>
void launch_axis(int io, dim3 g, int threads, size_t lds, hipStream_t stream, const LineFftAxis *ax, void *mv,
                 T *d, const Cx<T> *t, const uint32_t *rows)
{
    if (io == 1)
        k_fft_lines<T, 1><<<g, threads, lds, stream>>>(ax, mv, d, t, rows);
    else if (io == 2)
        k_fft_lines<T, 2><<<g, threads, lds, stream>>>(ax, mv, d, t, rows);
    else if (io == 3)
        k_fft_lines<T, 3><<<g, threads, lds, stream>>>(ax, mv, d, t, rows);
    else
        k_fft_lines<T, 0><<<g, threads, lds, stream>>>(ax, mv, d, t, rows);
}

}  // namespace

bool LineFft::run(void *data, int64_t vectors, hipStream_t stream, void *modes,
                  const uint32_t *rows) const
{
    if (vectors <= 0) return true;
    const size_t eb = f64_ ? 16 : 8;
    for (int64_t v0 = 0; v0 < vectors; v0 += 65535) {
        const unsigned vc = (unsigned)std::min<int64_t>(65535, vectors - v0);
        for (int a = 0; a < naxes_; ++a) {
            const LineFftAxis &x = ax_[a];
            const bool io = modes && a == (type_ == 2 ? 0 : naxes_ - 1);
            const int mode_io = io ? (type_ == 2 ? 1 : 2) : (rows && a == 2 ? 3 : 0);
            void *mv = io ? (void *)((char *)modes + (size_t)v0 * (size_t)x.mode_total * eb)
                          : nullptr;
            const int64_t groups = (x.nu * x.nv + x.lines - 1) / x.lines;
            if (groups == 0) continue;
            const dim3 g((unsigned)groups, vc);
            const size_t lds = (size_t)(x.lines + 1) * (size_t)x.n * eb;
            const LineFftAxis *hx = dev_ax_ + a;
            if (f64_) {
                double *d = (double *)data + 2 * v0 * fine_total_;
                launch_axis<double>(mode_io, g, x.threads, lds, stream, hx, mv, d,
                                    (const Cx<double> *)tw_[a], rows);
            } else {
                float *d = (float *)data + 2 * v0 * fine_total_;
                launch_axis<float>(mode_io, g, x.threads, lds, stream, hx, mv, d,
                                   (const Cx<float> *)tw_[a], rows);
            }
        }
    }
    return hip_ok(hipGetLastError(), "line FFT launch");
}

}  // namespace mnufft
