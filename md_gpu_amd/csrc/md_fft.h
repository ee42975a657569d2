// md_fft.h -- short discrete Fourier transforms in registers and the Stockham passes
// that build longer ones, for the transforms of smooth PME (pme_fft.hip).
//
// A length N = r_0 r_1 ... is done in one pass per factor (Stockham's self-sorting
// form): pass with radix R after factors of product Ns reads, for butterfly j in
// [0, N / R), the elements j + q N / R (q < R), multiplies element q by
// w_N^(k q N / (Ns R)), k = j mod Ns, transforms them by a DFT of length R and writes
// them to (j / Ns) Ns R + k + q Ns.  Input and output lie in different buffers, so one
// barrier separates two passes.  The inverse transform is the forward one with real and
// imaginary parts swapped on the way in and out.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define MD_FFT_MAXPASS 6

namespace fft {

// quotients by a fixed divisor: exact for a d < 2^32 (m = ceil(2^32 / d); d = 1 apart)
struct Div {
    uint32_t m;
    int d;
    Div() = default;
    __host__ __device__ explicit Div(int d_) : m(d_ > 1 ? 0xFFFFFFFFu / (uint32_t)d_ + 1u : 0u), d(d_) {}
    __host__ __device__ __forceinline__ int quot(int a) const {
        return d == 1 ? a : (int)(((uint64_t)(uint32_t)a * m) >> 32);
    }
};

}  // namespace fft

// Plan of one axis: the passes in order, each with its factor and the product of the
// factors before it (npass = 0: the length is not supported).
struct FftPlan {
    int n, npass;
    struct { int radix, step; fft::Div ns; } pass[MD_FFT_MAXPASS];   // step = n / (ns radix)
};

namespace fft {

constexpr double kPi = 3.14159265358979323846;

// cos and sin of 2 pi k / n by their series (|x| <= pi / 4 after folding the octants)
constexpr double ser_cos(double x) {
    double t = 1.0, s = 1.0;
    for (int i = 1; i < 12; i++) {
        t *= -x * x / ((2 * i - 1) * (2 * i));
        s += t;
    }
    return s;
}
constexpr double ser_sin(double x) {
    double t = x, s = x;
    for (int i = 1; i < 12; i++) {
        t *= -x * x / ((2 * i) * (2 * i + 1));
        s += t;
    }
    return s;
}
constexpr double turn_cos(int k, int n);
constexpr double turn_sin(int k, int n) {   // sin(2 pi k / n), 0 <= k < n
    if (2 * k > n) return -turn_sin(n - k, n);
    if (4 * k > n) return turn_sin(n - 2 * k, 2 * n);        // sin(pi - x)
    if (8 * k > n) return turn_cos(n - 4 * k, 4 * n);        // cos(pi / 2 - x)
    return ser_sin(2.0 * kPi * k / n);
}
constexpr double turn_cos(int k, int n) {
    if (2 * k > n) return turn_cos(n - k, n);
    if (4 * k > n) return -turn_cos(n - 2 * k, 2 * n);
    if (8 * k > n) return turn_sin(n - 4 * k, 4 * n);
    return ser_cos(2.0 * kPi * k / n);
}

template <int N>
struct Turns {   // w_N^k = c[k] - i s[k]
    double c[N], s[N];
    constexpr Turns() : c(), s() {
        for (int k = 0; k < N; k++) {
            c[k] = turn_cos(k, N);
            s[k] = turn_sin(k, N);
        }
    }
};
template <int N>
static constexpr Turns<N> turns{};

// complex numbers of the butterflies: T = double (the passes' arithmetic) between values
// stored as float2
template <class T>
struct Cx {
    T x, y;
};
__host__ __device__ __forceinline__ float fma_(float a, float b, float c) { return fmaf(a, b, c); }
__host__ __device__ __forceinline__ double fma_(double a, double b, double c) { return fma(a, b, c); }
template <class T>
__host__ __device__ __forceinline__ Cx<T> add(Cx<T> a, Cx<T> b) { return {a.x + b.x, a.y + b.y}; }
template <class T>
__host__ __device__ __forceinline__ Cx<T> sub(Cx<T> a, Cx<T> b) { return {a.x - b.x, a.y - b.y}; }
// a (c - i s)
template <class T>
__host__ __device__ __forceinline__ Cx<T> mulw(Cx<T> a, T c, T s) { return {fma_(a.x, c, a.y * s), fma_(a.y, c, -(a.x * s))}; }
// a w_N^k, k a constant once unrolled: quarter turns without multiplications
template <int N, class T>
__host__ __device__ __forceinline__ Cx<T> turn(Cx<T> a, int k) {
    k %= N;
    if (k == 0) return a;
    if (4 * k == N) return {a.y, -a.x};
    if (2 * k == N) return {-a.x, -a.y};
    if (4 * k == 3 * N) return {-a.y, a.x};
    return mulw(a, (T)turns<N>.c[k], (T)turns<N>.s[k]);
}

template <int R, class T>
struct Dft;
template <class T>
struct Dft<2, T> {
    static __host__ __device__ __forceinline__ void go(Cx<T>* v) {
        const Cx<T> a = add(v[0], v[1]), b = sub(v[0], v[1]);
        v[0] = a;
        v[1] = b;
    }
};
template <class T>
struct Dft<3, T> {
    static __host__ __device__ __forceinline__ void go(Cx<T>* v) {
        const T s3 = (T)0.86602540378443864676, h = (T)0.5;
        const Cx<T> p = add(v[1], v[2]), m = sub(v[1], v[2]);
        const Cx<T> a = {fma_(-h, p.x, v[0].x), fma_(-h, p.y, v[0].y)};
        v[0] = add(v[0], p);
        v[1] = {fma_(s3, m.y, a.x), fma_(-s3, m.x, a.y)};
        v[2] = {fma_(-s3, m.y, a.x), fma_(s3, m.x, a.y)};
    }
};
template <class T>
struct Dft<4, T> {
    static __host__ __device__ __forceinline__ void go(Cx<T>* v) {
        const Cx<T> a = add(v[0], v[2]), b = sub(v[0], v[2]), c = add(v[1], v[3]), d = sub(v[1], v[3]);
        v[0] = add(a, c);
        v[2] = sub(a, c);
        v[1] = {b.x + d.y, b.y - d.x};
        v[3] = {b.x - d.y, b.y + d.x};
    }
};
template <class T>
struct Dft<5, T> {
    static __host__ __device__ __forceinline__ void go(Cx<T>* v) {
        const T c1 = (T)turns<5>.c[1], c2 = (T)turns<5>.c[2], s1 = (T)turns<5>.s[1], s2 = (T)turns<5>.s[2];
        const Cx<T> p1 = add(v[1], v[4]), m1 = sub(v[1], v[4]), p2 = add(v[2], v[3]), m2 = sub(v[2], v[3]);
        const Cx<T> a = {fma_(c2, p2.x, fma_(c1, p1.x, v[0].x)), fma_(c2, p2.y, fma_(c1, p1.y, v[0].y))};
        const Cx<T> b = {fma_(c1, p2.x, fma_(c2, p1.x, v[0].x)), fma_(c1, p2.y, fma_(c2, p1.y, v[0].y))};
        const Cx<T> s = {fma_(s2, m2.x, s1 * m1.x), fma_(s2, m2.y, s1 * m1.y)};
        const Cx<T> t = {fma_(-s1, m2.x, s2 * m1.x), fma_(-s1, m2.y, s2 * m1.y)};
        v[0] = add(v[0], add(p1, p2));
        v[1] = {a.x + s.y, a.y - s.x};
        v[4] = {a.x - s.y, a.y + s.x};
        v[2] = {b.x + t.y, b.y - t.x};
        v[3] = {b.x - t.y, b.y + t.x};
    }
};
// N = A B: columns of length A, turns, rows of length B
template <int A, int B, class T>
struct DftAB {
    static __host__ __device__ __forceinline__ void go(Cx<T>* v) {
        Cx<T> u[A * B];
#pragma unroll
        for (int n = 0; n < B; n++) {
            Cx<T> t[A];
#pragma unroll
            for (int k = 0; k < A; k++) t[k] = v[B * k + n];
            Dft<A, T>::go(t);
#pragma unroll
            for (int k = 0; k < A; k++) u[B * k + n] = turn<A * B>(t[k], n * k);
        }
#pragma unroll
        for (int k = 0; k < A; k++) {
            Dft<B, T>::go(u + B * k);
#pragma unroll
            for (int q = 0; q < B; q++) v[k + A * q] = u[B * k + q];
        }
    }
};
template <class T> struct Dft<6, T> : DftAB<2, 3, T> {};
template <class T> struct Dft<8, T> : DftAB<2, 4, T> {};
template <class T> struct Dft<9, T> : DftAB<3, 3, T> {};
template <class T> struct Dft<10, T> : DftAB<2, 5, T> {};
template <class T> struct Dft<12, T> : DftAB<4, 3, T> {};
template <class T> struct Dft<16, T> : DftAB<4, 4, T> {};

// a * b for values below 2^23 (one full-rate instruction on the device)
__host__ __device__ __forceinline__ int mul24(int a, int b) {
#ifdef __HIP_DEVICE_COMPILE__
    return __mul24(a, b);
#else
    return a * b;
#endif
}

// One pass of radix R over `lines` transforms of length n by nth threads: thread items
// run over the lines fastest.  ld(line, j, s) reads element j + s of a line, st(line, o, s,
// v) writes element o + s; s is the same for every thread, so the offsets of a butterfly's
// elements are scalar.  step = n / (Ns R); tw holds (cos, sin)(2 pi k / n).
template <int R, class T, class LD, class ST>
__host__ __device__ __forceinline__ void pass(int nb, const Div& ds, int step, const Div& dl, const Cx<T>* tw, int tid, int nth, LD&& ld, ST&& st) {
    const int Ns = ds.d, lines = dl.d, total = nb * lines;
    for (int u = tid; u < total; u += nth) {
        const int j = dl.quot(u), line = u - mul24(j, lines);
        const int jn = ds.quot(j), k = j - mul24(jn, Ns);
        Cx<T> v[R];
#pragma unroll
        for (int q = 0; q < R; q++) {
            const float2 x = ld(line, j, q * nb);
            v[q] = {(T)x.x, (T)x.y};
        }
        if (Ns > 1) {
            const int t = mul24(k, step);
#pragma unroll
            for (int q = 1; q < R; q++) {
                const Cx<T> w = tw[mul24(t, q)];
                v[q] = mulw(v[q], w.x, w.y);
            }
        }
        Dft<R, T>::go(v);
        const int o = mul24(jn, Ns * R) + k;
#pragma unroll
        for (int q = 0; q < R; q++) st(line, o, q * Ns, make_float2((float)v[q].x, (float)v[q].y));
    }
}
// pass q of plan p over dl.d lines
template <class T, class LD, class ST>
__host__ __device__ __forceinline__ void pass_any(const FftPlan& p, int q, const Div& dl, const Cx<T>* tw, int tid, int nth, LD&& ld, ST&& st) {
    const int R = p.pass[q].radix;
    const Div ds = p.pass[q].ns;
    const int step = p.pass[q].step, nb = step * ds.d;   // n / (Ns R), n / R
    switch (R) {
    case 2: pass<2, T>(nb, ds, step, dl, tw, tid, nth, ld, st); break;
    case 3: pass<3, T>(nb, ds, step, dl, tw, tid, nth, ld, st); break;
    case 4: pass<4, T>(nb, ds, step, dl, tw, tid, nth, ld, st); break;
    case 5: pass<5, T>(nb, ds, step, dl, tw, tid, nth, ld, st); break;
    case 6: pass<6, T>(nb, ds, step, dl, tw, tid, nth, ld, st); break;
    case 8: pass<8, T>(nb, ds, step, dl, tw, tid, nth, ld, st); break;
    case 9: pass<9, T>(nb, ds, step, dl, tw, tid, nth, ld, st); break;
    case 10: pass<10, T>(nb, ds, step, dl, tw, tid, nth, ld, st); break;
    case 12: pass<12, T>(nb, ds, step, dl, tw, tid, nth, ld, st); break;
    default: pass<16, T>(nb, ds, step, dl, tw, tid, nth, ld, st); break;
    }
}

// Factors of n among the radices above, the fewest passes first and then the smallest
// largest factor (npass = 0 when n has another prime factor or needs too many passes).
inline FftPlan plan(int n) {
    static const int rs[] = {16, 12, 10, 9, 8, 6, 5, 4, 3, 2};
    FftPlan best{};
    best.n = n;
    int cur[MD_FFT_MAXPASS], bestmax = 1 << 30;
    struct Rec {
        static void go(int m, int depth, int from, int mx, int* cur, FftPlan& best, int& bestmax) {
            if (m == 1) {
                if (depth && (best.npass == 0 || depth < best.npass || (depth == best.npass && mx < bestmax))) {
                    best.npass = depth;
                    bestmax = mx;
                    int ns = 1;
                    for (int i = 0; i < depth; i++) {
                        best.pass[i].radix = cur[i];
                        best.pass[i].ns = Div(ns);
                        ns *= cur[i];
                        best.pass[i].step = best.n / ns;
                    }
                }
                return;
            }
            if (depth == MD_FFT_MAXPASS) return;
            for (int i = from; i < 10; i++)
                if (m % rs[i] == 0) {
                    cur[depth] = rs[i];
                    go(m / rs[i], depth + 1, i, mx > rs[i] ? mx : rs[i], cur, best, bestmax);
                }
        }
    };
    Rec::go(n, 0, 0, 0, cur, best, bestmax);
    return best;
}

}  // namespace fft
