// Transforms of a few points in registers and the in-place mixed-radix stages in LDS
// that the far field's FFT kernels are built from.
//
// A length N = f0 f1 .. is transformed by decimation in frequency: stage s takes
// blocks of Ls = N / (f0 .. f_{s-1}) elements, does an f_s-point transform over n1 for
// every n2 (element n1 ms + n2, ms = Ls / f_s), multiplies mode k1 by W_Ls^(n2 k1) and
// leaves it at k1 ms + n2, where the next stage finds its own blocks.  Every task reads
// and writes the same f_s places, so a stage needs one barrier and no second buffer;
// the modes end up in digit-reversed places (FftAxis::loc), and the inverse runs the
// same stages backwards from there with conjugate factors (unnormalised).
#pragma once
#include <hip/hip_runtime.h>

constexpr int FFT_MAXSTAGE = 4;

// factors of one axis and its device tables: tw[j] = exp(-2 pi i j / n), loc[k] = place of mode k
struct FftAxis {
    int n = 0, ns = 0;
    int f[FFT_MAXSTAGE] = {0, 0, 0, 0};
    const float2 *tw = nullptr;
    const unsigned short *loc = nullptr;
};

namespace fft {
// radices of fft::transform, and the fewest of them whose product is n (of those the split with
// the smallest largest radix): a stage costs a pass over LDS and a barrier
inline bool split_radices(int n, int depth, int *f)
{
    static const int radix[] = {16, 15, 12, 10, 9, 8, 6, 5, 4, 3, 2};
    if (depth == 1) {
        for (int r : radix)
            if (r == n) { f[0] = n; return true; }
        return false;
    }
    int best = 1 << 30;
    bool found = false;
    for (int r : radix) {
        int rest[FFT_MAXSTAGE];
        if (n % r || !split_radices(n / r, depth - 1, rest)) continue;
        int top = r;
        for (int k = 0; k + 1 < depth; ++k) top = rest[k] > top ? rest[k] : top;
        // an odd last radix (the stride of the last stage's lanes) avoids LDS bank conflicts
        const int cost = 4 * top + (rest[depth - 2] % 2 ? 0 : 1);
        if (cost < best) {
            best = cost;
            found = true;
            f[0] = r;
            for (int k = 0; k + 1 < depth; ++k) f[k + 1] = rest[k];
        }
    }
    return found;
}

inline bool split(int n, int *ns, int *f)
{
    for (int d = 1; d <= FFT_MAXSTAGE; ++d)
        if (split_radices(n, d, f)) { *ns = d; return true; }
    return false;
}

// place of mode k: digits k = k0 + f0 (k1 + f1 (k2 ..)), place = k0 n / f0 + k1 n / (f0 f1) + ..
inline int place_of(int n, int ns, const int *f, int k)
{
    int p = 0;
    for (int s = 0; s < ns; ++s) {
        n /= f[s];
        p += k % f[s] * n;
        k /= f[s];
    }
    return p;
}

// cos and sin of 2 pi k / n at compile time, by the Taylor series about 0 on [-pi, pi]
constexpr double turn_angle(int k, int n)
{
    k %= n;
    return 6.283185307179586476925 * (2 * k > n ? k - n : k) / n;
}
constexpr double series(double x, int first)
{
    double term = first ? x : 1.0, sum = term;
    for (int q = first + 1; q < 60; q += 2) {
        term *= -x * x / ((double)q * (q + 1));
        sum += term;
    }
    return sum;
}
template <int N>
struct Roots {
    float c[N], s[N];   // cos and -sin: W^k = c[k] + i s[k]
    constexpr Roots() : c(), s()
    {
        for (int k = 0; k < N; ++k) {
            c[k] = (float)series(turn_angle(k, N), 0);
            s[k] = (float)-series(turn_angle(k, N), 1);
        }
    }
};

__device__ __forceinline__ float2 add(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 sub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
template <bool INV>
__device__ __forceinline__ float2 mul_i(float2 v)   // v * (INV ? i : -i)
{
    return INV ? make_float2(-v.y, v.x) : make_float2(v.y, -v.x);
}
template <bool INV>
__device__ __forceinline__ float2 mul_w(float2 a, float2 w)   // a * w, or a * conj(w)
{
    return INV ? make_float2(a.x * w.x + a.y * w.y, a.y * w.x - a.x * w.y)
               : make_float2(a.x * w.x - a.y * w.y, a.x * w.y + a.y * w.x);
}

template <int R, bool INV>
struct Dft;   // run(x): x[k] <- sum_n x[n] W_R^(+-n k)

template <bool INV>
struct Dft<2, INV> {
    static __device__ __forceinline__ void run(float2 *x)
    {
        const float2 a = x[0];
        x[0] = add(a, x[1]);
        x[1] = sub(a, x[1]);
    }
};
template <bool INV>
struct Dft<3, INV> {
    static __device__ __forceinline__ void run(float2 *x)
    {
        constexpr float H = 0.86602540378443865f;   // sqrt(3) / 2
        const float2 s = add(x[1], x[2]), d = sub(x[1], x[2]);
        const float2 t = mul_i<INV>(make_float2(H * d.x, H * d.y));
        const float2 m = make_float2(x[0].x - 0.5f * s.x, x[0].y - 0.5f * s.y);
        x[0] = add(x[0], s);
        x[1] = add(m, t);
        x[2] = sub(m, t);
    }
};
template <bool INV>
struct Dft<4, INV> {
    static __device__ __forceinline__ void run(float2 *x)
    {
        const float2 t0 = add(x[0], x[2]), t1 = sub(x[0], x[2]), t2 = add(x[1], x[3]);
        const float2 t3 = mul_i<INV>(sub(x[1], x[3]));
        x[0] = add(t0, t2);
        x[2] = sub(t0, t2);
        x[1] = add(t1, t3);
        x[3] = sub(t1, t3);
    }
};
template <bool INV>
struct Dft<5, INV> {
    static __device__ __forceinline__ void run(float2 *x)
    {
        constexpr Roots<5> w;
        constexpr float c1 = w.c[1], c2 = w.c[2], s1 = -w.s[1], s2 = -w.s[2];
        const float2 p1 = add(x[1], x[4]), p2 = add(x[2], x[3]), m1 = sub(x[1], x[4]), m2 = sub(x[2], x[3]);
        const float2 a = make_float2(x[0].x + c1 * p1.x + c2 * p2.x, x[0].y + c1 * p1.y + c2 * p2.y);
        const float2 b = make_float2(x[0].x + c2 * p1.x + c1 * p2.x, x[0].y + c2 * p1.y + c1 * p2.y);
        const float2 d = mul_i<INV>(make_float2(s1 * m1.x + s2 * m2.x, s1 * m1.y + s2 * m2.y));
        const float2 e = mul_i<INV>(make_float2(s2 * m1.x - s1 * m2.x, s2 * m1.y - s1 * m2.y));
        x[0] = add(x[0], add(p1, p2));
        x[1] = add(a, d);
        x[4] = sub(a, d);
        x[2] = add(b, e);
        x[3] = sub(b, e);
    }
};
// A B points: n = B n1 + n2, k = k1 + A k2
template <int A, int B, bool INV>
struct DftProduct {
    static __device__ __forceinline__ void run(float2 *x)
    {
        constexpr Roots<A * B> w;
        float2 u[A][B];
#pragma unroll
        for (int n2 = 0; n2 < B; ++n2) {
            float2 t[A];
#pragma unroll
            for (int n1 = 0; n1 < A; ++n1) t[n1] = x[B * n1 + n2];
            Dft<A, INV>::run(t);
#pragma unroll
            for (int k1 = 0; k1 < A; ++k1)
                u[k1][n2] = n2 * k1 ? mul_w<INV>(t[k1], make_float2(w.c[n2 * k1], w.s[n2 * k1])) : t[k1];
        }
#pragma unroll
        for (int k1 = 0; k1 < A; ++k1) {
            Dft<B, INV>::run(u[k1]);
#pragma unroll
            for (int k2 = 0; k2 < B; ++k2) x[k1 + A * k2] = u[k1][k2];
        }
    }
};
template <bool INV> struct Dft<6, INV> : DftProduct<2, 3, INV> {};
template <bool INV> struct Dft<8, INV> : DftProduct<2, 4, INV> {};
template <bool INV> struct Dft<9, INV> : DftProduct<3, 3, INV> {};
template <bool INV> struct Dft<10, INV> : DftProduct<2, 5, INV> {};
template <bool INV> struct Dft<12, INV> : DftProduct<3, 4, INV> {};
template <bool INV> struct Dft<15, INV> : DftProduct<3, 5, INV> {};
template <bool INV> struct Dft<16, INV> : DftProduct<4, 4, INV> {};

// exact quotients of small non-negative integers (a < 2^20, d < 2^12) by a float reciprocal
struct FastDiv {
    float inv;
    int d;
    __device__ __forceinline__ explicit FastDiv(int d_) : inv(1.0f / (float)d_), d(d_) {}
    __device__ __forceinline__ int operator()(int a, int &rem) const
    {
        const int q = (int)(((float)a + 0.5f) * inv);
        rem = a - q * d;
        return q;
    }
};

// One stage of radix R on nseq sequences in buf.  place(idx, t): first element of the sequence
// that task idx belongs to and its number t inside the sequence (t < n / R); stride between
// consecutive elements.  tw: the axis' table (in LDS).
template <int R, bool INV, int NT, class Place>
__device__ __forceinline__ void stage_r(float2 *buf, int total, Place place, int stride, int ms, int step,
                                        const float2 *tw)
{
    const FastDiv by_ms(ms);
    const int st = ms * stride;
    for (int idx = threadIdx.x; idx < total; idx += NT) {
        int t, n2;
        float2 *p = buf + place(idx, t);
        const int b = by_ms(t, n2);
        p += (b * ms * R + n2) * stride;
        float2 x[R];
#pragma unroll
        for (int q = 0; q < R; ++q) x[q] = p[q * st];
        if (INV && ms > 1) {
#pragma unroll
            for (int q = 1; q < R; ++q) x[q] = mul_w<true>(x[q], tw[n2 * q * step]);
        }
        Dft<R, INV>::run(x);
        if (!INV && ms > 1) {
#pragma unroll
            for (int q = 1; q < R; ++q) x[q] = mul_w<false>(x[q], tw[n2 * q * step]);
        }
#pragma unroll
        for (int q = 0; q < R; ++q) p[q * st] = x[q];
    }
}

// all stages of an axis over nseq sequences, a barrier after each; place(f): the task map of a
// stage whose sequences have n / f tasks
template <bool INV, int NT, class MakePlace>
__device__ __forceinline__ void transform(float2 *buf, const FftAxis &ax, int nseq, MakePlace make, int stride,
                                          const float2 *tw)
{
    int L = INV ? 1 : ax.n;    // forward: block length of the stage; inverse: of the stage before
    for (int q = 0; q < ax.ns; ++q) {
        const int f = ax.f[INV ? ax.ns - 1 - q : q];
        const int Ls = INV ? L * f : L, ms = Ls / f, step = ax.n / Ls, total = nseq * (ax.n / f);
        auto place = make(ax.n / f);
        switch (f) {
#define FFT_RADIX(r) case r: stage_r<r, INV, NT>(buf, total, place, stride, ms, step, tw); break;
            FFT_RADIX(2) FFT_RADIX(3) FFT_RADIX(4) FFT_RADIX(5) FFT_RADIX(6) FFT_RADIX(8) FFT_RADIX(9)
            FFT_RADIX(10) FFT_RADIX(12) FFT_RADIX(15) FFT_RADIX(16)
#undef FFT_RADIX
            default: break;
        }
        L = INV ? Ls : ms;
        __syncthreads();
    }
}
}  // namespace fft
