// Saddle-point operator pieces, GMRES vector kernels (FP64 accumulation),
// right-hand-side assembly and the explicit Euler step with shear.
#include "fsd_internal.h"

#include <algorithm>

// ------------------------------------------------------------ vectors
__global__ void axpby_kernel(int64_t n, float a, const float *x, float b, const float *y, float *z)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) z[i] = a * x[i] + (y ? b * y[i] : 0.f);
}

int k_axpby(fsd_ctx *ctx, int64_t n, float a, const float *x, float b, const float *y, float *z)
{
    hipLaunchKernelGGL(axpby_kernel, dim3(nblk(n, 256)), dim3(256), 0, ctx->stream, n, a, x, b, y, z);
    FSD_HIP(hipGetLastError());
    return 0;
}

__global__ void copy_kernel(int64_t n, const float *x, float *y)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) y[i] = x[i];
}

int k_copy(fsd_ctx *ctx, int64_t n, const float *x, float *y)
{
    hipLaunchKernelGGL(copy_kernel, dim3(nblk(n, 256)), dim3(256), 0, ctx->stream, n, x, y);
    FSD_HIP(hipGetLastError());
    return 0;
}

__global__ void fill_kernel(int64_t n, float v, float *y)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) y[i] = v;
}

int k_fill(fsd_ctx *ctx, int64_t n, float v, float *y)
{
    hipLaunchKernelGGL(fill_kernel, dim3(nblk(n, 256)), dim3(256), 0, ctx->stream, n, v, y);
    FSD_HIP(hipGetLastError());
    return 0;
}

// ---------------------------------------------- Gram-Schmidt, norms, combinations
// The orthogonalisation of GMRES and Lanczos: two classical passes of h = V^T w, w -= V h, then
// v = w / |w|; FP64 sums of FP32 vectors.  The host never waits inside; what it needs (h, |w|) block 0
// writes to pinned memory.
//
// Short vectors (n up to GS_FUSED) are bound by launches and by the latency of a block's loads: four
// launches, in each of which every block first sums the partials of the launch before (in the same
// order in every block), and where a chunk of w stays in registers between w -= V h1 and its part of
// h2 = V^T w.  Long vectors are bound by reading V, and the partials that every block would read are
// no longer small against that: the sums get a launch of their own, and the products a block per vector
// and four chunks (17 us for a mean of 40 vectors at n = 557056; 25 us with eight vectors to a block, at
// one, two or four chunks).
//   short: dots | sum, axpy, dots | sum, axpy, norm | sum, scale
//   long:  dots | sum | axpy | dots | sum | axpy, norm | sum, scale
// In the short form's second launch a block goes through all K vectors twice, so with two passes it is the
// shorter one up to about 20 vectors only, 32 below 65536 numbers (the near-field square root of a Brownian
// step at N = 1000, some 40 steps of 6000 numbers: 813 us a call at 20, 790 at 32).  Mean over K = 1 .. R of both
// forms, us:
//   two passes      n = 17000     42500     102000    130900    204000    557056
//     R = 16           20 25     21 26      24 27     23 26     25 28     33 35
//     R = 32           24 26     26 27      29 30     27 29     33 33     50 47
//     R = 64           30 29     34 30      43 35     38 35     49 45     84 68
//   one pass
//     R = 64           16 18     19 19      21 21     20 21     24 26     45 38
//     R = 100          19 20     23 22      26 26     25 25     31 31     62 51
// The short products and the updates read the vectors eight at a time, and the eight sums over a wave's
// lanes share one butterfly (10 exchanges, 48 one by one).
#define GS_NT 256
#define GS_CH (4 * GS_NT)     // numbers of a block, four to a thread
#define GS_KMAX 256
#define GS_FUSED (1 << 17)
#define GS_LONG 4             // chunks of a block of the long products

static int gs_fused_k(int64_t n) { return n > (1 << 16) ? 20 : 32; }     // with two passes

static int gs_chunks(int64_t n) { return (int)((n + GS_CH - 1) / GS_CH); }
static int gs_dot_blocks(int64_t n, bool lng) { return lng ? (gs_chunks(n) + GS_LONG - 1) / GS_LONG : gs_chunks(n); }
int64_t gs_part_doubles(int64_t n, int K)      // for every length up to n, in either form
{
    const int64_t blocks = n > GS_FUSED ? std::max(gs_dot_blocks(n, true), GS_FUSED / GS_CH) : gs_chunks(n);
    return std::max(std::min(K, GS_KMAX) * blocks, (int64_t)gs_chunks(n));
}

static bool vec4_ok(int64_t n, int64_t ldv, const void *a, const void *b)
{
    return n % 4 == 0 && ldv % 4 == 0 && ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b)) & 15) == 0;
}

// this thread's four numbers of chunk c (VEC: 16-byte accesses), zero past the end
template <bool VEC>
__device__ __forceinline__ void gs_load(const float *p, int64_t n, int c, float (&x)[4])
{
    if (VEC) {
        const int64_t q = (int64_t)c * GS_NT + threadIdx.x;
        const float4 v = q < n / 4 ? reinterpret_cast<const float4 *>(p)[q] : make_float4(0.f, 0.f, 0.f, 0.f);
        x[0] = v.x; x[1] = v.y; x[2] = v.z; x[3] = v.w;
    } else {
        const int64_t q = (int64_t)c * GS_CH + threadIdx.x;
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = q + GS_NT * e < n ? p[q + GS_NT * e] : 0.f;
    }
}

template <bool VEC>
__device__ __forceinline__ void gs_store(float *p, int64_t n, int c, const float (&x)[4])
{
    if (VEC) {
        const int64_t q = (int64_t)c * GS_NT + threadIdx.x;
        if (q < n / 4) reinterpret_cast<float4 *>(p)[q] = make_float4(x[0], x[1], x[2], x[3]);
    } else {
        const int64_t q = (int64_t)c * GS_CH + threadIdx.x;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (q + GS_NT * e < n) p[q + GS_NT * e] = x[e];
    }
}

// x -= sum_k h[k] V_k on chunk c
template <bool VEC>
__device__ __forceinline__ void gs_update(const float *V, int64_t n, int c, int K, const float *h, float (&x)[4])
{
    for (int k0 = 0; k0 < K; k0 += 8) {
        float v[8][4];
#pragma unroll
        for (int k = 0; k < 8; ++k) gs_load<VEC>(V + (int64_t)min(k0 + k, K - 1) * n, n, c, v[k]);
#pragma unroll
        for (int k = 0; k < 8; ++k)
            if (k0 + k < K) {
                const float a = h[k0 + k];
#pragma unroll
                for (int e = 0; e < 4; ++e) x[e] -= a * v[k][e];
            }
    }
}

// p[k] += <V_{k0 + k}, x> on chunk c, k < 8
template <bool VEC>
__device__ __forceinline__ void gs_dots8(const float *V, int64_t n, int c, int K, int k0, const float (&x)[4],
                                         double (&p)[8])
{
    float v[8][4];
#pragma unroll
    for (int k = 0; k < 8; ++k) gs_load<VEC>(V + (int64_t)min(k0 + k, K - 1) * n, n, c, v[k]);
#pragma unroll
    for (int k = 0; k < 8; ++k)
        p[k] += (double)v[k][0] * (double)x[0] + (double)v[k][1] * (double)x[1] + (double)v[k][2] * (double)x[2] +
                (double)v[k][3] * (double)x[3];
}

// the eight sums over the wave: returns sum gs_mine(lane)
__device__ __forceinline__ int gs_mine(int lane) { return (lane >> 5 & 1) * 4 + (lane >> 4 & 1) * 2 + (lane >> 3 & 1); }
__device__ __forceinline__ double gs_butterfly(double (&p)[8], int lane)
{
    // halves of the eight go to either half of the lanes, three times
#pragma unroll
    for (int m = 4, o = 32; m >= 1; m >>= 1, o >>= 1) {
        const bool up = lane & o;
#pragma unroll
        for (int k = 0; k < m; ++k) {
            const double keep = up ? p[k + m] : p[k], give = up ? p[k] : p[k + m];
            p[k] = keep + __shfl_xor(give, o, 64);
        }
    }
    double s = p[0];
    for (int o = 4; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    return s;
}

// sum over the block (one value for every thread)
__device__ __forceinline__ double block_sum(double s, double (&red)[GS_NT / 64])
{
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    return red[0] + red[1] + red[2] + red[3];
}

// partials of V^T w, short vectors: block (c, g) takes the vectors 8 g .. 8 g + 7 on chunk c
template <bool VEC>
__global__ void __launch_bounds__(GS_NT) gs_dots_kernel(int64_t n, int K, const float *V, const float *w, double *out)
{
    __shared__ double s_d[GS_NT / 64][8];
    const int lane = threadIdx.x & 63, k0 = 8 * blockIdx.y;
    double p[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) p[k] = 0.0;
    float x[4];
    gs_load<VEC>(w, n, blockIdx.x, x);
    gs_dots8<VEC>(V, n, blockIdx.x, K, k0, x, p);
    const double s = gs_butterfly(p, lane);
    if ((lane & 7) == 0) s_d[threadIdx.x >> 6][gs_mine(lane)] = s;
    __syncthreads();
    const int k = threadIdx.x;
    if (k < 8 && k0 + k < K)
        out[(int64_t)(k0 + k) * gridDim.x + blockIdx.x] = s_d[0][k] + s_d[1][k] + s_d[2][k] + s_d[3][k];
}

// the same for long vectors: block (b, k) takes vector k on chunks GS_LONG b and on
template <bool VEC>
__global__ void __launch_bounds__(GS_NT) gs_dots_long_kernel(int64_t n, const float *V, const float *w, double *out)
{
    __shared__ double s_red[GS_NT / 64];
    const float *v = V + (int64_t)blockIdx.y * n;
    double s = 0.0;
#pragma unroll
    for (int c = 0; c < GS_LONG; ++c) {
        float a[4], x[4];
        gs_load<VEC>(v, n, GS_LONG * blockIdx.x + c, a);
        gs_load<VEC>(w, n, GS_LONG * blockIdx.x + c, x);
#pragma unroll
        for (int e = 0; e < 4; ++e) s += (double)a[e] * (double)x[e];
    }
    s = block_sum(s, s_red);
    if (threadIdx.x == 0) out[(int64_t)blockIdx.y * gridDim.x + blockIdx.x] = s;
}

// sums of np partials each; sum k (k >= kfirst) also to hout
__global__ void __launch_bounds__(GS_NT) gs_sum_kernel(const double *part, int np, double *out, double *hout, int kfirst)
{
    __shared__ double s_red[GS_NT / 64];
    const int k = blockIdx.x;
    double s = 0.0;
    for (int c = threadIdx.x; c < np; c += GS_NT) s += part[(int64_t)k * np + c];
    s = block_sum(s, s_red);
    if (threadIdx.x == 0) {
        out[k] = s;
        if (hout && k >= kfirst) hout[k - kfirst] = s;
    }
}

// AXPY: w -= V h, h the sums of part (K x np; np = 1: the sums themselves), which block 0 puts into
// hout (may be null) from kfirst on.  out: K x gridDim.x partial dots (DOT) or partial squares (NORM)
template <bool VEC, bool AXPY, bool DOT, bool NORM>
__global__ void __launch_bounds__(GS_NT) gs_kernel(int64_t n, int K, const float *V, float *w, const double *part,
                                                   int np, double *hout, int kfirst, double *out)
{
    __shared__ float s_h[GS_KMAX];
    __shared__ double s_d[GS_NT / 64][GS_KMAX], s_red[GS_NT / 64];
    const int c = blockIdx.x, lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    float x[4];
    gs_load<VEC>(w, n, c, x);
    if (AXPY) {
        // as many lanes per sum as the block has (at most a wave, at least eight), or one where there is nothing
        // to sum
        const int L = np == 1 ? 1 : K <= 4 ? 64 : K <= 8 ? 32 : K <= 16 ? 16 : 8, l = threadIdx.x & (L - 1);
        for (int kb = 0; kb < K; kb += GS_NT / L) {
            const int k = kb + threadIdx.x / L;
            double s = 0.0;
            if (k < K) {
                const double *p = part + (int64_t)k * np;
#pragma unroll 8
                for (int q = l; q < np; q += L) s += p[q];
            }
            for (int o = L >> 1; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
            if (l == 0 && k < K) {
                s_h[k] = (float)s;
                if (hout && c == 0 && k >= kfirst) hout[k - kfirst] = s;
            }
        }
        __syncthreads();
        gs_update<VEC>(V, n, c, K, s_h, x);
        gs_store<VEC>(w, n, c, x);
    }
    if (DOT) {
        for (int k0 = 0; k0 < K; k0 += 8) {
            double p[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) p[k] = 0.0;
            gs_dots8<VEC>(V, n, c, K, k0, x, p);
            const double s = gs_butterfly(p, lane);
            const int k = k0 + gs_mine(lane);
            if ((lane & 7) == 0 && k < K) s_d[wv][k] = s;
        }
        __syncthreads();
        for (int k = threadIdx.x; k < K; k += GS_NT)
            out[(int64_t)k * gridDim.x + c] = s_d[0][k] + s_d[1][k] + s_d[2][k] + s_d[3][k];
    }
    if (NORM) {
        double s = 0.0;
#pragma unroll
        for (int e = 0; e < 4; ++e) s += (double)x[e] * (double)x[e];
        s = block_sum(s, s_red);
        if (threadIdx.x == 0) out[c] = s;
    }
}

// v = w / |w| with |w|^2 the sum of nch partials; block 0 puts |w| into hn
template <bool VEC>
__global__ void __launch_bounds__(GS_NT) gs_scale_kernel(int64_t n, const float *w, float *v, const double *part,
                                                         double *hn)
{
    __shared__ double s_red[GS_NT / 64];
    float x[4];
    gs_load<VEC>(w, n, blockIdx.x, x);
    double s = 0.0;
#pragma unroll 4
    for (int c = threadIdx.x; c < (int)gridDim.x; c += GS_NT) s += part[c];
    const double h = sqrt(block_sum(s, s_red));
    if (hn && blockIdx.x == 0 && threadIdx.x == 0) *hn = h;
    const float inv = h > 0.0 ? (float)(1.0 / h) : 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) x[e] *= inv;
    gs_store<VEC>(v, n, blockIdx.x, x);
}

// out = x0 - sum_k c[k] V_k (x0 may be null); with part also the partials of |prev - out|^2 and |out|^2
struct GsCoef { float c[GS_KMAX]; };
template <bool VEC>
__global__ void __launch_bounds__(GS_NT) gs_combine_kernel(int64_t n, int K, const float *V, GsCoef coef,
                                                           const float *x0, float *out, const float *prev,
                                                           double *part)
{
    __shared__ float s_h[GS_KMAX];
    __shared__ double s_red[GS_NT / 64];
    for (int k = threadIdx.x; k < K; k += GS_NT) s_h[k] = coef.c[k];
    float x[4];
    if (x0) {
        gs_load<VEC>(x0, n, blockIdx.x, x);
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = 0.f;
    }
    __syncthreads();
    gs_update<VEC>(V, n, blockIdx.x, K, s_h, x);
    gs_store<VEC>(out, n, blockIdx.x, x);
    if (part) {
        float y[4];
        gs_load<VEC>(prev, n, blockIdx.x, y);
        double d = 0.0, s = 0.0;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const double t = (double)(y[e] - x[e]);
            d += t * t;
            s += (double)x[e] * (double)x[e];
        }
        d = block_sum(d, s_red);
        s = block_sum(s, s_red);
        if (threadIdx.x == 0) { part[2 * blockIdx.x] = d; part[2 * blockIdx.x + 1] = s; }
    }
}

template <bool AXPY, bool DOT, bool NORM>
static int gs_launch(fsd_ctx *ctx, int64_t n, int K, const float *V, const float *w, const double *part, int np,
                     double *hout, int kfirst, double *out)
{
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(gs_chunks(n)), dim3(GS_NT), 0, ctx->stream, n, K, V, const_cast<float *>(w),
                           part, np, hout, kfirst, out);
    };
    if (vec4_ok(n, n, V ? V : w, w)) go(gs_kernel<true, AXPY, DOT, NORM>);
    else go(gs_kernel<false, AXPY, DOT, NORM>);
    FSD_HIP(hipGetLastError());
    return 0;
}

static int gs_dots(fsd_ctx *ctx, int64_t n, int K, const float *V, const float *w, double *out, bool lng)
{
    const bool vec = vec4_ok(n, n, V, w);
    const dim3 grid(gs_dot_blocks(n, lng), lng ? K : (K + 7) / 8);
    if (lng) {
        auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(GS_NT), 0, ctx->stream, n, V, w, out); };
        vec ? go(gs_dots_long_kernel<true>) : go(gs_dots_long_kernel<false>);
    } else {
        auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(GS_NT), 0, ctx->stream, n, K, V, w, out); };
        vec ? go(gs_dots_kernel<true>) : go(gs_dots_kernel<false>);
    }
    FSD_HIP(hipGetLastError());
    return 0;
}

int k_gs_orthonormalise(fsd_ctx *ctx, int64_t n, int K, const float *V, float *w, int passes, int kfirst, double *h1,
                        double *h2, double *norm)
{
    if (K > GS_KMAX) { ctx->err = "more than 256 vectors to orthogonalise against or to combine"; return FSD_E_PARAM; }
    const bool lng = n > GS_FUSED || (passes == 2 && K > gs_fused_k(n));
    double *a = ctx->d_part[0], *b = ctx->d_part[1];
    int rc = gs_dots(ctx, n, K, V, w, a, lng);
    for (int pass = 1; pass <= passes && !rc; ++pass) {
        double *h = pass == 1 ? h1 : h2;
        const bool last = pass == passes;
        int np = gs_dot_blocks(n, lng);
        if (lng) {
            hipLaunchKernelGGL(gs_sum_kernel, dim3(K), dim3(GS_NT), 0, ctx->stream, a, np, b, h, kfirst);
            std::swap(a, b);
            np = 1;
            h = nullptr;
        }
        if (last) rc = gs_launch<true, false, true>(ctx, n, K, V, w, a, np, h, kfirst, b);
        else if (lng) rc = gs_launch<true, false, false>(ctx, n, K, V, w, a, np, h, kfirst, nullptr);
        else rc = gs_launch<true, true, false>(ctx, n, K, V, w, a, np, h, kfirst, b);
        if (!last && lng && !rc) rc = gs_dots(ctx, n, K, V, w, b, lng);
        std::swap(a, b);
    }
    return rc ? rc : k_gs_scale(ctx, n, w, w, a, norm);
}

int k_gs_norm(fsd_ctx *ctx, int64_t n, const float *w, double *out, int *nch)
{
    if (nch) *nch = gs_chunks(n);
    return gs_launch<false, false, true>(ctx, n, 0, nullptr, w, nullptr, 0, nullptr, 0, out);
}

int k_gs_scale(fsd_ctx *ctx, int64_t n, const float *w, float *v, const double *part, double *hn)
{
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(gs_chunks(n)), dim3(GS_NT), 0, ctx->stream, n, w, v, part, hn);
    };
    const bool vec = vec4_ok(n, n, w, v);
    vec ? go(gs_scale_kernel<true>) : go(gs_scale_kernel<false>);
    FSD_HIP(hipGetLastError());
    return 0;
}

int k_gs_combine(fsd_ctx *ctx, int64_t n, int K, const float *V, const double *c, const float *x0, float *out,
                 const float *prev, double *part, int *nch)
{
    if (K > GS_KMAX) { ctx->err = "more than 256 vectors to orthogonalise against or to combine"; return FSD_E_PARAM; }
    GsCoef coef;
    for (int k = 0; k < GS_KMAX; ++k) coef.c[k] = k < K ? (float)c[k] : 0.f;
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(gs_chunks(n)), dim3(GS_NT), 0, ctx->stream, n, K, V, coef, x0, out, prev, part);
    };
    const bool vec = vec4_ok(n, n, V, out) && vec4_ok(n, n, x0, prev);
    vec ? go(gs_combine_kernel<true>) : go(gs_combine_kernel<false>);
    if (nch) *nch = gs_chunks(n);
    FSD_HIP(hipGetLastError());
    return 0;
}

// ------------------------------------------------------------ saddle
// Saddle_Preconditioner (Saddle.cu:171-264):
//   x_F = b_F - G b_F + G b_U,  x_S = b_S,  x_U = G b_F - G b_U
__global__ void saddle_combine_kernel(int N, const float *b, const float *gF, const float *gU, float *x)
{
    int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t n6 = 6 * (int64_t)N;
    if (q < n6) {
        const float f = gF[q], u = gU[q];
        x[q] = b[q] - f + u;
        x[11 * (int64_t)N + q] = f - u;
    } else if (q < 11 * (int64_t)N) {
        x[q] = b[q];
    }
}

int k_precond_apply2(fsd_ctx *ctx, const float *b0, const float *b1, float *y0, float *y1, int n_rhs);
int k_saddle_precond_tp(fsd_ctx *ctx, const float *b, float *x);

int k_saddle_precond(fsd_ctx *ctx, const float *b, float *x)
{
    if (ctx->precond_mode == 2 && lp_active(ctx)) return lp_apply(ctx, b, b + 11 * (int64_t)ctx->N, b, x, 1);
    if (ctx->ic_jac_k > 0) return k_saddle_precond_jacobi(ctx, b, x);
    // one sweep pair on d = b_F - b_U when the one-launch sweeps are built
    const int tp = k_saddle_precond_tp(ctx, b, x);
    if (tp <= 0) return tp;
    const int N = ctx->N;
    float *gF = ctx->d_g12, *gU = ctx->d_g12 + 6 * (int64_t)N;
    int rc = k_precond_apply2(ctx, b, b + 11 * (int64_t)N, gF, gU, 2);
    if (rc) return rc;
    hipLaunchKernelGGL(saddle_combine_kernel, dim3(nblk(11 * (int64_t)N, 256)), dim3(256), 0, ctx->stream, N, b, gF,
                       gU, x);
    FSD_HIP(hipGetLastError());
    return 0;
}

// Saddle_Multiply (Saddle.cu:80-151): y_top = M x_top + [x_U; 0], y_bot = x_F - R_FU x_U
int k_saddle_multiply(fsd_ctx *ctx, const float4 *pos, const float *x, float *y)
{
    const int64_t N = ctx->N;
    int rc = k_mobility(ctx, pos, x, y, 3, x + 11 * N);
    if (rc) return rc;
    return k_rfu_apply(ctx, x + 11 * N, y + 11 * N, x, -1.0f);
}

// ------------------------------------------------------------ RHS
// Integrator_AddStrainRate_kernel (Helper_Integrator.cu:114-158) and
// rhs[11N:] -= F_applied (Integrator.cu:831-841); rhs assumed zeroed.
__global__ void strain_rhs_kernel(int N, float *rhs, float shear_rate, float B2, const float *mask2, const float *ori,
                                  const float *F)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    float *e = rhs + 6 * (int64_t)N + 5 * (int64_t)i;
    e[1] += shear_rate;
    if (B2 != 0.f && ori) {
        const float px = ori[3 * i], py = ori[3 * i + 1], pz = ori[3 * i + 2];
        const float b2 = -0.6f * B2 * mask2[i];
        e[0] -= b2 * (px * px - pz * pz);
        e[1] -= b2 * (2.f * px * py);
        e[2] -= b2 * (2.f * px * pz);
        e[3] -= b2 * (2.f * py * pz);
        e[4] -= b2 * (py * py - pz * pz);
    }
    float *u = rhs + 11 * (int64_t)N + 6 * (int64_t)i;
    for (int a = 0; a < 6; ++a) u[a] -= F[6 * (int64_t)i + a];
}

int k_strain_rhs(fsd_ctx *ctx, float *rhs, float shear_rate, const float *ori, const float *force)
{
    hipLaunchKernelGGL(strain_rhs_kernel, dim3(nblk(ctx->N, 256)), dim3(256), 0, ctx->stream, ctx->N, rhs, shear_rate,
                       ori ? ctx->p.sqm_B2 : 0.f, ctx->d_mask2, ori, force);
    FSD_HIP(hipGetLastError());
    return 0;
}

// ------------------------------------------------------------ Euler
// Integrator_ExplicitEuler_Shear_kernel (Integrator.cu:126-228)
__global__ void euler_shear_kernel(int N, float4 *pos, float *ori, float4 *pos_gb, int *image, const float *vel,
                                   float B1, const float *mask1, const float *noise, BoxF b, float dt, float shear_rate)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    float4 p4 = pos[i];
    float px = p4.x, py = p4.y, pz = p4.z;
    float vx = vel[6 * (int64_t)i], vy = vel[6 * (int64_t)i + 1], vz = vel[6 * (int64_t)i + 2];
    float wx = vel[6 * (int64_t)i + 3], wy = vel[6 * (int64_t)i + 4], wz = vel[6 * (int64_t)i + 5];
    vx += shear_rate * py;
    wz -= shear_rate / 2.f;
    if (noise) { wx += noise[3 * i]; wy += noise[3 * i + 1]; wz += noise[3 * i + 2]; }
    float q0 = 1.f, qx = 0.f, qy = 0.f, qz = 0.f;
    float aw = sqrtf(wx * wx + wy * wy + wz * wz);
    if (aw > 1e-6f) {
        float ang = aw * dt;
        q0 = cosf(ang / 2.f);
        float s = sinf(ang / 2.f) / aw;
        qx = wx * s; qy = wy * s; qz = wz * s;
    }
    float ox = 0.f, oy = 0.f, oz = 0.f;
    if (ori) { ox = ori[3 * i]; oy = ori[3 * i + 1]; oz = ori[3 * i + 2]; }
    const float m1 = mask1 ? mask1[i] : 1.f;
    const float act = -2.f / 3.f * B1 * m1;
    vx -= act * ox; vy -= act * oy; vz -= act * oz;
    float4 g = pos_gb[i];
    g.x += (vx - shear_rate * py + shear_rate * g.y) * dt;
    g.y += vy * dt;
    g.z += vz * dt;
    pos_gb[i] = g;
    px += vx * dt; py += vy * dt; pz += vz * dt;
    int ix = image[3 * i], iy = image[3 * i + 1], iz = image[3 * i + 2];
    box_wrap(b, px, py, pz, ix, iy, iz);
    pos[i] = make_float4(px, py, pz, p4.w);
    image[3 * i] = ix; image[3 * i + 1] = iy; image[3 * i + 2] = iz;
    if (ori) {
        float qq = qx * qx + qy * qy + qz * qz, qp = qx * ox + qy * oy + qz * oz;
        float cx = qy * oz - qz * oy, cy = qz * ox - qx * oz, cz = qx * oy - qy * ox;
        float nx = (q0 * q0 - qq) * ox + 2.f * qp * qx + 2.f * q0 * cx;
        float ny = (q0 * q0 - qq) * oy + 2.f * qp * qy + 2.f * q0 * cy;
        float nz = (q0 * q0 - qq) * oz + 2.f * qp * qz + 2.f * q0 * cz;
        float m = sqrtf(nx * nx + ny * ny + nz * nz);
        ori[3 * i] = nx / m; ori[3 * i + 1] = ny / m; ori[3 * i + 2] = nz / m;
    }
}

// Director rotation pv <- q pv q* with the quaternion of angular velocity w over
// time tau (Integrator.cu:278-286, 312-321), renormalised
__device__ inline void rotate_director(float wx, float wy, float wz, float tau, float &ox, float &oy, float &oz)
{
    float q0 = 1.f, qx = 0.f, qy = 0.f, qz = 0.f;
    const float aw = sqrtf(wx * wx + wy * wy + wz * wz);
    if (aw > 1e-6f) {
        const float ang = aw * tau;
        q0 = cosf(ang / 2.f);
        const float s = sinf(ang / 2.f) / aw;
        qx = wx * s; qy = wy * s; qz = wz * s;
    }
    const float qq = qx * qx + qy * qy + qz * qz, qp = qx * ox + qy * oy + qz * oz;
    const float cx = qy * oz - qz * oy, cy = qz * ox - qx * oz, cz = qx * oy - qy * ox;
    const float nx = (q0 * q0 - qq) * ox + 2.f * qp * qx + 2.f * q0 * cx;
    const float ny = (q0 * q0 - qq) * oy + 2.f * qp * qy + 2.f * q0 * cy;
    const float nz = (q0 * q0 - qq) * oz + 2.f * qp * qz + 2.f * q0 * cz;
    const float m = sqrtf(nx * nx + ny * ny + nz * nz);
    ox = nx / m; oy = ny / m; oz = nz / m;
}

// Integrator_ExplicitEuler1_Shear_kernel (Integrator.cu:232-326): first stage of
// the second-order Runge-Kutta scheme.  The unwrapped position advances half a
// step, the periodic position a full step without wrapping (the second stage
// averages it), pos.w is kept.
__global__ void rk2_stage1_kernel(int N, const float4 *pos_in, const float *ori_in, float4 *pos_out, float *ori_out,
                                  float4 *pos_gb, const float *vel, float B1, const float *mask1, const float *noise,
                                  float dt, float shear_rate)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    const float4 p4 = pos_in[i];
    float px = p4.x, py = p4.y, pz = p4.z;
    float vx = vel[6 * (int64_t)i], vy = vel[6 * (int64_t)i + 1], vz = vel[6 * (int64_t)i + 2];
    float wx = vel[6 * (int64_t)i + 3], wy = vel[6 * (int64_t)i + 4], wz = vel[6 * (int64_t)i + 5];
    vx += shear_rate * py;
    wz -= shear_rate / 2.f;
    if (noise) { wx += noise[3 * i]; wy += noise[3 * i + 1]; wz += noise[3 * i + 2]; }
    float ox = ori_in[3 * i], oy = ori_in[3 * i + 1], oz = ori_in[3 * i + 2];
    const float act = -2.f / 3.f * B1 * (mask1 ? mask1[i] : 1.f);
    vx -= act * ox; vy -= act * oy; vz -= act * oz;
    float4 g = pos_gb[i];
    g.x += (vx - shear_rate * py + shear_rate * g.y) * 0.5f * dt;
    g.y += vy * 0.5f * dt;
    g.z += vz * 0.5f * dt;
    pos_gb[i] = g;
    px += vx * dt; py += vy * dt; pz += vz * dt;
    pos_out[i] = make_float4(px, py, pz, p4.w);
    rotate_director(wx, wy, wz, dt, ox, oy, oz);
    ori_out[3 * i] = ox; ori_out[3 * i + 1] = oy; ori_out[3 * i + 2] = oz;
}

// Integrator_RK_Shear_kernel (Integrator.cu:329-438): second stage.  Position
// and director are the combinations c1 * state1 + c2 * state2 (the director
// renormalised), moved by c3 * dt and wrapped; the unwrapped position advances
// half a step; pos.w is written as 0 as the reference does.
__global__ void rk2_stage2_kernel(int N, float c1, const float4 *pos1, const float *ori1, float c2, const float4 *pos2,
                                  const float *ori2, float4 *pos_out, float *ori_out, float4 *pos_gb, const float *vel,
                                  float B1, const float *mask1, const float *noise, int *image, BoxF b, float c3,
                                  float dt, float shear_rate)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    const float4 a4 = pos1[i], b4 = pos2[i];
    float px = c1 * a4.x + c2 * b4.x, py = c1 * a4.y + c2 * b4.y, pz = c1 * a4.z + c2 * b4.z;
    float vx = vel[6 * (int64_t)i], vy = vel[6 * (int64_t)i + 1], vz = vel[6 * (int64_t)i + 2];
    float wx = vel[6 * (int64_t)i + 3], wy = vel[6 * (int64_t)i + 4], wz = vel[6 * (int64_t)i + 5];
    vx += shear_rate * py;
    wz -= shear_rate / 2.f;
    if (noise) { wx += noise[3 * i]; wy += noise[3 * i + 1]; wz += noise[3 * i + 2]; }
    float ox = ori1[3 * i] * c1 + ori2[3 * i] * c2;
    float oy = ori1[3 * i + 1] * c1 + ori2[3 * i + 1] * c2;
    float oz = ori1[3 * i + 2] * c1 + ori2[3 * i + 2] * c2;
    const float m0 = sqrtf(ox * ox + oy * oy + oz * oz);
    ox /= m0; oy /= m0; oz /= m0;
    const float act = -2.f / 3.f * B1 * (mask1 ? mask1[i] : 1.f);
    vx -= act * ox; vy -= act * oy; vz -= act * oz;
    float4 g = pos_gb[i];
    g.x += (vx - shear_rate * py + shear_rate * g.y) * 0.5f * dt;
    g.y += vy * 0.5f * dt;
    g.z += vz * 0.5f * dt;
    pos_gb[i] = g;
    px += vx * dt * c3; py += vy * dt * c3; pz += vz * dt * c3;
    int ix = image[3 * i], iy = image[3 * i + 1], iz = image[3 * i + 2];
    box_wrap(b, px, py, pz, ix, iy, iz);
    pos_out[i] = make_float4(px, py, pz, 0.f);
    image[3 * i] = ix; image[3 * i + 1] = iy; image[3 * i + 2] = iz;
    rotate_director(wx, wy, wz, dt * c3, ox, oy, oz);
    ori_out[3 * i] = ox; ori_out[3 * i + 1] = oy; ori_out[3 * i + 2] = oz;
}

int k_rk2_stage1(fsd_ctx *ctx, const float4 *pos_in, const float *ori_in, float4 *pos_out, float *ori_out,
                 float4 *pos_gb, const float *vel, const float *mask1, const float *noise, float dt, float shear_rate)
{
    hipLaunchKernelGGL(rk2_stage1_kernel, dim3(nblk(ctx->N, 256)), dim3(256), 0, ctx->stream, ctx->N, pos_in, ori_in,
                       pos_out, ori_out, pos_gb, vel, ctx->p.sqm_B1, mask1, noise, dt, shear_rate);
    FSD_HIP(hipGetLastError());
    return 0;
}

int k_rk2_stage2(fsd_ctx *ctx, float c1, const float4 *pos1, const float *ori1, float c2, const float4 *pos2,
                 const float *ori2, float4 *pos_out, float *ori_out, float4 *pos_gb, const float *vel,
                 const float *mask1, const float *noise, int *image, float c3, float dt, float shear_rate)
{
    hipLaunchKernelGGL(rk2_stage2_kernel, dim3(nblk(ctx->N, 256)), dim3(256), 0, ctx->stream, ctx->N, c1, pos1, ori1,
                       c2, pos2, ori2, pos_out, ori_out, pos_gb, vel, ctx->p.sqm_B1, mask1, noise, image, ctx->box, c3,
                       dt, shear_rate);
    FSD_HIP(hipGetLastError());
    return 0;
}

int k_euler_shear(fsd_ctx *ctx, float4 *pos, float *ori, float4 *pos_gb, int *image, const float *vel,
                  const float *mask1, const float *noise, float dt, float shear_rate, float B1)
{
    hipLaunchKernelGGL(euler_shear_kernel, dim3(nblk(ctx->N, 256)), dim3(256), 0, ctx->stream, ctx->N, pos, ori,
                       pos_gb, image, vel, B1, mask1, noise, ctx->box, dt, shear_rate);
    FSD_HIP(hipGetLastError());
    return 0;
}
