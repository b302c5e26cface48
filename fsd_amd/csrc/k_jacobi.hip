// Preconditioner application by Jacobi iterations on the triangular factors.
//
// G = P^T L^-T L^-1 P is applied without the level-by-level dependency chain
// (Anzt, Chow & Dongarra, "Iterative sparse triangular solves for
// preconditioning", Euro-Par 2015).  Both factors are brought to one form, a
// forward and a backward solve with unit diagonal blocks, iterated k times each:
//     c = R t,   y <- c - F y (from y = c),   u <- y - T u (from u = y),
//   IC(0):       R = Z = L_PP^-1,  F_PQ = Z_P L_PQ,     T_PQ = F_QP^T,           G t = Z^T u;
//   learned LDL^T (D + W) D^-1 (D + W)^T:
//                R = D^-1,         F_PQ = D_P^-1 W_PQ,  T_PQ = D_P^-1 W_QP^T,    G t = u.
// Every iteration reads each block once and is fully parallel over the N block
// rows, so an application is 2k + 1 short launches over all CUs instead of two chains
// of ~120 dependent steps on one CU.  For a fixed k the result is a fixed
// linear operator (a truncated Neumann series of the exact solves), so GMRES
// needs no flexible variant; k -> depth of the DAG gives the exact solves.
//
// Layout: every per-row vector is [N][6] in permuted order P; F is in the order of the lower
// pattern and T in the order of the upper one, so both directions run the same kernel.  A 64-lane
// wave owns 10 rows, six lanes per row (lane a computes component a), so the six lanes of a row
// read one row-major block's 144 contiguous bytes.  (Blocks stored as [3][6] pairs, so that each of
// a lane's three loads is contiguous over its row's lanes, took 6.2 instead of 5.6 us.)
// An iteration is bound by latency, not by its 12 MB (N = 32768, 78 K blocks): a row's first
// four columns lie in one int4, so its blocks and neighbour values are all loaded after one
// dependent load, where walking the row's list waited for a column and a gather per block.
// Measured there (learned factor, k = 5): 5.6 us per iteration in both directions, where the list
// walk with the inverse pivots applied in every iteration took 5.9 forward and 8.2 backward.
#include <algorithm>

#include "fsd_internal.h"

namespace {
constexpr int JROWS = 10;   // block rows per 64-lane wave (lanes 60..63 idle)
constexpr int ELL = 4;      // columns of a row held in its int4

// row and component of this lane; lanes without a row (false) get a valid one to load from
__device__ __forceinline__ bool jac_row(int N, int &P, int &a)
{
    const int lane = threadIdx.x & 63;
    // rows in one contiguous range per XCD (cache lines shared by neighbouring rows stay in one L2)
    const int wave = (int)((xcd_remap(blockIdx.x, gridDim.x) * (int64_t)blockDim.x + threadIdx.x) >> 6);
    const int g = lane / 6;
    a = lane - 6 * g;
    P = wave * JROWS + g;
    const bool ok = g < JROWS && P < N;
    P = min(P, N - 1);
    return ok;
}

inline int jac_blocks(int N) { return nblk(nblk(N, JROWS) * 64, 256); }

// the six lanes' values of this lane's row
__device__ __forceinline__ void row_values(float v, float out[6])
{
    const int lane = threadIdx.x & 63, base = min(lane / 6, JROWS - 1) * 6;
#pragma unroll
    for (int q = 0; q < 6; ++q) out[q] = __shfl(v, base + q, 64);
}

struct Row6 { float2 v[3]; };
__device__ __forceinline__ Row6 load6(const float *p)
{
    const float2 *q = reinterpret_cast<const float2 *>(p);
    return Row6{{q[0], q[1], q[2]}};
}
// row a of block e
__device__ __forceinline__ Row6 load_block(const float *F, int64_t e, int a) { return load6(F + 36 * e + 6 * a); }
__device__ __forceinline__ void store_block(float *F, int64_t e, int a, const float r[6])
{
    float2 *q = reinterpret_cast<float2 *>(F + 36 * e + 6 * a);
#pragma unroll
    for (int j = 0; j < 3; ++j) q[j] = make_float2(r[2 * j], r[2 * j + 1]);
}
__device__ __forceinline__ float dot6(const Row6 &f, const Row6 &y)
{
    return f.v[0].x * y.v[0].x + f.v[0].y * y.v[0].y + f.v[1].x * y.v[1].x + f.v[1].y * y.v[1].y +
           f.v[2].x * y.v[2].x + f.v[2].y * y.v[2].y;
}
}  // namespace

// first columns of every row: (col of entry 0 .. 3), the row's own number where it has fewer
__global__ void bj_ell_kernel(int N, const int *lrow, const int *lcol, const int *urow, const int *ucol, int4 *lell,
                              int4 *uell)
{
    const int P = blockIdx.x * blockDim.x + threadIdx.x;
    if (P >= N) return;
    for (int d = 0; d < 2; ++d) {
        const int *row = d ? urow : lrow, *col = d ? ucol : lcol;
        const int e0 = row[P], n = row[P + 1] - e0;
        int c[ELL];
#pragma unroll
        for (int k = 0; k < ELL; ++k) c[k] = k < n ? col[e0 + k] : P;
        (d ? uell : lell)[P] = make_int4(c[0], c[1], c[2], c[3]);
    }
}

// F of row P's lower blocks and T of its upper ones; six lanes per row, lane a forms row a
template <bool LDL>
__global__ void bj_fold_kernel(int N, const int *lrow, const int *urow, const int *ucol, const int *upos,
                               const float *R, const float *blk, float *F, float *T)
{
    int P, a;
    if (!jac_row(N, P, a)) return;
    float A[6];
#pragma unroll
    for (int q = 0; q < 6; ++q) A[q] = R[(int64_t)P * 36 + 6 * a + q];
    for (int e = lrow[P]; e < lrow[P + 1]; ++e) {
        const float *B = blk + (int64_t)e * 36;
        float r[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int q = 0; q < 6; ++q)
            if (LDL || q <= a)   // Z is lower triangular
#pragma unroll
                for (int c = 0; c < 6; ++c) r[c] += A[q] * B[6 * q + c];
        store_block(F, e, a, r);
    }
    for (int u = urow[P]; u < urow[P + 1]; ++u) {
        const float *B = blk + (int64_t)upos[u] * 36, *Z = R + (int64_t)ucol[u] * 36;
        float r[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < 6; ++c)
#pragma unroll
            for (int q = 0; q < 6; ++q) {
                if (LDL) r[c] += A[q] * B[6 * c + q];
                else if (q <= c) r[c] += Z[6 * c + q] * B[6 * q + a];
            }
        store_block(T, u, a, r);
    }
}

// c_P = R_P t_P with t_P = (b0 - b1)[perm P] (b1 may be null)
__global__ void __launch_bounds__(256) bj_pre_kernel(int N, const int *perm, const float *R, const float *b0,
                                                     const float *b1, float *c)
{
    int P, a;
    const bool ok = jac_row(N, P, a);
    const Row6 r = load6(R + (int64_t)P * 36 + 6 * a);
    const int64_t i = perm[P];
    float t = b0[6 * i + a];
    if (b1) t -= b1[6 * i + a];
    float t6[6];
    row_values(t, t6);
    if (!ok) return;
    c[6 * (int64_t)P + a] = dot6(r, Row6{{make_float2(t6[0], t6[1]), make_float2(t6[2], t6[3]), make_float2(t6[4], t6[5])}});
}

// what the last backward iteration does with u: g = P^T Z^T u (Z null: P^T u); mode 0: out = g (6N);
// mode 1: the saddle preconditioner's combination x_F = b_F - g, x_S = b_S, x_U = g
// (Saddle.cu:171-264 with g = G (b_F - b_U))
struct BjPost {
    const int *perm;
    const float *Z, *b;
    float *x;
    int mode;
};

// u: the row's six values, or (Z null) this lane's value in u[0]
__device__ __forceinline__ void bj_write(const BjPost &post, int N, int P, int a, const float u[6])
{
    float g = u[0];
    if (post.Z) {
        g = 0.f;
#pragma unroll
        for (int r = 0; r < 6; ++r)
            if (r >= a) g += post.Z[(int64_t)P * 36 + 6 * r + a] * u[r];
    }
    const int64_t i = post.perm[P], n6 = 6 * (int64_t)N, n11 = 11 * (int64_t)N;
    if (post.mode == 0) {
        post.x[6 * i + a] = g;
        return;
    }
    post.x[6 * i + a] = post.b[6 * i + a] - g;
    post.x[n11 + 6 * i + a] = g;
    if (a < 5) post.x[n6 + 5 * i + a] = post.b[n6 + 5 * i + a];
}

// yout_P = c_P - sum_e F_e yin_col(e)
template <bool LAST>
__global__ void __launch_bounds__(256) bj_iter_kernel(int N, const int *row, const int4 *ell, const int *col,
                                                      const float *F, const float *c, const float *yin, float *yout,
                                                      BjPost post)
{
    int P, a;
    const bool ok = jac_row(N, P, a);
    const int4 q = ell[P];
    const int e0 = row[P], n = row[P + 1] - e0;
    float v = c[6 * (int64_t)P + a];
    const int cols[ELL] = {q.x, q.y, q.z, q.w};
    Row6 f[ELL], y[ELL];
#pragma unroll
    for (int k = 0; k < ELL; ++k) {   // past the row's end: its last block (or the next row's first) again, not used
        f[k] = load_block(F, e0 + min(k, max(n - 1, 0)), a);
        y[k] = load6(yin + 6 * (int64_t)cols[k]);
    }
#pragma unroll
    for (int k = 0; k < ELL; ++k) v = k < n ? v - dot6(f[k], y[k]) : v;
    for (int k = ELL; k < n; ++k)
        v -= dot6(load_block(F, e0 + k, a), load6(yin + 6 * (int64_t)col[e0 + k]));
    if (!LAST) {
        if (ok) yout[6 * (int64_t)P + a] = v;
        return;
    }
    float u[6] = {v, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (post.Z) row_values(v, u);
    if (ok) bj_write(post, N, P, a, u);
}

// The whole application by one workgroup, for factors that fit a CU: the iterates live in LDS and
// each direction's blocks in registers, a block or two per thread.  An iteration is one 6x6 product
// per block into LDS, a barrier, the sum of every row's products, a barrier: 2 us where a launch with
// its gap takes 4 (N = 700, phi = 0.4, k = 8: 39 us against 70; the call 95 -> 70 us).  Bound by the one
// CU's LDS and VALU.  (Six lanes per block as in bj_iter_kernel read each neighbour's values six times: 54 us.)
constexpr int BS_NT = 1024, BS_HOLD = 2;
constexpr int BS_MAXN = 1900;   // two vectors of 24 bytes a row and the products of 2048 blocks: 145 of 160 KB of LDS
// What it saves per iteration has to pay for its first and last steps, which one CU takes over all rows: k
// from about N / 300 on, and from 5 on for every size (11 launches take 70 to 90 us a call, by the gap between
// them, which has two values here).  Calls by one workgroup and by launches, us, at k = 1, 2, 3, 5, 8:
//   N = 343,  828 blocks   41 44 45 49 54   42 48 55 71 91
//   N = 700,  1465         48 50 53 58 65   41 47 55 73 90
//   N = 1000, 1563         52 54 57 63 72   41 48 54 71 89
//   N = 1500, 1462         57 60 62 67 75   40 46 52 69 87
//   N = 1900, 2046         63 66 70 78 89   41 46 53 69 88
inline bool bs_pays(int N, int k) { return k >= 5 || N <= 300 * k + 50; }
constexpr int BS_SUM = 3;       // products of a row read together
template <int HOLD>
__global__ void __launch_bounds__(BS_NT) bj_small_kernel(int N, int nlow, int k, const int *lrow, const int *lcol,
                                                         const float *F, const int *urow, const int *ucol,
                                                         const float *T, const float *R, const float *b0,
                                                         const float *b1, BjPost post)
{
    extern __shared__ float lds[];
    const int n6 = 6 * N, tid = threadIdx.x;
    float *c = lds, *y = lds + n6, *prod = lds + 2 * n6;    // prod: [nlow + 1][6]
    unsigned short *first = reinterpret_cast<unsigned short *>(prod + 6 * (nlow + 1));   // of each row, N + 1
#pragma unroll 1
    for (int q = tid; q < n6; q += BS_NT) {
        const int64_t i = post.perm[q / 6];
        float t = b0[6 * i + q % 6];
        if (b1) t -= b1[6 * i + q % 6];
        y[q] = t;
    }
    __syncthreads();
#pragma unroll 1
    for (int q = tid; q < n6; q += BS_NT) c[q] = dot6(load6(R + 6 * (int64_t)q), load6(y + 6 * (q / 6)));
    __syncthreads();
#pragma unroll 1
    for (int dir = 0; dir < 2; ++dir) {
        const int *row = dir ? urow : lrow, *col = dir ? ucol : lcol;
        const float4 *blk = reinterpret_cast<const float4 *>(dir ? T : F);
        float4 f[HOLD][9];
        int at[HOLD];                                       // the neighbour's values of each block
#pragma unroll
        for (int h = 0; h < HOLD; ++h) {
            const int e = tid + h * BS_NT;
            at[h] = e < nlow ? 6 * col[e] : -1;
#pragma unroll
            for (int q = 0; q < 9; ++q) f[h][q] = blk[9 * (int64_t)(e < nlow ? e : 0) + q];
        }
#pragma unroll 1
        for (int q = tid; q <= N; q += BS_NT) first[q] = (unsigned short)row[q];
        // the iterates start from c
#pragma unroll 1
        for (int q = tid; q < n6; q += BS_NT) y[q] = c[q];
        __syncthreads();
#pragma unroll 1
        for (int it = 0; it < k; ++it) {
#pragma unroll
            for (int h = 0; h < HOLD; ++h)
                if (at[h] >= 0) {
                    const Row6 v = load6(y + at[h]);
                    const float *m = reinterpret_cast<const float *>(f[h]);
                    float p[6];
#pragma unroll
                    for (int r = 0; r < 6; ++r)
                        p[r] = m[6 * r] * v.v[0].x + m[6 * r + 1] * v.v[0].y + m[6 * r + 2] * v.v[1].x +
                               m[6 * r + 3] * v.v[1].y + m[6 * r + 4] * v.v[2].x + m[6 * r + 5] * v.v[2].y;
                    float2 *o = reinterpret_cast<float2 *>(prod + 6 * (tid + h * BS_NT));
#pragma unroll
                    for (int r = 0; r < 3; ++r) o[r] = make_float2(p[2 * r], p[2 * r + 1]);
                }
            __syncthreads();
#pragma unroll 1
            for (int P = tid; P < N; P += BS_NT) {
                const int e0 = first[P], n = first[P + 1] - e0;
                Row6 v = load6(c + 6 * P);
                for (int j = 0; j < n; j += BS_SUM) {
                    Row6 d[BS_SUM];
#pragma unroll
                    for (int u = 0; u < BS_SUM; ++u) d[u] = load6(prod + 6 * (e0 + min(j + u, n - 1)));
#pragma unroll
                    for (int u = 0; u < BS_SUM; ++u)
                        if (j + u < n)
#pragma unroll
                            for (int q = 0; q < 3; ++q) { v.v[q].x -= d[u].v[q].x; v.v[q].y -= d[u].v[q].y; }
                }
                float2 *o = reinterpret_cast<float2 *>(y + 6 * P);
#pragma unroll
                for (int q = 0; q < 3; ++q) o[q] = v.v[q];
            }
            __syncthreads();
        }
        if (dir == 0) {                                     // the backward solve starts from the forward one's result
            float *t = c;
            c = y;
            y = t;
        }
    }
#pragma unroll 1
    for (int q = tid; q < n6; q += BS_NT) {
        const float *u = y + 6 * (q / 6);
        const float v[6] = {post.Z ? u[0] : y[q], u[1], u[2], u[3], u[4], u[5]};
        bj_write(post, N, q / 6, q % 6, v);
    }
}

int k_jacobi_init(fsd_ctx *ctx)
{
    for (auto k : {bj_small_kernel<1>, bj_small_kernel<BS_HOLD>})
        FSD_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(k), hipFuncAttributeMaxDynamicSharedMemorySize,
                                    160 * 1024));
    return 0;
}

int k_jacobi_ell(fsd_ctx *ctx)
{
    hipLaunchKernelGGL(bj_ell_kernel, dim3(nblk(ctx->N, 256)), dim3(256), 0, ctx->stream, ctx->N, ctx->d_lrow,
                       ctx->d_lcol, ctx->d_urow, ctx->d_ucol, ctx->d_lell, ctx->d_uell);
    FSD_HIP(hipGetLastError());
    return 0;
}

// folded blocks of the IC(0) factor (and its diagonal block inverses)
int k_jacobi_pack(fsd_ctx *ctx)
{
    const int N = ctx->N;
    const int r = k_diag_inverse(ctx);
    if (r) return r;
    hipLaunchKernelGGL(bj_fold_kernel<false>, dim3(jac_blocks(N)), dim3(256), 0, ctx->stream, N, ctx->d_lrow,
                       ctx->d_urow, ctx->d_ucol, ctx->d_upos, ctx->d_tp_Z, ctx->d_Lblk, ctx->d_Fblk, ctx->d_Tblk);
    FSD_HIP(hipGetLastError());
    return 0;
}

// folded blocks of the learned factor: pair blocks W, inverse pivots Dinv
int k_jacobi_pack_ldl(fsd_ctx *ctx, const float *W, const float *Dinv)
{
    const int N = ctx->N;
    hipLaunchKernelGGL(bj_fold_kernel<true>, dim3(jac_blocks(N)), dim3(256), 0, ctx->stream, N, ctx->d_lrow,
                       ctx->d_urow, ctx->d_ucol, ctx->d_upos, Dinv, W, ctx->d_Fblk, ctx->d_Tblk);
    FSD_HIP(hipGetLastError());
    return 0;
}

// The folded factor applied by k iterations each way; R: its diagonal matrices, Zpost: Z of the last
// step (null for the learned factor); bsaddle, x, mode: BjPost.  prof_slot: the class of the forward
// iterations.
int k_bj_apply(fsd_ctx *ctx, int k, int prof_slot, const float *R, const float *Zpost, const float *b0,
               const float *b1, const float *bsaddle, float *x, int mode)
{
    const int N = ctx->N;
    const int64_t n6 = 6 * (int64_t)N;
    hipEvent_t ev, e1;
    const int nlow = (int)ctx->pch.nlow;
    if (N <= BS_MAXN && nlow <= BS_HOLD * BS_NT && bs_pays(N, k)) {
        const size_t lds = sizeof(float) * (2 * n6 + 6 * (nlow + 1)) + sizeof(unsigned short) * (N + 2);
        const BjPost post{ctx->d_perm, Zpost, bsaddle, x, mode};
        auto go = [&](auto kernel) -> int {
            hipLaunchKernelGGL(kernel, dim3(1), dim3(BS_NT), lds, ctx->stream, N, nlow, k, ctx->d_lrow, ctx->d_lcol,
                               ctx->d_Fblk, ctx->d_urow, ctx->d_ucol, ctx->d_Tblk, R, b0, b1, post);
            FSD_HIP(hipGetLastError());
            return 0;
        };
        prof_begin(ctx, PROF_TRSV, &ev);
        const int rc = nlow <= BS_NT ? go(bj_small_kernel<1>) : go(bj_small_kernel<BS_HOLD>);
        prof_end(ctx, PROF_TRSV, ev);
        return rc;
    }
    prof_begin(ctx, PROF_TRSV, &ev);
    const dim3 g(jac_blocks(N)), b(256);
    float *const buf[4] = {ctx->d_jac, ctx->d_jac + n6, ctx->d_jac + 2 * n6, ctx->d_jac + 3 * n6};
    hipLaunchKernelGGL(bj_pre_kernel, g, b, 0, ctx->stream, N, ctx->d_perm, R, b0, b1, buf[0]);
    const float *c = buf[0], *y = c;
    float *fo[2] = {buf[1], buf[2]};
    prof_begin(ctx, prof_slot, &e1);   // the k forward iterations, one event pair
    for (int it = 0; it < k; ++it) {
        float *out = fo[it & 1];
        hipLaunchKernelGGL(bj_iter_kernel<false>, g, b, 0, ctx->stream, N, ctx->d_lrow, ctx->d_lell, ctx->d_lcol,
                           ctx->d_Fblk, c, y, out, BjPost{});
        y = out;
    }
    prof_end_n(ctx, prof_slot, e1, k);
    // the backward iterates never overwrite y: they alternate between buf[3] and the forward buffer y does not use
    float *bo[2] = {buf[3], (y == buf[1]) ? buf[2] : buf[1]};
    const float *u = y;
    for (int it = 0; it < k; ++it) {   // the last iteration writes the preconditioner's output
        float *out = bo[it & 1];
        if (it < k - 1)
            hipLaunchKernelGGL(bj_iter_kernel<false>, g, b, 0, ctx->stream, N, ctx->d_urow, ctx->d_uell, ctx->d_ucol,
                               ctx->d_Tblk, y, u, out, BjPost{});
        else
            hipLaunchKernelGGL(bj_iter_kernel<true>, g, b, 0, ctx->stream, N, ctx->d_urow, ctx->d_uell, ctx->d_ucol,
                               ctx->d_Tblk, y, u, out, BjPost{ctx->d_perm, Zpost, bsaddle, x, mode});
        u = out;
    }
    FSD_HIP(hipGetLastError());
    prof_end(ctx, PROF_TRSV, ev);
    return 0;
}

// x = saddle preconditioner of b (17N) with g = G (b_F - b_U)
int k_saddle_precond_jacobi(fsd_ctx *ctx, const float *b, float *x)
{
    return k_bj_apply(ctx, ctx->ic_jac_k, PROF_JAC, ctx->d_tp_Z, ctx->d_tp_Z, b, b + 11 * (int64_t)ctx->N, b, x, 1);
}

// y = G b (6N)
int k_precond_apply_jacobi(fsd_ctx *ctx, const float *b, float *y)
{
    return k_bj_apply(ctx, ctx->ic_jac_k, PROF_JAC, ctx->d_tp_Z, ctx->d_tp_Z, b, nullptr, nullptr, y, 0);
}
