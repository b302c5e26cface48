// Transforms of the far field's grids: 11 real fields [11][Nx][Ny][Nz] <-> half spectra
// [11][Nx][Ny][Nz / 2 + 1] (the layout of a real-to-complex 3-D transform), with the
// Green's function between the forward and the inverse transform along x.
//
//   yz_forward_kernel   one workgroup per plane (field, x): the plane is read into LDS once,
//                       transformed along z and y there and written once;
//   x_green_kernel      one workgroup per ky and XKC consecutive kz of all 11 fields: forward
//                       along x, Green's function, inverse along x;
//   yz_inverse_kernel   the planes back to real space;
//
// with the library's 2-D transforms in the place of the first and the last where a plane exceeds LDS.
//
// Bound: HBM for large grids, the barriers between the LDS stages for small ones.  Measured
// (mobility product, kernel trace): 135^3, three passes 252 us where the 3-D library plans of this
// odd length and the separate Green's function took 1113 us; 72^3, 64 us as with the library's 2-D
// transforms; 40^3, 30 us against 37; 20^3, 22 us against 23 (3-D plans).
// Each pass reads and writes its data once, so a product moves 6 x 11 x 4 M bytes here
// whatever the lengths' factors are.  Grid lengths are 2^a 3^b 5^c; fft::split splits
// them into few large radices, which a thread transforms in registers.
#include <algorithm>
#include <cmath>
#include <vector>

#include "fsd_internal.h"
#include "green.h"

namespace {
struct YzArgs {
    FftAxis y, z;
    int Nx, Ny, Nz, Nzh, zpairs;   // zpairs: pairs of y rows
    int pz;                        // floats of a grid row in memory, a multiple of 4
};

// LDS: the plane, row y at y Nzh complex (rows 2p, 2p + 1 share 2 Nzh places while they are one
// complex row of length Nz), then the tables
__device__ __forceinline__ void load_tables(const FftAxis &y, const FftAxis &z, float2 *tw, unsigned short *loc)
{
    for (int i = threadIdx.x; i < y.n; i += blockDim.x) { tw[i] = y.tw[i]; loc[i] = y.loc[i]; }
    for (int i = threadIdx.x; i < z.n; i += blockDim.x) { tw[y.n + i] = z.tw[i]; loc[y.n + i] = z.loc[i]; }
}

constexpr int YZ_LOADS = 4;        // global loads of 16 bytes a thread has in flight

// most (row pair, kz) tasks of a thread in the real unpacking: bounds the plane to NT YZ_HOLD pairs of modes
template <int NT>
constexpr int yz_hold() { return NT == 256 ? 4 : 10; }

__device__ __forceinline__ float2 *plane_of(char *lds) { return reinterpret_cast<float2 *>(lds); }

// rows of a pair along z (tasks of a row consecutive), and columns along y (columns consecutive)
struct ZRows {
    fft::FastDiv per;
    int row;
    __device__ ZRows(int tasks, int row_) : per(tasks), row(row_) {}
    __device__ __forceinline__ int operator()(int idx, int &t) const { return per(idx, t) * row; }
};
struct YColumns {
    fft::FastDiv cols;
    __device__ explicit YColumns(int n) : cols(n) {}
    __device__ __forceinline__ int operator()(int idx, int &t) const
    {
        int c;
        t = cols(idx, c);
        return c;
    }
};
}  // namespace

template <int NT>
__global__ void __launch_bounds__(NT) yz_forward_kernel(YzArgs a, const float *grid, float2 *spec)
{
    extern __shared__ char lds[];
    float2 *buf = plane_of(lds);
    const int Nz = a.Nz, Nzh = a.Nzh, Ny = a.Ny, pairs = a.zpairs, row = 2 * Nzh;
    float2 *tw = buf + (int64_t)pairs * row;
    unsigned short *loc = reinterpret_cast<unsigned short *>(tw + Ny + Nz);
    load_tables(a.y, a.z, tw, loc);
    // real rows 2p and 2p + 1 as the real and imaginary part of one row
    const int p4 = a.pz / 4, np = Ny * p4;
    const float4 *in = reinterpret_cast<const float4 *>(grid + (int64_t)blockIdx.x * Ny * a.pz);
    const fft::FastDiv by_z(p4);
    float *fb = reinterpret_cast<float *>(buf);
    for (int i0 = 0; i0 < np; i0 += NT * YZ_LOADS) {
        float4 v[YZ_LOADS];
#pragma unroll
        for (int u = 0; u < YZ_LOADS; ++u) v[u] = in[min(i0 + u * NT + (int)threadIdx.x, np - 1)];
#pragma unroll
        for (int u = 0; u < YZ_LOADS; ++u) {
            const int i = i0 + u * NT + threadIdx.x;
            int z;
            const int y = by_z(i, z);
            if (i < np) {
                float *o = fb + 2 * ((y >> 1) * row + 4 * z) + (y & 1);
                const float w[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    if (4 * z + k < Nz) o[2 * k] = w[k];
            }
        }
    }
    if (Ny & 1)   // the last row's missing partner
        for (int z = threadIdx.x; z < Nz; z += NT) fb[2 * ((pairs - 1) * row + z) + 1] = 0.f;
    __syncthreads();
    fft::transform<false, NT>(buf, a.z, pairs, [&](int tasks) { return ZRows(tasks, row); }, 1, tw + Ny);
    // S = A + i B of the two real rows: A_k = (S_k + conj S_-k) / 2, B_k = (S_k - conj S_-k) / 2i
    {
        constexpr int HOLD = yz_hold<NT>();
        const fft::FastDiv by_h(Nzh);
        const int total = pairs * Nzh;
        const unsigned short *lz = loc + Ny;
        float2 A[HOLD], B[HOLD];
#pragma unroll
        for (int u = 0; u < HOLD; ++u) {
            const int i = u * NT + threadIdx.x;
            if (i < total) {
                int k;
                const float2 *p = buf + by_h(i, k) * row;
                const float2 s = p[lz[k]], c = p[lz[k ? Nz - k : 0]];
                A[u] = make_float2(0.5f * (s.x + c.x), 0.5f * (s.y - c.y));
                B[u] = make_float2(0.5f * (s.y + c.y), 0.5f * (c.x - s.x));
            }
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < HOLD; ++u) {
            const int i = u * NT + threadIdx.x;
            if (i < total) {
                int k;
                float2 *p = buf + by_h(i, k) * row;
                p[k] = A[u];
                p[Nzh + k] = B[u];
            }
        }
        __syncthreads();
    }
    fft::transform<false, NT>(buf, a.y, Nzh, [&](int) { return YColumns(Nzh); }, Nzh, tw);
    const int nh = Ny * Nzh;
    float2 *out = spec + (int64_t)blockIdx.x * nh;
    const fft::FastDiv by_h(Nzh);
    for (int i = threadIdx.x; i < nh; i += NT) {
        int k;
        const int ky = by_h(i, k);
        out[i] = buf[loc[ky] * Nzh + k];
    }
}

template <int NT>
__global__ void __launch_bounds__(NT) yz_inverse_kernel(YzArgs a, const float2 *spec, float *grid)
{
    extern __shared__ char lds[];
    float2 *buf = plane_of(lds);
    const int Nz = a.Nz, Nzh = a.Nzh, Ny = a.Ny, pairs = a.zpairs, row = 2 * Nzh;
    float2 *tw = buf + (int64_t)pairs * row;
    unsigned short *loc = reinterpret_cast<unsigned short *>(tw + Ny + Nz);
    load_tables(a.y, a.z, tw, loc);
    const int nh = Ny * Nzh;
    const float2 *in = spec + (int64_t)blockIdx.x * nh;
    const fft::FastDiv by_h(Nzh);
    if (Ny & 1)
        for (int k = threadIdx.x; k < Nzh; k += NT) buf[Ny * Nzh + k] = make_float2(0.f, 0.f);
    constexpr int LOADS = 2 * YZ_LOADS;
    for (int i0 = 0; i0 < nh; i0 += NT * LOADS) {
        float2 v[LOADS];
        unsigned short r[LOADS];
#pragma unroll
        for (int u = 0; u < LOADS; ++u) {
            const int i = i0 + u * NT + threadIdx.x;
            int k;
            v[u] = i < nh ? in[i] : make_float2(0.f, 0.f);
            r[u] = i < nh ? a.y.loc[by_h(i, k)] : 0;
        }
#pragma unroll
        for (int u = 0; u < LOADS; ++u) {
            const int i = i0 + u * NT + threadIdx.x;
            int k;
            by_h(i, k);
            if (i < nh) buf[r[u] * Nzh + k] = v[u];
        }
    }
    __syncthreads();
    fft::transform<true, NT>(buf, a.y, Nzh, [&](int) { return YColumns(Nzh); }, Nzh, tw);
    // the two rows' half spectra as one complex row S = A + i B, S_-k = conj(A_k) + i conj(B_k); the modes
    // that are their own conjugates (kz = 0 and, for even Nz, Nz / 2) are real
    {
        constexpr int HOLD = yz_hold<NT>();
        const int total = pairs * Nzh;
        const unsigned short *lz = loc + Ny;
        float2 P[HOLD], Q[HOLD];
#pragma unroll
        for (int u = 0; u < HOLD; ++u) {
            const int i = u * NT + threadIdx.x;
            if (i < total) {
                int k;
                const float2 *p = buf + by_h(i, k) * row;
                float2 A = p[k], B = p[Nzh + k];
                if (k == 0 || 2 * k == Nz) A.y = B.y = 0.f;
                P[u] = make_float2(A.x - B.y, A.y + B.x);
                Q[u] = make_float2(A.x + B.y, B.x - A.y);
            }
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < HOLD; ++u) {
            const int i = u * NT + threadIdx.x;
            if (i < total) {
                int k;
                float2 *p = buf + by_h(i, k) * row;
                p[lz[k]] = P[u];
                if (k && 2 * k != Nz) p[lz[Nz - k]] = Q[u];
            }
        }
        __syncthreads();
    }
    fft::transform<true, NT>(buf, a.z, pairs, [&](int tasks) { return ZRows(tasks, row); }, 1, tw + Ny);
    // rows of pz floats; the padding repeats the row's end
    const int p4 = a.pz / 4, np = Ny * p4;
    float4 *out = reinterpret_cast<float4 *>(grid + (int64_t)blockIdx.x * Ny * a.pz);
    const float *fb = reinterpret_cast<const float *>(buf);
    const fft::FastDiv by_z(p4);
    for (int i = threadIdx.x; i < np; i += NT) {
        int z;
        const int y = by_z(i, z);
        const float *v = fb + 2 * ((y >> 1) * row) + (y & 1);
        z *= 4;
        out[i] = make_float4(v[2 * z], v[2 * min(z + 1, Nz - 1)], v[2 * min(z + 2, Nz - 1)], v[2 * min(z + 3, Nz - 1)]);
    }
}

// The x direction: element (c, x, ky, kz) at c Mh + (x Ny + ky) Nzh + kz.  A workgroup holds every
// mode of its columns with all 11 fields, so green_update applies point by point between the two
// transforms.  GREEN false: the inverse alone, for spectra that are already scaled.
// The chunks of a ky row share cache lines (a chunk is XKC of the row's Nzh modes): a contiguous
// range of rows per XCD keeps every line's readers and writers on one L2.
namespace {
template <int KC>
struct XColumns {   // LDS [field][x][kz of the chunk]; kz fastest over the tasks, then x
    fft::FastDiv per;
    int nx;
    __device__ XColumns(int tasks, int nx_) : per(tasks), nx(nx_) {}
    __device__ __forceinline__ int operator()(int idx, int &t) const
    {
        const int z = idx % KC;
        const int c = per(idx / KC, t);
        return c * nx * KC + z;
    }
};
}  // namespace

template <int KC, int NT, bool GREEN>
__global__ void __launch_bounds__(NT) x_green_kernel(FftAxis ax, float2 *spec, const float4 *gk, int64_t Mh,
                                                     GreenGeom g)
{
    extern __shared__ char lds[];
    float2 *buf = reinterpret_cast<float2 *>(lds);       // [11][Nx][KC]
    const int Nx = ax.n, Nzh = g.Nz / 2 + 1;
    float2 *tw = buf + 11 * Nx * KC;
    unsigned short *loc = reinterpret_cast<unsigned short *>(tw + Nx);
    const int nchunk = (Nzh + KC - 1) / KC;
    const int blk = xcd_remap(blockIdx.x, gridDim.x);
    const int ky = blk / nchunk, kz0 = (blk % nchunk) * KC;
    for (int i = threadIdx.x; i < Nx; i += NT) { tw[i] = ax.tw[i]; loc[i] = ax.loc[i]; }
    const int total = 11 * Nx * KC;
    const fft::FastDiv by_x(Nx);
    const int64_t xs = (int64_t)g.Ny * Nzh, at0 = (int64_t)ky * Nzh + kz0;
    constexpr int LOADS = 8;
    for (int i0 = 0; i0 < total; i0 += NT * LOADS) {
        float2 v[LOADS];
#pragma unroll
        for (int u = 0; u < LOADS; ++u) {
            const int i = i0 + u * NT + threadIdx.x, z = i % KC;
            int x;
            const int c = by_x(i / KC, x);
            v[u] = (i < total && kz0 + z < Nzh) ? spec[c * Mh + x * xs + at0 + z] : make_float2(0.f, 0.f);
        }
#pragma unroll
        for (int u = 0; u < LOADS; ++u) {
            const int i = i0 + u * NT + threadIdx.x;
            if (GREEN) {
                if (i < total) buf[i] = v[u];
            } else {
                int x;
                const int c = by_x(i / KC, x);
                if (i < total) buf[(c * Nx + ax.loc[x]) * KC + i % KC] = v[u];
            }
        }
    }
    __syncthreads();
    auto columns = [&](int tasks) { return XColumns<KC>(tasks, Nx); };
    if (GREEN) {
        fft::transform<false, NT>(buf, ax, 11 * KC, columns, KC, tw);
        for (int pt = threadIdx.x; pt < Nx * KC; pt += NT) {
            const int kx = pt / KC, z = pt % KC, k = kz0 + z;
            if (k >= Nzh) continue;
            float2 *p = buf + loc[kx] * KC + z;
            float2 v[11];
#pragma unroll
            for (int c = 0; c < 11; ++c) v[c] = p[c * Nx * KC];
            green_update(g, gk, kx, ky, k, v);
#pragma unroll
            for (int c = 0; c < 11; ++c) p[c * Nx * KC] = v[c];
        }
        __syncthreads();
    }
    fft::transform<true, NT>(buf, ax, 11 * KC, columns, KC, tw);
    for (int i = threadIdx.x; i < total; i += NT) {
        const int z = i % KC;
        int x;
        const int c = by_x(i / KC, x);
        if (kz0 + z < Nzh) spec[c * Mh + x * xs + at0 + z] = buf[i];
    }
}

// ------------------------------------------------------------------ launch
namespace {
constexpr int XKC = 4;
constexpr size_t LDS_MAX = 160 * 1024;

size_t yz_lds(int Ny, int Nz)
{
    const size_t rows = (Ny + 1) / 2 * 2, nzh = Nz / 2 + 1;
    return rows * nzh * sizeof(float2) + (size_t)(Ny + Nz) * (sizeof(float2) + sizeof(unsigned short));
}
size_t x_lds(int Nx) { return (size_t)Nx * (11 * XKC * sizeof(float2) + sizeof(float2) + sizeof(unsigned short)); }

// threads of a plane's workgroup, by its LDS: 256 for planes that leave room for ten on a CU, 512
// while two share one, 1024 for a plane that has the CU to itself
int yz_threads(size_t lds) { return lds <= 16 * 1024 ? 256 : (lds <= LDS_MAX / 2 ? 512 : 1024); }

template <class K>
hipError_t allow_lds(K kernel, size_t bytes)
{
    return hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)bytes);
}
}  // namespace

// Tables of the three axes when the grid's x columns fit in LDS (up to about 450 points); otherwise
// ctx->fft_x stays false and the 3-D library plans are used.  The planes are a matter of their own:
// those that fit LDS (up to about 200 points per axis) are transformed there, larger ones by the
// library's 2-D plans, from X_ALONE points along x on.  Wave part of a product that way and with the 3-D
// plans, us: 40 x 225 x 240 656 and 706, 48 x 200 x 216 514 and 680, 72 x 225 x 240 1205 and 1373, 80 x 256^2
// 1254 and 1335, 135 x 216 x 225 2940 and 4246, 200^3 1813 and 2039, 225^3 6879 and 8581, 256^3 4520 and 4642,
// 400 x 200^2 3934 and 5590; shorter axes gain nothing (24 x 225 x 240 473 and 470, 12 x 225 x 240 326 and 333).
constexpr int X_ALONE = 40;
int fft_init(fsd_ctx *ctx)
{
    const int n[3] = {ctx->pse.Nx, ctx->pse.Ny, ctx->pse.Nz};
    ctx->fft_x = ctx->fft_yz = false;
    const bool planes = yz_lds(n[1], n[2]) <= LDS_MAX;
    if (x_lds(n[0]) > LDS_MAX || (!planes && n[0] < X_ALONE)) return 0;
    const int total = n[0] + n[1] + n[2];
    std::vector<float2> tw(total);
    std::vector<unsigned short> loc(total);
    FftAxis ax[3];
    for (int a = 0, o = 0; a < 3; o += n[a], ++a) {
        ax[a].n = n[a];
        if (!fft::split(n[a], &ax[a].ns, ax[a].f)) return 0;
        for (int k = 0; k < n[a]; ++k) {
            const double t = -2.0 * 3.14159265358979323846 * k / n[a];
            tw[o + k] = make_float2((float)std::cos(t), (float)std::sin(t));
            loc[o + k] = (unsigned short)fft::place_of(n[a], ax[a].ns, ax[a].f, k);
        }
    }
    FSD_HIP(hipMalloc(&ctx->d_fft_tw, sizeof(float2) * total));
    FSD_HIP(hipMalloc(&ctx->d_fft_loc, sizeof(unsigned short) * total));
    FSD_HIP(hipMemcpy(ctx->d_fft_tw, tw.data(), sizeof(float2) * total, hipMemcpyHostToDevice));
    FSD_HIP(hipMemcpy(ctx->d_fft_loc, loc.data(), sizeof(unsigned short) * total, hipMemcpyHostToDevice));
    for (int a = 0, o = 0; a < 3; o += n[a], ++a) {
        ax[a].tw = ctx->d_fft_tw + o;
        ax[a].loc = ctx->d_fft_loc + o;
        ctx->fft_axis[a] = ax[a];
    }
    for (auto k : {yz_forward_kernel<256>, yz_forward_kernel<512>, yz_forward_kernel<1024>})
        FSD_HIP(allow_lds(k, LDS_MAX));
    for (auto k : {yz_inverse_kernel<256>, yz_inverse_kernel<512>, yz_inverse_kernel<1024>})
        FSD_HIP(allow_lds(k, LDS_MAX));
    FSD_HIP(allow_lds(x_green_kernel<XKC, 256, true>, LDS_MAX));
    FSD_HIP(allow_lds(x_green_kernel<XKC, 256, false>, LDS_MAX));
    if (!planes) {
        const int rc = fft_plans_2d(ctx);
        if (rc) return rc;
    }
    ctx->fft_x = true;
    ctx->fft_yz = planes;
    return 0;
}

static YzArgs yz_args(const fsd_ctx *ctx)
{
    YzArgs a;
    a.y = ctx->fft_axis[1];
    a.z = ctx->fft_axis[2];
    a.Nx = ctx->pse.Nx; a.Ny = ctx->pse.Ny; a.Nz = ctx->pse.Nz;
    a.Nzh = a.Nz / 2 + 1;
    a.zpairs = (a.Ny + 1) / 2;
    a.pz = grid_pitch(ctx);
    return a;
}

static int library_result(fsd_ctx *ctx, const char *failed)
{
    if (!failed) return 0;
    ctx->err = failed;
    return FSD_E_HIP;
}

// (y, z) transform of the 11 grids in d_grid into d_spec
int k_fft_yz_forward(fsd_ctx *ctx)
{
    if (!ctx->fft_yz) return library_result(ctx, ctx->fft2.forward(ctx->d_grid, ctx->d_spec));
    const YzArgs a = yz_args(ctx);
    const size_t lds = yz_lds(a.Ny, a.Nz);
    const dim3 grid(11 * a.Nx);
    switch (yz_threads(lds)) {
        case 256: hipLaunchKernelGGL(yz_forward_kernel<256>, grid, dim3(256), lds, ctx->stream, a, ctx->d_grid, ctx->d_spec); break;
        case 512: hipLaunchKernelGGL(yz_forward_kernel<512>, grid, dim3(512), lds, ctx->stream, a, ctx->d_grid, ctx->d_spec); break;
        default: hipLaunchKernelGGL(yz_forward_kernel<1024>, grid, dim3(1024), lds, ctx->stream, a, ctx->d_grid, ctx->d_spec);
    }
    FSD_HIP(hipGetLastError());
    return 0;
}

int k_fft_yz_inverse(fsd_ctx *ctx)
{
    if (!ctx->fft_yz) return library_result(ctx, ctx->fft2.inverse(ctx->d_spec, ctx->d_grid));
    const YzArgs a = yz_args(ctx);
    const size_t lds = yz_lds(a.Ny, a.Nz);
    const dim3 grid(11 * a.Nx);
    switch (yz_threads(lds)) {
        case 256: hipLaunchKernelGGL(yz_inverse_kernel<256>, grid, dim3(256), lds, ctx->stream, a, ctx->d_spec, ctx->d_grid); break;
        case 512: hipLaunchKernelGGL(yz_inverse_kernel<512>, grid, dim3(512), lds, ctx->stream, a, ctx->d_spec, ctx->d_grid); break;
        default: hipLaunchKernelGGL(yz_inverse_kernel<1024>, grid, dim3(1024), lds, ctx->stream, a, ctx->d_spec, ctx->d_grid);
    }
    FSD_HIP(hipGetLastError());
    return 0;
}

// x direction of the spectra in d_spec: forward, Green's function and inverse, or the inverse alone
int k_fft_x(fsd_ctx *ctx, bool green)
{
    const fsd_pse_info &ps = ctx->pse;
    const GreenGeom gg{ps.Nx, ps.Ny, ps.Nz, ctx->box, ctx->p.xi, ps.eta, k_twopi(ctx)};
    const int nchunk = (ps.Nz / 2 + 1 + XKC - 1) / XKC;
    const dim3 grid(ps.Ny * nchunk);
    const size_t lds = x_lds(ps.Nx);
    if (green)
        hipLaunchKernelGGL((x_green_kernel<XKC, 256, true>), grid, dim3(256), lds, ctx->stream, ctx->fft_axis[0],
                           ctx->d_spec, ctx->d_gridk, (int64_t)ctx->Mh, gg);
    else
        hipLaunchKernelGGL((x_green_kernel<XKC, 256, false>), grid, dim3(256), lds, ctx->stream, ctx->fft_axis[0],
                           ctx->d_spec, ctx->d_gridk, (int64_t)ctx->Mh, gg);
    FSD_HIP(hipGetLastError());
    return 0;
}
