// PSE far-field grand mobility on MI355X.
//
//   wave space:  particle records -> tile-gather spreading (no global atomics)
//                -> real-to-complex transform (11 fields, k_fft.hip), Green's function
//                on the half spectrum and back -> per-particle contraction;
//   real space:  table-interpolated FTS pair sum, 16 lanes per particle, with an
//                epilogue that adds the wave-space result, converts the velocity
//                gradient to (W, E) and writes the generalised velocity.
// Restates Mobility.cu:131-1542 and Helper_Mobility.cu:88-410.
#include <algorithm>

#include "fsd_internal.h"
#include "green.h"

#define FSD_TILE 8

// ------------------------------------------------------------- k vectors
// Mobility_SetGridk_kernel (Helper_Mobility.cu:351-410) on the R2C half
// spectrum: index (i, j, k) with k in [0, Nz/2].
__global__ void gridk_kernel(float4 *gk, int Nx, int Ny, int Nz, BoxF b, float xi, float eta, float twopi_k)
{
    const int Nzh = Nz / 2 + 1;
    const int64_t Mh = (int64_t)Nx * Ny * Nzh;
    int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (tid >= Mh) return;
    int i = (int)(tid / ((int64_t)Ny * Nzh));
    int j = (int)((tid / Nzh) % Ny);
    int k = (int)(tid % Nzh);
    gk[tid] = gridk_value(i, j, k, Nx, Ny, Nz, b, xi, eta, twopi_k);
}

// 2 pi of the k vectors: the reference's constant 3.1416926536 with parity
// (Helper_Mobility.cu:389-391)
float k_twopi(const fsd_ctx *ctx)
{
    return (float)(2.0 * (ctx->p.parity ? 3.1416926536 : 3.14159265358979323846));
}

int k_gridk(fsd_ctx *ctx)
{
    hipLaunchKernelGGL(gridk_kernel, dim3(nblk(ctx->Mh, 256)), dim3(256), 0, ctx->stream, ctx->d_gridk, ctx->pse.Nx,
                       ctx->pse.Ny, ctx->pse.Nz, ctx->box, ctx->p.xi, ctx->pse.eta, k_twopi(ctx));
    FSD_HIP(hipGetLastError());
    return 0;
}

// ------------------------------------------------- force + couplet records
// per slot one 64-byte record (half a cache line): position, F (3), the stresslet S (xx, xy, xz, yz, yy)
// and w = -T/2, the couplet's antisymmetric part (Mobility_TS2C_kernel, Helper_Mobility.cu:294-336)
__device__ __forceinline__ void write_record(const float *gF, int N, int id, float4 p, float4 *r)
{
    const float *f = gF + 6 * (int64_t)id;
    const float *s = gF + 6 * (int64_t)N + 5 * (int64_t)id;
    r[0] = make_float4(p.x, p.y, p.z, f[0]);
    r[1] = make_float4(f[1], f[2], s[0], s[1]);
    r[2] = make_float4(s[2], s[3], s[4], -0.5f * f[3]);
    r[3] = make_float4(-0.5f * f[4], -0.5f * f[5], 0.f, 0.f);
}

__global__ void fc_records_kernel(const float *gF, const float4 *pos, const int *order, int N, float4 *rec)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    const int id = order ? order[i] : i;
    write_record(gF, N, id, pos[id], rec + 4 * (int64_t)i);
}

// ------------------------------------------------- spreading set-up (per step)
// Stencil origin exactly as Mobility.cu:203-225 (float fraction, truncation);
// particles are then counting-sorted by the grid cell of their (wrapped)
// origin, ascending inside a cell, so spreading and contraction
// can find the particles of any block of origin cells as contiguous runs.
//
// Particles stand by slot, their place in the neighbour list's cell order: what the wave part and
// the real-space sum read of a particle's surroundings lies close together.
//
// Four launches (origins, counts and the product's records; scan within chunks; scatter; order and
// starts), each a few dependent loads long, so their number is what they cost (eight took 27 us at
// N = 4072): the counting atomics give each particle its place in its cell, the last launch leaves
// the counts zero, and the chunks' offsets are summed where they are used.
__global__ void stencil_origin_kernel(const float4 *pos, const int *order, int N, BoxF b, int Nx, int Ny, int Nz,
                                      int P, const float *gF, float4 *rec, float4 *spos, int *orig, int *ocell,
                                      int *orank, int *ocount)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    const int id = order ? order[i] : i;
    float4 p = pos[id];
    spos[i] = make_float4(p.x, p.y, p.z, __int_as_float(id));
    float fx, fy, fz;
    box_make_fraction(b, p.x, p.y, p.z, fx, fy, fz);
    fx *= (float)Nx; fy *= (float)Ny; fz *= (float)Nz;
    int x = (int)fx, y = (int)fy, z = (int)fz;
    const int Pd2 = P / 2;
    int ox = x - Pd2 + 1 - (P % 2) * ((fx - (float)x) < 0.5f);
    int oy = y - Pd2 + 1 - (P % 2) * ((fy - (float)y) < 0.5f);
    int oz = z - Pd2 + 1 - (P % 2) * ((fz - (float)z) < 0.5f);
    orig[3 * i] = ox; orig[3 * i + 1] = oy; orig[3 * i + 2] = oz;
    int wx = ((ox % Nx) + Nx) % Nx, wy = ((oy % Ny) + Ny) % Ny, wz = ((oz % Nz) + Nz) % Nz;
    const int c = (wx * Ny + wy) * Nz + wz;
    ocell[i] = c;
    orank[i] = atomicAdd(&ocount[c], 1);
    if (gF) write_record(gF, N, id, p, rec + 4 * (int64_t)i);
}

// offset of the chunks before chunk c (part: totals, or the offsets themselves), for the whole block
__device__ __forceinline__ int chunk_offset(const int *part, bool totals, int c)
{
    if (!totals) return part[c];
    __shared__ int s_w[4];
    int s = 0;
    for (int q = threadIdx.x; q < c; q += 256) s += part[q];
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if ((threadIdx.x & 63) == 0) s_w[threadIdx.x >> 6] = s;
    __syncthreads();
    return s_w[0] + s_w[1] + s_w[2] + s_w[3];
}

__global__ void __launch_bounds__(256) ocell_scatter_kernel(const int *ocell, const int *orank, int N, const int *start,
                                                            const int *part, int nc, bool totals, int *list)
{
    // offsets of all chunks (at most SCAN_SELF when they are not given): four to a thread
    __shared__ int s_off[SCAN_SELF], s_w[4];
    const int lt = threadIdx.x, i = blockIdx.x * blockDim.x + lt;
    const int c = i < N ? ocell[i] : 0, r = i < N ? orank[i] : 0;
    const int st = start[c];
    if (totals) {
        int v[4], s = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            v[k] = 4 * lt + k < nc ? part[4 * lt + k] : 0;
            s += v[k];
        }
        int inc = s;
        for (int o = 1; o < 64; o <<= 1) {
            const int y = __shfl_up(inc, o, 64);
            if ((lt & 63) >= o) inc += y;
        }
        if ((lt & 63) == 63) s_w[lt >> 6] = inc;
        __syncthreads();
        int pre = inc - s;
        for (int w = 0; w < (lt >> 6); ++w) pre += s_w[w];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            s_off[4 * lt + k] = pre;
            pre += v[k];
        }
        __syncthreads();
    }
    if (i < N) list[st + (totals ? s_off[c / SCAN_CHUNK] : part[c / SCAN_CHUNK]) + r] = i;
}

// orders the cells' slots, completes their starts and clears the counts
__global__ void __launch_bounds__(256) ocell_sort_kernel(int *start, int *count, const int *part, bool totals,
                                                         int ncell, int N, int *list)
{
    static_assert(SCAN_CHUNK % 256 == 0, "a block's cells lie in one chunk");
    const int c = blockIdx.x * 256 + threadIdx.x;
    const int n = c < ncell ? count[c] : 0, s0 = c < ncell ? start[c] : 0;
    const int s = s0 + chunk_offset(part, totals, blockIdx.x * 256 / SCAN_CHUNK), e = s + n;
    if (c >= ncell) return;
    start[c] = s;
    count[c] = 0;
    if (c == ncell - 1) start[ncell] = N;
    for (int a = s + 1; a < e; ++a) {
        int key = list[a], q = a - 1;
        while (q >= s && list[q] > key) { list[q + 1] = list[q]; --q; }
        list[q + 1] = key;
    }
}

// the order of the slots
static const int *slot_order(const fsd_ctx *ctx)
{
    return (ctx->nlist_valid && ctx->use_cells) ? ctx->d_cell_list : nullptr;
}

int k_setup_spread(fsd_ctx *ctx, const float4 *pos, const float *gF)
{
    const int N = ctx->N, M = ctx->M;
    if (!ctx->ocount_zero) FSD_HIP(hipMemsetAsync(ctx->d_ocount, 0, sizeof(int) * M, ctx->stream));
    ctx->ocount_zero = false;
    hipLaunchKernelGGL(stencil_origin_kernel, dim3(nblk(N, 256)), dim3(256), 0, ctx->stream, pos, slot_order(ctx), N,
                       ctx->box, ctx->pse.Nx, ctx->pse.Ny, ctx->pse.Nz, ctx->pse.P, gF, ctx->d_rec, ctx->d_spos,
                       ctx->d_porig, ctx->d_ocell, ctx->d_orank, ctx->d_ocount);
    bool totals;
    const int *part = ctx->d_scan_tmp, nc = scan_excl_chunks(M);
    if (scan_chunked(ctx, ctx->d_ocount, ctx->d_ostart, M, ctx->d_scan_tmp, &totals)) return FSD_E_HIP;
    hipLaunchKernelGGL(ocell_scatter_kernel, dim3(nblk(N, 256)), dim3(256), 0, ctx->stream, ctx->d_ocell, ctx->d_orank,
                       N, ctx->d_ostart, part, nc, totals, ctx->d_olist);
    hipLaunchKernelGGL(ocell_sort_kernel, dim3(nblk(M, 256)), dim3(256), 0, ctx->stream, ctx->d_ostart, ctx->d_ocount,
                       part, totals, M, N, ctx->d_olist);
    FSD_HIP(hipGetLastError());
    ctx->ocount_zero = true;
    ctx->spread_valid = true;
    ctx->spread_pos = (const float *)pos;
    return 0;
}

// F and the couplet's stored components XX XY XZ YZ YY YX ZX ZY of a record: the 11 grid fields
__device__ __forceinline__ void record_fields(const float4 q[4], float4 f[3])
{
    const float sxy = q[1].w, sxz = q[2].x, syz = q[2].y, wx = q[2].w, wy = q[3].x, wz = q[3].y;
    f[0] = make_float4(q[0].w, q[1].x, q[1].y, q[1].z);
    f[1] = make_float4(sxy + wz, sxz - wy, syz + wx, q[2].z);
    f[2] = make_float4(sxy - wz, sxz + wy, syz - wx, 0.f);
}

// ------------------------------------------------------------ spreading
struct SpreadGeom {
    int Nx, Ny, Nz, P, tile, tnx, tny, tnz;
    int pz;                    // row length of the grids in memory (grid_pitch)
    float hx, hy, hz, Lx2, Ly2, Lz2, xy;
    float prefac, expfac;
};

static SpreadGeom spread_geom(const fsd_ctx *ctx)
{
    const fsd_pse_info &ps = ctx->pse;
    SpreadGeom g;
    g.Nx = ps.Nx; g.Ny = ps.Ny; g.Nz = ps.Nz; g.P = ps.P; g.tile = ctx->tile;
    g.tnx = ctx->tiles[0]; g.tny = ctx->tiles[1]; g.tnz = ctx->tiles[2];
    g.pz = grid_pitch(ctx);
    g.hx = ps.gridh_x; g.hy = ps.gridh_y; g.hz = ps.gridh_z;
    g.Lx2 = ctx->box.Lx / 2.0f; g.Ly2 = ctx->box.Ly / 2.0f; g.Lz2 = ctx->box.Lz / 2.0f; g.xy = ctx->box.xy;
    g.prefac = ps.prefac; g.expfac = ps.expfac;
    return g;
}

// The origin cells whose stencils reach a tile [t0, t0 + tile) on one axis are
// t0 - P + 1 .. t0 + tile - 1 (wrapped): `halo_axis` lists them once each
// (fewer when the grid is shorter than the list) and returns the count.
__device__ int halo_axis(int t0, int tile, int P, int n, int *list)
{
    int cnt = 0;
    for (int o = t0 - P + 1; o <= t0 + tile - 1; ++o) {
        const int w = ((o % n) + n) % n;
        bool seen = false;
        for (int q = 0; q < cnt; ++q) seen |= (list[q] == w);
        if (!seen) list[cnt++] = w;
    }
    return cnt;
}

// One workgroup per tile of TILE^3 grid points, one thread per point.  The
// particles whose origin lies in the tile's halo of origin cells (the exact
// set whose stencils can reach the tile) are found as runs of the
// origin-cell-sorted list and streamed through LDS in chunks; every point
// accumulates its 11 fields in registers and is written once (no atomics).
#define SP_CH 256
#define SP_MAXAX 32
__global__ void __launch_bounds__(512) spread_kernel(SpreadGeom g, const int *orig, const float4 *rec, const int *ostart,
                                                     const int *olist, float *grid, int64_t M)
{
    __shared__ int s_ax[3][SP_MAXAX];
    __shared__ int s_nax[3];
    __shared__ int s_zrun[SP_MAXAX][2];   // z runs: [first cell, one past last cell)
    __shared__ int s_nzrun;
    __shared__ int s_seg_beg[SP_MAXAX * SP_MAXAX * 2];
    __shared__ int s_seg_off[SP_MAXAX * SP_MAXAX * 2 + 1];
    __shared__ int s_nseg;
    __shared__ int s_o[SP_CH][3];
    __shared__ float s_p[SP_CH][3];
    __shared__ float4 s_r[SP_CH][3];

    const int tile_id = blockIdx.x;
    const int tz_i = tile_id % g.tnz, ty_i = (tile_id / g.tnz) % g.tny, tx_i = tile_id / (g.tnz * g.tny);
    const int x0 = tx_i * g.tile, y0 = ty_i * g.tile, z0 = tz_i * g.tile;
    const int lt = threadIdx.x;
    const int lx = lt / (g.tile * g.tile), ly = (lt / g.tile) % g.tile, lz = lt % g.tile;
    const int gx = x0 + lx, gy = y0 + ly, gz = z0 + lz;
    const bool inside = (gx < g.Nx) && (gy < g.Ny) && (gz < g.Nz);

    if (lt < 3) {
        const int t0 = (lt == 0) ? x0 : (lt == 1) ? y0 : z0;
        const int n = (lt == 0) ? g.Nx : (lt == 1) ? g.Ny : g.Nz;
        s_nax[lt] = halo_axis(t0, g.tile, g.P, n, s_ax[lt]);
    }
    __syncthreads();
    if (lt == 0) {
        // group the z cells into runs of consecutive indices
        int nr = 0;
        for (int q = 0; q < s_nax[2]; ++q) {
            const int z = s_ax[2][q];
            if (nr > 0 && s_zrun[nr - 1][1] == z) s_zrun[nr - 1][1] = z + 1;
            else { s_zrun[nr][0] = z; s_zrun[nr][1] = z + 1; ++nr; }
        }
        s_nzrun = nr;
        s_nseg = s_nax[0] * s_nax[1] * nr;
    }
    __syncthreads();
    const int nseg = s_nseg, nzr = s_nzrun, ny = s_nax[1];
    for (int sg = lt; sg < nseg; sg += blockDim.x) {
        const int zr = sg % nzr, xy = sg / nzr;
        const int x = s_ax[0][xy / ny], y = s_ax[1][xy % ny];
        const int cbase = (x * g.Ny + y) * g.Nz;
        const int b0 = ostart[cbase + s_zrun[zr][0]], b1 = ostart[cbase + s_zrun[zr][1]];
        s_seg_beg[sg] = b0;
        s_seg_off[sg + 1] = b1 - b0;
    }
    __syncthreads();
    if (lt == 0) {
        s_seg_off[0] = 0;
        for (int sg = 0; sg < nseg; ++sg) s_seg_off[sg + 1] += s_seg_off[sg];
    }
    __syncthreads();
    const int total = s_seg_off[nseg];

    float acc[11];
#pragma unroll
    for (int c = 0; c < 11; ++c) acc[c] = 0.f;

    for (int base = 0; base < total; base += SP_CH) {
        const int nch = min(SP_CH, total - base);
        __syncthreads();
        if (lt < nch) {
            const int q = base + lt;
            int lo = 0, hi = nseg - 1;          // segment sg with off[sg] <= q < off[sg + 1]
            while (lo < hi) {
                const int mid = (lo + hi + 1) >> 1;
                if (s_seg_off[mid] <= q) lo = mid; else hi = mid - 1;
            }
            const int i = olist[s_seg_beg[lo] + (q - s_seg_off[lo])];
            s_o[lt][0] = orig[3 * i]; s_o[lt][1] = orig[3 * i + 1]; s_o[lt][2] = orig[3 * i + 2];
            float4 r[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) r[k] = rec[4 * (int64_t)i + k];
            s_p[lt][0] = r[0].x; s_p[lt][1] = r[0].y; s_p[lt][2] = r[0].z;
            record_fields(r, s_r[lt]);
        }
        __syncthreads();
        if (inside) {
            for (int q = 0; q < nch; ++q) {
                int tx = gx - s_o[q][0]; tx += (tx < 0) ? g.Nx : 0; tx -= (tx >= g.Nx) ? g.Nx : 0;
                int ty = gy - s_o[q][1]; ty += (ty < 0) ? g.Ny : 0; ty -= (ty >= g.Ny) ? g.Ny : 0;
                int tz = gz - s_o[q][2]; tz += (tz < 0) ? g.Nz : 0; tz -= (tz >= g.Nz) ? g.Nz : 0;
                if (tx < g.P && ty < g.P && tz < g.P) {
                    // unwrapped grid node of this stencil point, relative to the particle
                    const float uy = g.hy * (float)(s_o[q][1] + ty) - g.Ly2;
                    const float dx = g.hx * (float)(s_o[q][0] + tx) - g.Lx2 + g.xy * uy - s_p[q][0];
                    const float dy = uy - s_p[q][1];
                    const float dz = g.hz * (float)(s_o[q][2] + tz) - g.Lz2 - s_p[q][2];
                    const float w = g.prefac * __expf(-g.expfac * (dx * dx + dy * dy + dz * dz));
                    const float4 r0 = s_r[q][0], r1 = s_r[q][1], r2 = s_r[q][2];
                    acc[0] += w * r0.x; acc[1] += w * r0.y; acc[2] += w * r0.z;
                    acc[3] += w * r0.w; acc[4] += w * r1.x; acc[5] += w * r1.y; acc[6] += w * r1.z;
                    acc[7] += w * r1.w; acc[8] += w * r2.x; acc[9] += w * r2.y; acc[10] += w * r2.z;
                }
            }
        }
    }
    if (inside) {
        const int64_t id = ((int64_t)gx * g.Ny + gy) * g.pz + gz;
#pragma unroll
        for (int c = 0; c < 11; ++c) grid[c * M + id] = acc[c];
    }
}

// Spreading for the usual stencil (P = 6) on the matrix cores: one workgroup per tile of 8^3
// nodes, one wave per 4 x 4 columns by 4 nodes along z.
//
// A node lies in the stencils of ~19 spheres at volume fraction 0.45 and each adds 11
// products.  For the 16 columns of a wave and one z that is a matrix product,
//   grid[field, column] = sum over spheres rec[field, sphere] (e[sphere, column] w[sphere, z]),
// with e the Gaussian along x and y (zero outside the sphere's stencil) and w its factor along
// z: mfma 16x16x4 in FP32 takes four spheres at a time, fields (11 of 16 rows) by columns.  A
// lane forms one e per step and multiplies it by the four w, so the four products of a step
// share it and the records.  Per node this takes 64 spheres (those that reach any of the 4 x 4
// x 4 nodes), of which 19 count, at twice the VALU's rate.  The same sums on the VALU were bound
// by lanes that waited for the longest of 36 short runs of spheres (34.6 us per product at N =
// 32768) or, with those runs merged, by LDS bank conflicts (each lane its own sphere: 34.6 us); this form takes
// 21 us (13 us at N = 4072), of which half are the dependent loads before the products and the
// stores after them.
// The tile's halo of 13^3 origin cells is staged in LDS.  Its spheres are in the order of buckets
// (x, third of z, y): a wave of the lower nodes needs the first two thirds, one of the upper
// nodes the last two, so its spheres are 18 runs of nine buckets each, which it lists.  A halo of
// more than SP2_CAP spheres is staged in parts.  Every node sums its spheres in bucket order and is
// written once (no atomics).
#define SP2_CAP 256
typedef float mfma_f4 __attribute__((ext_vector_type(4)));
template <int PP>
__global__ void __launch_bounds__(512, 6) spread_mfma_kernel(SpreadGeom g, const int *orig, const float4 *rec,
                                                             const int *ostart, const int *olist, float *grid, int64_t M)
{
    constexpr int T = 8, BL = 4, H = T + PP - 1, HB = BL + PP - 1, NT = 512, NW = NT / 64;
    constexpr int ZP[4] = {0, H - HB, HB, H};     // thirds of the halo's z cells: 4, 5 and 4 of them
    constexpr int NB = 3 * H * H;                 // buckets
    static_assert(NB <= NT && SP2_CAP <= NT, "a bucket and a staged sphere per thread");
    __shared__ int s_base[NB + 1];                // exclusive scan of the buckets' counts
    __shared__ int s_beg[2][NB];                  // olist position of a bucket's two pieces (z may wrap) ...
    __shared__ int s_first[NB];                   // ... and the count of the first
    __shared__ int s_wsum[NW];
    __shared__ float4 s_c[SP2_CAP];               // scaled offsets of the tile's first column (x, y), its columns
    __shared__ float4 s_z[SP2_CAP][2];            // factors along z
    __shared__ float s_r[SP2_CAP * 12 + 4];       // fields; rows 12 to 15 of a product read past a sphere's 12
    __shared__ unsigned short s_list[NW][SP2_CAP + 8];

    const int tile_id = xcd_remap(blockIdx.x, gridDim.x);
    const int tz_i = tile_id % g.tnz, ty_i = (tile_id / g.tnz) % g.tny, tx_i = tile_id / (g.tnz * g.tny);
    const int x0 = tx_i * T, y0 = ty_i * T, z0 = tz_i * T;
    const int lt = threadIdx.x, lane = lt & 63, wv = lt >> 6;
    auto wrap = [](int v, int n) {
        v += (v < 0) ? n : 0;
        v -= (v >= n) ? n : 0;
        return v - ((v >= n) ? n : 0);
    };
    // a third's cells: n0 from cell za on, the others from cell 0 on (grids have at least 8 points)
    auto third = [&](int p, int &za, int &n0) {
        za = wrap(z0 - (PP - 1) + ZP[p], g.Nz);
        n0 = min(ZP[p + 1] - ZP[p], g.Nz - za);
    };
    int cnt = 0;
    if (lt < NB) {
        const int hx = lt / (3 * H), r = lt - hx * (3 * H), p = r / H, hy = r - p * H;
        const int c = (wrap(x0 - (PP - 1) + hx, g.Nx) * g.Ny + wrap(y0 - (PP - 1) + hy, g.Ny)) * g.Nz;
        int za, n0;
        third(p, za, n0);
        const int nz = ZP[p + 1] - ZP[p];
        const int b0 = ostart[c + za], e0 = ostart[c + za + n0];
        const int b1 = n0 < nz ? ostart[c] : 0, e1 = n0 < nz ? ostart[c + nz - n0] : 0;
        s_beg[0][lt] = b0;
        s_beg[1][lt] = b1;
        s_first[lt] = e0 - b0;
        cnt = (e0 - b0) + (e1 - b1);
    }
    int inc = cnt;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int v = __shfl_up(inc, o, 64);
        if (lane >= o) inc += v;
    }
    if (lane == 63) s_wsum[wv] = inc;
    __syncthreads();
    int before = 0, total = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
        before += w < wv ? s_wsum[w] : 0;
        total += s_wsum[w];
    }
    if (lt < NB) s_base[lt] = before + inc - cnt;
    if (lt == 0) s_base[NB] = total;
    __syncthreads();

    // lengths in units in which the Gaussian is 2^-(d^2)
    const float unit = sqrtf(g.expfac * 1.44269504088896341f);
    const int col = lane & 15, quad = lane >> 4;
    const int bx = (wv >> 1 & 1) * BL, by = (wv & 1) * BL, half = wv >> 2;   // the wave's nodes
    const int lx = bx + col / BL, ly = by + col % BL;
    const float ay = unit * (g.hy * (float)ly);
    const float ax = unit * (g.hx * (float)lx) + g.xy * ay;
    const unsigned here = (1u << lx) | (1u << (T + ly));
    mfma_f4 acc[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) acc[k] = mfma_f4{0.f, 0.f, 0.f, 0.f};

    for (int base = 0; base < total; base += SP2_CAP) {
        if (base) __syncthreads();                // the part before is done with
        const int p = base + lt;
        if (lt < SP2_CAP && p < total) {
            // the bucket by binary search over the scan (the last one whose base is not above the position
            // holds it), then the index and the records
            int lo = 0, hi = NB - 1;
#pragma unroll
            for (int step = 0; step < 9; ++step) {   // 2^9 > NB
                const int mid = (lo + hi + 1) >> 1;
                const bool right = lo < hi && s_base[mid] <= p;
                hi = (lo < hi && !right) ? mid - 1 : hi;
                lo = right ? mid : lo;
            }
            const int o = p - s_base[lo], n1 = s_first[lo];
            const bool second = o >= n1;
            const int i = olist[second ? s_beg[1][lo] + (o - n1) : s_beg[0][lo] + o];
            const int ox = orig[3 * i], oy = orig[3 * i + 1], oz = orig[3 * i + 2];
            float4 r[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) r[k] = rec[4 * (int64_t)i + k];
            const float4 q = r[0];
            // the sphere's origin is the halo cell (hc) up to the period, so a node at local (lx, ly, lz)
            // of its stencil is node o + (P - 1) - hc + l: with the node's position
            // h (o + P - 1 - hc) - L/2 + h l, its offset from the sphere is c + h l
            const int hxc = lo / (3 * H), rb = lo - hxc * (3 * H), zp = rb / H, hyc = rb - zp * H;
            int za, n0;
            third(zp, za, n0);
            const int wz = ((oz % g.Nz) + g.Nz) % g.Nz;
            const int hzc = ZP[zp] + (second ? n0 + wz : wz - za);
            const float cy = g.hy * (float)(oy + (PP - 1) - hyc) - g.Ly2;
            const float cx = g.hx * (float)(ox + (PP - 1) - hxc) - g.Lx2 - q.x + g.xy * cy;
            const float cz = g.hz * (float)(oz + (PP - 1) - hzc) - g.Lz2 - q.z;
            float w[T];
#pragma unroll
            for (int k = 0; k < T; ++k) {
                const float dz = unit * (cz + g.hz * (float)k);
                const int s = k + (PP - 1) - hzc;     // node of the stencil
                w[k] = (s >= 0 && s < PP) ? g.prefac * __builtin_amdgcn_exp2f(-(dz * dz)) : 0.f;
            }
            // columns of the tile inside the stencil: hc - P + 1 .. hc along each axis
            const unsigned six = (1u << PP) - 1u;
            const unsigned mx = ((six << hxc) >> (PP - 1)) & 0xffu, my = ((six << hyc) >> (PP - 1)) & 0xffu;
            s_c[lt] = make_float4(unit * cx, unit * (cy - q.y), __uint_as_float(mx | (my << T)), 0.f);
            s_z[lt][0] = make_float4(w[0], w[1], w[2], w[3]);
            s_z[lt][1] = make_float4(w[4], w[5], w[6], w[7]);
            record_fields(r, reinterpret_cast<float4 *>(s_r + 12 * lt));
        }
        // this wave's spheres of the part: lane k < 18 lists run k
        unsigned short *list = s_list[wv];
        int len = 0;
        {
            int b = 0, n = 0;
            if (lane < 2 * HB) {
                const int q = ((bx + (lane >> 1)) * 3 + half + (lane & 1)) * H + by;
                b = max(s_base[q] - base, 0);
                n = max(min(s_base[q + HB] - base, SP2_CAP) - b, 0);
            }
            int at = n;
#pragma unroll
            for (int o = 1; o < 32; o <<= 1) {
                const int v = __shfl_up(at, o, 64);
                if (lane >= o) at += v;
            }
            len = __shfl(at, 31, 64);
            at -= n;
            for (int k = 0; k < n; ++k) list[at + k] = (unsigned short)(b + k);
            if (lane < 8) list[len + lane] = 0;   // idle spheres of the last step
        }
        __syncthreads();
        for (int t0 = 0; t0 < len; t0 += 8) {
            const int t = t0 + quad, sa = list[t], sb = list[t + 4];
            const float4 ca = s_c[sa], cb = s_c[sb], za = s_z[sa][half], zb = s_z[sb][half];
            const float ra = s_r[12 * sa + col], rb = s_r[12 * sb + col];
            const float dxa = ca.x + ax, dya = ca.y + ay, dxb = cb.x + ax, dyb = cb.y + ay;
            const bool ina = (__float_as_uint(ca.z) & here) == here && t < len;
            const bool inb = (__float_as_uint(cb.z) & here) == here && t + 4 < len;
            const float ea = ina ? __builtin_amdgcn_exp2f(-(dxa * dxa + dya * dya)) : 0.f;
            const float eb = inb ? __builtin_amdgcn_exp2f(-(dxb * dxb + dyb * dyb)) : 0.f;
            acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(ra, ea * za.x, acc[0], 0, 0, 0);
            acc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(ra, ea * za.y, acc[1], 0, 0, 0);
            acc[2] = __builtin_amdgcn_mfma_f32_16x16x4f32(ra, ea * za.z, acc[2], 0, 0, 0);
            acc[3] = __builtin_amdgcn_mfma_f32_16x16x4f32(ra, ea * za.w, acc[3], 0, 0, 0);
            acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(rb, eb * zb.x, acc[0], 0, 0, 0);
            acc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(rb, eb * zb.y, acc[1], 0, 0, 0);
            acc[2] = __builtin_amdgcn_mfma_f32_16x16x4f32(rb, eb * zb.z, acc[2], 0, 0, 0);
            acc[3] = __builtin_amdgcn_mfma_f32_16x16x4f32(rb, eb * zb.w, acc[3], 0, 0, 0);
        }
    }
    // a lane holds fields 4 quad .. 4 quad + 3 of its column
    const int gx = x0 + lx, gy = y0 + ly, gz = z0 + 4 * half;
    if (gx >= g.Nx || gy >= g.Ny || gz >= g.Nz) return;
    const int64_t id = ((int64_t)gx * g.Ny + gy) * g.pz + gz;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int f = 4 * quad + q;
        if (f >= 11) break;
        // 16-byte aligned rows (grid_pitch), whose padding takes the rest: 82 us at 64 x 243 x 250 and N =
        // 2000, where rows of 250 floats, stored node by node in this lane order, took 209
        *reinterpret_cast<float4 *>(grid + (int64_t)f * M + id) = make_float4(acc[0][q], acc[1][q], acc[2][q], acc[3][q]);
    }
}

// ------------------------------------------------------------ Green kernel
__global__ void green_kernel(float2 *spec, const float4 *gk, int64_t Mh, GreenGeom g)
{
    int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= Mh) return;
    const int Nzh = g.Nz / 2 + 1;
    const int k = (int)(id % Nzh), j = (int)((id / Nzh) % g.Ny), i = (int)(id / ((int64_t)Nzh * g.Ny));
    float2 v[11];
#pragma unroll
    for (int c = 0; c < 11; ++c) v[c] = spec[c * Mh + id];
    green_update(g, gk, i, j, k, v);
#pragma unroll
    for (int c = 0; c < 11; ++c) spec[c * Mh + id] = v[c];
}

// ------------------------------------------------------------ contraction
// Mobility_WaveSpace_ContractU/D (Mobility.cu:503-841): one wavefront per
// particle, lanes over the (y, z) stencil pairs, loop over x.  Output per
// particle: u (3) then the gradient in the reference's transposed slots.
__global__ void __launch_bounds__(256) contract_kernel(SpreadGeom g, const float4 *spos, const int *orig,
                                                       const float *grid, int64_t M, int N, float quadw_prefac,
                                                       float *wave)
{
    const int wave_id = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int lane = threadIdx.x & 63;
    if (wave_id >= N) return;
    const int i = wave_id;
    const int ox = orig[3 * i], oy = orig[3 * i + 1], oz = orig[3 * i + 2];
    const float4 p = spos[i];
    float acc[11];
#pragma unroll
    for (int c = 0; c < 11; ++c) acc[c] = 0.f;
    const int P = g.P;
    for (int yz = lane; yz < P * P; yz += 64) {
        const int ty = yz / P, tz = yz % P;
        int y = oy + ty; const float uy = g.hy * (float)y - g.Ly2;
        int z = oz + tz; const float dz = g.hz * (float)z - g.Lz2 - p.z;
        const float dy = uy - p.y;
        y = ((y % g.Ny) + g.Ny) % g.Ny;
        z = ((z % g.Nz) + g.Nz) % g.Nz;
        for (int tx = 0; tx < P; ++tx) {
            int x = ox + tx;
            const float dx = g.hx * (float)x - g.Lx2 + g.xy * uy - p.x;
            x = ((x % g.Nx) + g.Nx) % g.Nx;
            const float w = quadw_prefac * __expf(-g.expfac * (dx * dx + dy * dy + dz * dz));
            const int64_t id = ((int64_t)x * g.Ny + y) * g.pz + z;
#pragma unroll
            for (int c = 0; c < 11; ++c) acc[c] += w * grid[c * M + id];
        }
    }
#pragma unroll
    for (int c = 0; c < 11; ++c)
        for (int o = 32; o > 0; o >>= 1) acc[c] += __shfl_xor(acc[c], o, 64);
    if (lane == 0) {
        float *w = wave + 11 * (int64_t)__float_as_int(p.w);
        w[0] = acc[0]; w[1] = acc[1]; w[2] = acc[2];
        // fields XX XY XZ YZ YY YX ZX ZY -> slots {XX, YX, ZX, ZY, YY, XY, XZ, YZ}
        w[3] = acc[3]; w[4] = acc[8]; w[5] = acc[9]; w[6] = acc[10];
        w[7] = acc[7]; w[8] = acc[4]; w[9] = acc[5]; w[10] = acc[6];
    }
}

// Tile form of the contraction: one workgroup per tile of TILE^3 origin
// cells stages the grid block [t0, t0 + TILE + P - 1)^3 of all 11 fields in
// LDS (coalesced loads, wrapped indices), then contracts the particles whose
// origin lies in the tile, one wavefront per particle, from LDS.  Requires
// 11 (TILE + P - 1)^3 floats of LDS (TILE 8, P 6: 96.7 KB).
#define CT_S 13
__global__ void __launch_bounds__(512) contract_tile_kernel(SpreadGeom g, const float4 *spos, const int *orig,
                                                            const int *ostart, const int *olist, const float *grid,
                                                            int64_t M, float quadw_prefac, float *wave)
{
    extern __shared__ float s_g[];           // [11][S][S][S]
    __shared__ int s_run_beg[64], s_run_off[65];
    const int S = g.tile + g.P - 1;
    const int S3 = S * S * S;
    const int tile_id = xcd_remap(blockIdx.x, gridDim.x);   // a slab of tiles per XCD: halos shared in its L2
    const int tz_i = tile_id % g.tnz, ty_i = (tile_id / g.tnz) % g.tny, tx_i = tile_id / (g.tnz * g.tny);
    const int x0 = tx_i * g.tile, y0 = ty_i * g.tile, z0 = tz_i * g.tile;
    const int lt = threadIdx.x;
    // origin cells of the tile: columns (x, y), z in [z0, z1)
    const int xe = min(x0 + g.tile, g.Nx), ye = min(y0 + g.tile, g.Ny), z1 = min(z0 + g.tile, g.Nz);
    const int ncx = xe - x0, ncy = ye - y0;
    if (lt < ncx * ncy) {
        const int x = x0 + lt / ncy, y = y0 + lt % ncy;
        const int cb = (x * g.Ny + y) * g.Nz;
        const int b0 = ostart[cb + z0], b1 = ostart[cb + z1];
        s_run_beg[lt] = b0;
        s_run_off[lt + 1] = b1 - b0;
    }
    // grid block, wrapped
    for (int idx = lt; idx < 11 * S3; idx += blockDim.x) {
        const int c = idx / S3, r = idx - c * S3;
        const int ax = r / (S * S), ay = (r / S) % S, az = r % S;
        int x = x0 + ax, y = y0 + ay, z = z0 + az;
        x -= (x >= g.Nx) ? g.Nx : 0; x -= (x >= g.Nx) ? g.Nx : 0;
        y -= (y >= g.Ny) ? g.Ny : 0; y -= (y >= g.Ny) ? g.Ny : 0;
        z -= (z >= g.Nz) ? g.Nz : 0; z -= (z >= g.Nz) ? g.Nz : 0;
        s_g[idx] = grid[c * M + ((int64_t)x * g.Ny + y) * g.pz + z];
    }
    __syncthreads();
    if (lt == 0) {
        s_run_off[0] = 0;
        for (int q = 0; q < ncx * ncy; ++q) s_run_off[q + 1] += s_run_off[q];
    }
    __syncthreads();
    const int nruns = ncx * ncy;
    const int total = s_run_off[nruns];
    const int wv = lt >> 6, lane = lt & 63, nw = blockDim.x >> 6;
    const int P = g.P;
    for (int q = wv; q < total; q += nw) {
        int lo = 0, hi = nruns - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (s_run_off[mid] <= q) lo = mid; else hi = mid - 1;
        }
        const int i = olist[s_run_beg[lo] + (q - s_run_off[lo])];
        const int ox = orig[3 * i], oy = orig[3 * i + 1], oz = orig[3 * i + 2];
        const float4 p = spos[i];
        // local block coordinates of the stencil's first node (wrapped origin - tile start)
        const int bx = (((ox % g.Nx) + g.Nx) % g.Nx) - x0;
        const int by = (((oy % g.Ny) + g.Ny) % g.Ny) - y0;
        const int bz = (((oz % g.Nz) + g.Nz) % g.Nz) - z0;
        float acc[11];
#pragma unroll
        for (int c = 0; c < 11; ++c) acc[c] = 0.f;
        if (lane < P * P) {
            const int ty = lane / P, tz = lane - P * ty;
            const float uy = g.hy * (float)(oy + ty) - g.Ly2;
            const float dz = g.hz * (float)(oz + tz) - g.Lz2 - p.z;
            const float dy = uy - p.y;
            for (int tx = 0; tx < P; ++tx) {
                const float dx = g.hx * (float)(ox + tx) - g.Lx2 + g.xy * uy - p.x;
                const float w = quadw_prefac * __expf(-g.expfac * (dx * dx + dy * dy + dz * dz));
                const int r = ((bx + tx) * S + (by + ty)) * S + (bz + tz);
#pragma unroll
                for (int c = 0; c < 11; ++c) acc[c] += w * s_g[c * S3 + r];
            }
        }
#pragma unroll
        for (int c = 0; c < 11; ++c)
            for (int o = 32; o > 0; o >>= 1) acc[c] += __shfl_xor(acc[c], o, 64);
        if (lane == 0) {
            float *w = wave + 11 * (int64_t)__float_as_int(p.w);
            w[0] = acc[0]; w[1] = acc[1]; w[2] = acc[2];
            // fields XX XY XZ YZ YY YX ZX ZY -> slots {XX, YX, ZX, ZY, YY, XY, XZ, YZ}
            w[3] = acc[3]; w[4] = acc[8]; w[5] = acc[9]; w[6] = acc[10];
            w[7] = acc[7]; w[8] = acc[4]; w[9] = acc[5]; w[10] = acc[6];
        }
    }
}

// The tile contraction for the usual stencil (P = 6, tile 8, S = 13) with
// compile-time sizes, the 11 fields split over two workgroups per tile
// (fields [0, 6) and [6, 11)) so that three workgroups share a CU and one's
// halo load overlaps another's arithmetic.
//
// Bound by VALU and LDS issue, not by HBM (18.8 MB at N = 32768 take 4 us).  So a
// particle has 16 lanes, not a wave: 12 of them each sum 18 of its 216 nodes (one z,
// three y, all x) and the sums over lanes are four DPP steps inside a row of 16, for
// four particles at once (a wave per particle kept 36 lanes busy and spent more on the
// sums than on the nodes).  The LDS block is node-major, six fields to a node, so a node
// is three 8-byte reads; lanes of consecutive z are six words apart, which conflicts
// nowhere inside a particle.  The block is loaded by the seven waves that
// do not stage particles, 30 values of a thread in flight.  Per product at N = 32768: 43 us with a
// wave per particle, 23 us so.
#define CT_NF 6
#define CT_PCAP 128   // particles of a tile staged in LDS (about 45 in an 8^3 tile at volume fraction 0.45)
template <int S, int PP>
__global__ void __launch_bounds__(512, 4) contract_tile2_kernel(SpreadGeom g, const float4 *spos, const int *orig,
                                                             const int *ostart, const int *olist, const float *grid,
                                                             int64_t M, float quadw_prefac, float *wave)
{
    constexpr int S2 = S * S, TILE = S - PP + 1, NT = 512, RL = 16;   // RL: lanes of a particle
    static_assert(TILE * TILE == 64 && PP == 6 && CT_NF % 2 == 0, "a wave scans the tile's columns");
    extern __shared__ float s_g[];           // [S][S][S][CT_NF]
    __shared__ int s_run_beg[TILE * TILE], s_run_off[TILE * TILE + 1];
    __shared__ int s_pi[CT_PCAP], s_pb[CT_PCAP];      // staged particles: index, local origin (bytes)
    __shared__ float4 s_pc[CT_PCAP];                  //   and offsets from the particle
    const int item = xcd_remap(blockIdx.x, gridDim.x);   // a slab of tiles per XCD: halos shared in its L2
    const int tile_id = item >> 1, grp = item & 1;
    const int f0 = grp ? CT_NF : 0, nf = grp ? 11 - CT_NF : CT_NF;
    const int tz_i = tile_id % g.tnz, ty_i = (tile_id / g.tnz) % g.tny, tx_i = tile_id / (g.tnz * g.tny);
    const int x0 = tx_i * TILE, y0 = ty_i * TILE, z0 = tz_i * TILE;
    const int lt = threadIdx.x, lane16 = lt % RL;
    const int xe = min(x0 + TILE, g.Nx), ye = min(y0 + TILE, g.Ny), z1 = min(z0 + TILE, g.Nz);
    const int ncx = xe - x0, ncy = ye - y0, nruns = ncx * ncy;
    auto wrap = [](int v, int n) {           // v < 3 n (the halo may pass a short axis twice)
        v -= (v >= n) ? n : 0;
        return v - ((v >= n) ? n : 0);
    };
    // Wave 0 finds and stages the tile's particles (three dependent loads: column bounds, index,
    // position) while the other waves load the grid block, every load of a thread in flight at once.
    const bool scout = lt < 64;
    int run_n = 0;
    if (scout) {
        if (lt < nruns) {
            const int x = x0 + lt / ncy, y = y0 + lt % ncy;
            const int cb = (x * g.Ny + y) * g.Nz;
            const int b0 = ostart[cb + z0];
            run_n = ostart[cb + z1] - b0;
            s_run_beg[lt] = b0;
        }
    }
    // olist entry of the tile's q-th particle (runs are the tile's (x, y) cell columns)
    auto entry = [&](int q) {
        int lo = 0, hi = nruns - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (s_run_off[mid] <= q) lo = mid; else hi = mid - 1;
        }
        return s_run_beg[lo] + (q - s_run_off[lo]);
    };
    // a staged particle (so the contraction loop below issues no global load; a tile with more than
    // CT_PCAP particles reads the rest from global memory): the index, the stencil origin in the
    // block's local frame (packed bytes) and the offsets (h o - L/2 - p) of the stencil's first node
    // from the particle, y also without p_y
    auto stage = [&](int i, int &id, int &bpk, float4 &c) {
        const int ox = orig[3 * i], oy = orig[3 * i + 1], oz = orig[3 * i + 2];
        const float4 p = spos[i];
        id = __float_as_int(p.w);
        const int bx = (((ox % g.Nx) + g.Nx) % g.Nx) - x0;
        const int by = (((oy % g.Ny) + g.Ny) % g.Ny) - y0;
        const int bz = (((oz % g.Nz) + g.Nz) % g.Nz) - z0;
        bpk = bx | (by << 8) | (bz << 16);
        const float cy = g.hy * (float)oy - g.Ly2;
        c = make_float4(g.hx * (float)ox - g.Lx2 - p.x, cy, cy - p.y, g.hz * (float)oz - g.Lz2 - p.z);
    };
    if (scout) {
        int inc = run_n;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int v = __shfl_up(inc, o, 64);
            if (lt >= o) inc += v;
        }
        s_run_off[lt + 1] = inc;             // runs past nruns are empty
        if (lt == 0) s_run_off[0] = 0;
        const int nst = min(__shfl(inc, 63, 64), CT_PCAP);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        for (int q = lt; q < nst; q += 64) {
            int id, bpk;
            float4 c;
            stage(olist[entry(q)], id, bpk, c);
            s_pi[q] = id;
            s_pb[q] = bpk;
            s_pc[q] = c;
        }
    } else {
        // node e of the block: its grid offset serves every field, whose base address is uniform
        constexpr int PER = (S2 * S + NT - 64 - 1) / (NT - 64);
        int e[PER], off[PER];
        float v[PER][CT_NF];
#pragma unroll
        for (int u = 0; u < PER; ++u) {
            e[u] = min(lt - 64 + u * (NT - 64), S2 * S - 1);   // past the end: the last node again
            const int r = e[u] / S, az = e[u] - r * S, ax = r / S, ay = r - ax * S;
            off[u] = (wrap(x0 + ax, g.Nx) * g.Ny + wrap(y0 + ay, g.Ny)) * g.pz + wrap(z0 + az, g.Nz);
        }
#pragma unroll
        for (int c = 0; c < CT_NF; ++c) {
            // the second group's sixth field repeats its fifth and is not written out
            const float *gc = grid + (int64_t)(f0 + min(c, nf - 1)) * M;
#pragma unroll
            for (int u = 0; u < PER; ++u) v[u][c] = gc[off[u]];
        }
#pragma unroll
        for (int u = 0; u < PER; ++u) {
            float2 *o = reinterpret_cast<float2 *>(s_g + e[u] * CT_NF);
#pragma unroll
            for (int c = 0; c < CT_NF; c += 2) o[c / 2] = make_float2(v[u][c], v[u][c + 1]);
        }
    }
    __syncthreads();
    const int total = s_run_off[TILE * TILE];
    // fields XX XY XZ YZ YY YX ZX ZY (grid order 3..10) -> slots {XX, YX, ZX, ZY, YY, XY, XZ, YZ}
    constexpr int slot_of[11] = {0, 1, 2, 3, 8, 9, 10, 7, 4, 5, 6};
    // this lane's nodes: z = tz, y = ty0 .. ty0 + 2, every x; lanes 12 to 15 of a particle have none
    const bool active = lane16 < 2 * PP;
    const int tz = active ? lane16 % PP : 0, ty0 = active ? lane16 / PP * (PP / 2) : 0;
    const float atz = g.hz * (float)tz;
    const float gq = __expf(-2.0f * g.expfac * g.hx * g.hx);
    int slot = 0;
#pragma unroll
    for (int f = 0; f < CT_NF; ++f)
        slot = (lane16 == f) ? (grp ? slot_of[CT_NF + (f < 11 - CT_NF ? f : 0)] : slot_of[f]) : slot;
    for (int q = lt / RL; q < total; q += NT / RL) {
        int i, bpk;
        float4 c;
        if (q < CT_PCAP) {
            i = s_pi[q];
            bpk = s_pb[q];
            c = s_pc[q];
        } else {
            stage(olist[entry(q)], i, bpk, c);
        }
        const int bx = bpk & 0xff, by = (bpk >> 8) & 0xff, bz = bpk >> 16;
        const float *node = s_g + ((bx * S + by + ty0) * S + bz + tz) * CT_NF;
        float acc[CT_NF];
#pragma unroll
        for (int f = 0; f < CT_NF; ++f) acc[f] = 0.f;
        const float dz = c.w + atz;
#pragma unroll
        for (int ty = 0; ty < PP / 2; ++ty) {
            const float ay = g.hy * (float)(ty0 + ty);
            const float uy = c.y + ay, dy = c.z + ay;
            const float dx0 = c.x + g.xy * uy;
            // the weights along x by the fast-Gaussian-gridding recurrence (Greengard and Lee,
            // SIAM Rev. 2004): w(tx + 1) = w(tx) r(tx), r(tx + 1) = r(tx) q with
            // r(0) = exp(-a hx (2 dx0 + hx)) and q = exp(-2 a hx^2)
            float w = __expf(-g.expfac * (dx0 * dx0 + (dy * dy + dz * dz)));
            float r = __expf(-g.expfac * g.hx * (2.0f * dx0 + g.hx));
#pragma unroll
            for (int tx = 0; tx < PP; ++tx) {
                const float2 *v = reinterpret_cast<const float2 *>(node + (tx * S2 + ty * S) * CT_NF);
                const float2 v0 = v[0], v1 = v[1], v2 = v[2];
                acc[0] += w * v0.x; acc[1] += w * v0.y; acc[2] += w * v1.x;
                acc[3] += w * v1.y; acc[4] += w * v2.x; acc[5] += w * v2.y;
                w *= r;
                r *= gq;
            }
        }
        float mine = 0.f;
#pragma unroll
        for (int f = 0; f < CT_NF; ++f) {
            const float t = group_sum<RL>(active ? acc[f] : 0.f);
            mine = (lane16 == f) ? t : mine;
        }
        if (lane16 < nf) wave[11 * (int64_t)i + slot] = quadw_prefac * mine;
    }
}

// LDS bytes of the tile contraction, 0 when it does not fit (then the
// per-particle contraction runs); sets the launch attribute once
int k_contract_lds(fsd_ctx *ctx)
{
    const int S = ctx->tile + ctx->pse.P - 1;
    if (S == 13 && ctx->pse.P == 6) {
        const size_t b2 = sizeof(float) * CT_NF * 13 * 13 * 13;
        if (hipFuncSetAttribute((const void *)contract_tile2_kernel<13, 6>,
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)b2) == hipSuccess) {
            ctx->contract_split = true;
            return (int)b2;
        }
    }
    const size_t bytes = sizeof(float) * 11 * (size_t)S * S * S;
    int dev = 0, maxlds = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&maxlds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess)
        return 0;
    if (ctx->tile * ctx->tile > 64 || bytes + 1024 > (size_t)maxlds) return 0;   // 64 origin columns per tile
    if (hipFuncSetAttribute((const void *)contract_tile_kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)bytes) != hipSuccess)
        return 0;
    return (int)bytes;
}

// ------------------------------------------------------------ real space
struct RealParams {
    BoxF b;
    float rcut, dr, self_x, self_y;
    int ewald_n;
    float x_scale, inv_dr;   // ewald_n / (rcut - dr), 1 / dr
};

// ------------------------------------------------------ real-space sum
struct RealPair {
    float dx, dy, dz, idist, fac;
    int row;         // of the table
    bool in;         // inside the cutoff
};
__device__ __forceinline__ RealPair real_pair(const RealParams &rp, float xi, float yi, float zi, float4 qj)
{
    RealPair p;
    p.dx = xi - qj.x; p.dy = yi - qj.y; p.dz = zi - qj.z;
    box_min_image(rp.b, p.dx, p.dy, p.dz);
    const float d2 = dist2_nc(p.dx, p.dy, p.dz);
    p.in = d2 < rp.rcut * rp.rcut && d2 >= rp.dr * rp.dr;
    // distance and its inverse to their last bits, both from the unit's reciprocal square root by Newton steps
    // (the root and the quotient apart take twice the instructions); d2 = 0 is not inside
    const float y = __builtin_amdgcn_rsqf(d2);
    float dist = d2 * y, h = 0.5f * y;
    const float e = fmaf(-h, dist, 0.5f);
    dist = fmaf(dist, e, dist);
    h = fmaf(h, e, h);
    dist = fmaf(fmaf(-dist, dist, d2), h, dist);
    p.idist = h + h;
    p.idist = fmaf(fmaf(-dist, p.idist, 1.0f), p.idist, p.idist);
    // table position with the divisions by constants done once on the host (x_scale =
    // ewald_n / (rcut - dr), inv_dr = 1 / dr)
    const float xr = (dist - rp.dr) * rp.x_scale;
    const int r = (int)floorf(xr);
    p.row = r < 0 ? 0 : (r > rp.ewald_n - 1 ? rp.ewald_n - 1 : r);
    p.fac = dist * rp.inv_dr - (float)p.row - 1.0f;
    return p;
}

// A particle's sums: velocity, antisymmetric part of the velocity gradient, (yz - zy, zx - xz, xy - yx) / 2,
// and its symmetric part (xx, 2 xy, 2 xz, 2 yz, yy)
struct RealSum {
    float u[3], t[3], e[5];
};

// Adds the pair's part (Mobility_RealSpace_kernel, Mobility.cu:1046-1226): q the neighbour's record, m and p the
// table's rows row and row + 1.  With the unit separation R and the couplet C = S + A, A x = x cross w, the pair
// sums are over s = S R and a = A R (C R = s + a, R C = s - a):
//   u += f1 F + (f2 - f1)(R.F) R + g1 (C R - rCr R) + g2 (R C - 4 rCr R)
//   D += X R + R Y + K2 1 + h1 C + (-4 h1 - h3) C^T
//   X = K1 R - g2 F + h3 (C R + R C),  Y = -g1 F + h2 C R + h3 R C
// of which the symmetric part takes only X + Y and the antisymmetric part (X - Y) cross R, a third fewer
// operations than the nine components of D.
__device__ __forceinline__ void real_add(const RealPair &w, const float4 q[4], float4 m1, float4 m2, float4 p1,
                                         float4 p2, RealSum &o)
{
    const float fac = w.fac;
    const float f1 = m1.x + (p1.x - m1.x) * fac;
    const float f2 = m1.y + (p1.y - m1.y) * fac;
    const float g1 = -(m1.z + (p1.z - m1.z) * fac);
    const float g2 = -(m1.w + (p1.w - m1.w) * fac);
    const float h1 = m2.x + (p2.x - m2.x) * fac;
    const float h2 = m2.y + (p2.y - m2.y) * fac;
    const float h3 = m2.z + (p2.z - m2.z) * fac;
    const float R[3] = {w.dx * w.idist, w.dy * w.idist, w.dz * w.idist};
    const float F[3] = {q[0].w, q[1].x, q[1].y};
    const float sxx = q[1].z, sxy = q[1].w, sxz = q[2].x, syz = q[2].y, syy = q[2].z;
    const float W[3] = {q[2].w, q[3].x, q[3].y};
    const float s[3] = {sxx * R[0] + sxy * R[1] + sxz * R[2], sxy * R[0] + syy * R[1] + syz * R[2],
                        sxz * R[0] + syz * R[1] - (sxx + syy) * R[2]};
    const float a[3] = {R[1] * W[2] - R[2] * W[1], R[2] * W[0] - R[0] * W[2], R[0] * W[1] - R[1] * W[0]};
    const float rF = R[0] * F[0] + R[1] * F[1] + R[2] * F[2];
    const float rCr = R[0] * s[0] + R[1] * s[1] + R[2] * s[2];
    const float gs = g1 + g2, gd = g1 - g2, gk = g1 + 4.f * g2, hd = h2 - h3, hs = h2 + 3.f * h3;
    const float ku = (f2 - f1) * rF - gk * rCr;
    const float K1 = gk * rF - (h2 + 6.f * h3) * rCr;
    const float K2 = h3 * rCr - g2 * rF;
    float Z[3], V[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        o.u[c] += f1 * F[c] + gs * s[c] + gd * a[c] + ku * R[c];
        Z[c] = K1 * R[c] - gs * F[c] + hs * s[c] + hd * a[c];
        V[c] = 0.5f * gd * F[c] - 0.5f * hd * (s[c] + a[c]);
    }
    const float ht = 5.f * h1 + h3, he = -3.f * h1 - h3;
    o.t[0] += V[1] * R[2] - V[2] * R[1] + ht * W[0];
    o.t[1] += V[2] * R[0] - V[0] * R[2] + ht * W[1];
    o.t[2] += V[0] * R[1] - V[1] * R[0] + ht * W[2];
    o.e[0] += Z[0] * R[0] + he * sxx + K2;
    o.e[1] += Z[0] * R[1] + R[0] * Z[1] + 2.f * he * sxy;
    o.e[2] += Z[0] * R[2] + R[0] * Z[2] + 2.f * he * sxz;
    o.e[3] += Z[1] * R[2] + R[1] * Z[2] + 2.f * he * syz;
    o.e[4] += Z[1] * R[1] + he * syy + K2;
}

// Sums over the G lanes of particle i, its own part, the wave-space result (wave, may be null),
// Mobility_D2WE_kernel (Helper_Mobility.cu:235-283) and Saddle_MakeGeneralizedU_kernel with the
// saddle's x_U term (addU, may be null).  Every lane forms the results; lane l writes number l.
template <int G>
__device__ __forceinline__ void real_finish(const RealParams &rp, const float4 *rec, int N, const float *wave,
                                            const float *addU, int use_real, float *gU, bool active, int slot, int i,
                                            int lane, RealSum &o)
{
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        o.u[c] = group_sum<G>(o.u[c]);
        o.t[c] = group_sum<G>(o.t[c]);
    }
#pragma unroll
    for (int c = 0; c < 5; ++c) o.e[c] = group_sum<G>(o.e[c]);
    if (!active) return;
    if (use_real) {
        const float4 q0 = rec[4 * (int64_t)slot], q1 = rec[4 * (int64_t)slot + 1], q2 = rec[4 * (int64_t)slot + 2],
                     q3 = rec[4 * (int64_t)slot + 3];
        // self_y (C - 4 C^T)
        const float x = rp.self_x, y = rp.self_y;
        o.u[0] += x * q0.w; o.u[1] += x * q1.x; o.u[2] += x * q1.y;
        o.t[0] += y * 5.f * q2.w; o.t[1] += y * 5.f * q3.x; o.t[2] += y * 5.f * q3.y;
        o.e[0] -= y * 3.f * q1.z; o.e[4] -= y * 3.f * q2.z;
        o.e[1] -= y * 6.f * q1.w; o.e[2] -= y * 6.f * q2.x; o.e[3] -= y * 6.f * q2.y;
    }
    if (wave) {
        const float *w = wave + 11 * (int64_t)i, *D = w + 3;
        o.u[0] += w[0]; o.u[1] += w[1]; o.u[2] += w[2];
        o.t[0] += 0.5f * (D[3] - D[7]); o.t[1] += 0.5f * (D[6] - D[2]); o.t[2] += 0.5f * (D[1] - D[5]);
        o.e[0] += D[0]; o.e[1] += D[1] + D[5]; o.e[2] += D[2] + D[6]; o.e[3] += D[3] + D[7]; o.e[4] += D[4];
    }
    const float out[11] = {o.u[0], o.u[1], o.u[2], o.t[0], o.t[1], o.t[2],
                           2.f * o.e[0] + o.e[4], o.e[1], o.e[2], o.e[3], 2.f * o.e[4] + o.e[0]};
    for (int l = lane; l < 11; l += G) {     // one round for 16 lanes
        float v = out[0];
#pragma unroll
        for (int q = 1; q < 11; ++q) v = (l == q) ? out[q] : v;
        if (addU && l < 6) v += addU[6 * (int64_t)i + l];
        gU[l < 6 ? 6 * (int64_t)i + l : 6 * (int64_t)N + 5 * (int64_t)i + l - 6] = v;
    }
}

// One particle by G lanes, its neighbours by slot (snn, nslot); table(row, m1, m2, p1, p2) gives the table's rows row and row + 1.
template <int G, typename Tab>
__device__ __forceinline__ void real_particle(const RealParams &rp, const float4 *rec, Tab table, const int *snn,
                                              const int *nslot, int maxn, int N, const float *wave, const float *addU,
                                              int use_real, float *gU, bool active, int slot, const int *order,
                                              int lane)
{
    RealSum o = {};
    const int i = (active && order) ? order[slot] : slot;
    if (active && use_real) {
        const float4 qi = rec[4 * (int64_t)slot];
        const int nn = snn[slot];
        for (int k = lane; k < nn; k += G) {
            const int64_t j = nslot[(int64_t)slot * maxn + k];
            float4 q[4];
            q[0] = rec[4 * j];
            const RealPair w = real_pair(rp, qi.x, qi.y, qi.z, q[0]);
            if (!w.in) continue;
#pragma unroll
            for (int r = 1; r < 4; ++r) q[r] = rec[4 * j + r];
            float4 m1, m2, p1, p2;
            table(w.row, m1, m2, p1, p2);
            real_add(w, q, m1, m2, p1, p2, o);
        }
    }
    real_finish<G>(rp, rec, N, wave, addU, use_real, gU, active, slot, i, lane, o);
}

// Particles are taken by slot (cell order) with each XCD given one contiguous range of workgroups, so
// the records gathered by concurrent particles lie close together in that XCD's L2; a particle's count,
// list and record are found from its slot alone, in one round of loads.  Bound by its gathers at 16-byte
// lanes (the texture units are busy all the time: four loads for a neighbour's record, four for the
// table) with VALU work of two thirds of that: 31.5 us at N = 32768 and volume fraction 0.45, 8.1 us at
// N = 4072 (by particle index, with the gradient's nine components: 36.6 and 9.0).
template <int G>
__global__ void __launch_bounds__(256) realspace_kernel(RealParams rp, const float4 *rec, const float4 *tab,
                                                        const int *snn, const int *nslot, int maxn, int N,
                                                        const float *wave, const float *addU, int use_real, float *gU,
                                                        const int *order)
{
    const int gid = xcd_remap(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
    const int slot = gid / G, lane = gid % G;
    const bool active = slot < N;
    real_particle<G>(
        rp, rec,
        [&](int r, float4 &m1, float4 &m2, float4 &p1, float4 &p2) {
            m1 = tab[2 * r]; p1 = tab[2 * r + 2];
            m2 = tab[2 * r + 1]; p2 = tab[2 * r + 3];
        },
        snn, nslot, maxn, N, wave, addU, use_real, gU, active, slot, order, lane);
}

// The same with the table in LDS, one workgroup per CU with a contiguous range of the slots, which takes
// half of the gathers off the texture units: 27.4 us at N = 32768, 180 us at N = 262144 (volume fraction
// 0.4; 200 from global memory).  Held are the rows from r = RS_RMIN on (spheres that do not overlap read
// no others; those come from global memory), as two arrays of 16-byte rows, which spreads random rows
// over all banks.
//
// Every workgroup loads the table (107 KB at xi = 0.5), so the list has to be long enough.  Table in LDS
// and from global memory, by list entries: 0.33 M 12.0 and 11.3 us, 0.50 M 12.3 and 12.8, 0.75 M 14.4 and
// 16.0, 1.0 M 18.9 and 18.1 (its workgroups end with a short pass), 1.1 M 16.5 and 19.2, 2.7 M 30 and 33,
// 5.2 M 52 and 61.
constexpr float RS_DR = 0.001f;          // distance between rows
constexpr float RS_RMIN = 1.9f;
constexpr int RS_ROWS = 5000;            // 156 KB of LDS; a longer table (xi below 0.38) stays in global memory
constexpr int64_t RS_LDS_MIN = 700000;
static int rs_first_row(const fsd_ctx *ctx)
{
    return std::max(0, std::min((int)(RS_RMIN / RS_DR) - 1, ctx->ewald_nR - 2));
}
bool real_table_in_lds(const fsd_ctx *ctx)
{
    return ctx->nlist_total >= RS_LDS_MIN && ctx->ewald_nR - rs_first_row(ctx) <= RS_ROWS;
}
template <int G>
__global__ void __launch_bounds__(1024) realspace_lds_kernel(RealParams rp, const float4 *rec, const float4 *tab,
                                                             int row0, int nrows, const int *snn, const int *nslot,
                                                             int maxn, int N, const float *wave, const float *addU,
                                                             float *gU, const int *order)
{
    extern __shared__ float4 s_tab[];        // [2][nrows]
    float4 *s_a = s_tab, *s_b = s_tab + nrows;
    for (int q = threadIdx.x; q < 2 * nrows; q += 1024) (q & 1 ? s_b : s_a)[q >> 1] = tab[2 * row0 + q];
    __syncthreads();
    const int per = (N + gridDim.x - 1) / gridDim.x, first = xcd_remap(blockIdx.x, gridDim.x) * per;
    const int last = min(first + per, N), lane = threadIdx.x % G;
    for (int s0 = first; s0 < last; s0 += 1024 / G) {
        const int slot = s0 + threadIdx.x / G;
        const bool active = slot < last;
        real_particle<G>(
            rp, rec,
            [&](int r, float4 &m1, float4 &m2, float4 &p1, float4 &p2) {
                const int q = r - row0;
                if (q >= 0) {
                    m1 = s_a[q]; p1 = s_a[q + 1];
                    m2 = s_b[q]; p2 = s_b[q + 1];
                } else {
                    m1 = tab[2 * r]; p1 = tab[2 * r + 2];
                    m2 = tab[2 * r + 1]; p2 = tab[2 * r + 3];
                }
            },
            snn, nslot, maxn, N, wave, addU, 1, gU, active, slot, order, lane);
    }
}

int k_real_init(fsd_ctx *ctx)
{
    for (auto k : {realspace_lds_kernel<4>, realspace_lds_kernel<8>, realspace_lds_kernel<16>})
        if (hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize,
                                2 * sizeof(float4) * RS_ROWS) != hipSuccess)
            return -1;
    return 0;
}

// inverse transform of the 11 half spectra in d_spec and contraction of the
// grids at the particles into d_wave (u and the velocity gradient); with x_done
// only the (y, z) part of the inverse remains
int k_wave_contract(fsd_ctx *ctx, const float4 *pos, bool x_done)
{
    const int N = ctx->N;
    const fsd_pse_info &ps = ctx->pse;
    if (!ctx->spread_valid || ctx->spread_pos != (const float *)pos) {
        const int rc = k_setup_spread(ctx, pos);
        if (rc) return rc;
    }
    const SpreadGeom g = spread_geom(ctx);
    const int64_t Mp = (int64_t)ps.Nx * ps.Ny * g.pz;   // grid field stride
    hipEvent_t ev;
    prof_begin(ctx, PROF_FFT, &ev);
    if (use_fft_x(ctx)) {
        int rc = x_done ? 0 : k_fft_x(ctx, false);
        if (!rc) rc = k_fft_yz_inverse(ctx);
        if (rc) return rc;
    } else {
        const int rc = fft_plans_3d(ctx);
        if (rc) return rc;
        if (const char *failed = ctx->fft3.inverse(ctx->d_spec, ctx->d_grid)) {
            ctx->err = failed;
            return FSD_E_HIP;
        }
    }
    prof_end(ctx, PROF_FFT, ev);
    prof_begin(ctx, PROF_CONTRACT, &ev);
    const bool tiled = ctx->tune.contract == 0 && ctx->contract_lds;
    if (tiled && ctx->contract_split)
        hipLaunchKernelGGL((contract_tile2_kernel<13, 6>), dim3(2 * ctx->ntiles), dim3(512), ctx->contract_lds,
                           ctx->stream, g, ctx->d_spos, ctx->d_porig, ctx->d_ostart, ctx->d_olist, ctx->d_grid, Mp,
                           ps.quadW * ps.prefac, ctx->d_wave);
    else if (tiled)
        hipLaunchKernelGGL(contract_tile_kernel, dim3(ctx->ntiles), dim3(512), ctx->contract_lds, ctx->stream, g, ctx->d_spos,
                           ctx->d_porig, ctx->d_ostart, ctx->d_olist, ctx->d_grid, Mp,
                           ps.quadW * ps.prefac, ctx->d_wave);
    else
        hipLaunchKernelGGL(contract_kernel, dim3(nblk((int64_t)N * 64, 256)), dim3(256), 0, ctx->stream, g, ctx->d_spos,
                           ctx->d_porig, ctx->d_grid, Mp, N, ps.quadW * ps.prefac, ctx->d_wave);
    FSD_HIP(hipGetLastError());
    prof_end(ctx, PROF_CONTRACT, ev);
    return 0;
}

// ------------------------------------------------------------ driver
// gU = M gF (+ addU on the first 6N rows); parts: 1 real, 2 wave, 3 both
int k_mobility(fsd_ctx *ctx, const float4 *pos, const float *gF, float *gU, int parts, const float *addU,
               const std::function<int(bool *)> *before_real)
{
    const int N = ctx->N;
    const fsd_pse_info &ps = ctx->pse;
    float4 *rec = ctx->d_rec;
    const int *order = slot_order(ctx);
    auto records = [&]() {
        hipLaunchKernelGGL(fc_records_kernel, dim3(nblk(N, 256)), dim3(256), 0, ctx->stream, gF, pos, order, N, rec);
    };
    if ((parts & 2) && (!ctx->spread_valid || ctx->spread_pos != (const float *)pos)) {
        const int rc = k_setup_spread(ctx, pos, gF);
        if (rc) return rc;
    } else {
        records();
    }
    FSD_HIP(hipGetLastError());
    const SpreadGeom g = spread_geom(ctx);
    const int64_t Mp = (int64_t)ps.Nx * ps.Ny * g.pz;   // grid field stride
    const float *wave = nullptr;
    if (parts & 2) {
        hipEvent_t ev;
        prof_begin(ctx, PROF_SPREAD, &ev);
        if (ctx->tile == 8 && ctx->pse.P == 6 && ctx->tune.spread == 0)
            hipLaunchKernelGGL(spread_mfma_kernel<6>, dim3(ctx->ntiles), dim3(512), 0, ctx->stream, g,
                               ctx->d_porig, rec, ctx->d_ostart, ctx->d_olist, ctx->d_grid, Mp);
        else
            hipLaunchKernelGGL(spread_kernel, dim3(ctx->ntiles), dim3(ctx->tile * ctx->tile * ctx->tile), 0,
                               ctx->stream, g, ctx->d_porig, rec, ctx->d_ostart, ctx->d_olist, ctx->d_grid,
                               Mp);
        FSD_HIP(hipGetLastError());
        prof_end(ctx, PROF_SPREAD, ev);
        const bool fx = use_fft_x(ctx);
        prof_begin(ctx, PROF_FFT, &ev);
        if (fx) {
            const int rc = k_fft_yz_forward(ctx);
            if (rc) return rc;
        } else {
            const int rc = fft_plans_3d(ctx);
            if (rc) return rc;
            if (const char *failed = ctx->fft3.forward(ctx->d_grid, ctx->d_spec)) {
                ctx->err = failed;
                return FSD_E_HIP;
            }
        }
        prof_end(ctx, PROF_FFT, ev);
        prof_begin(ctx, PROF_GREEN, &ev);
        if (fx) {   // x transforms and the Green's function in one pass
            const int rc = k_fft_x(ctx, true);
            if (rc) return rc;
        } else {
            GreenGeom gg{ps.Nx, ps.Ny, ps.Nz, ctx->box, ctx->p.xi, ps.eta, k_twopi(ctx)};
            hipLaunchKernelGGL(green_kernel, dim3(nblk(ctx->Mh, 256)), dim3(256), 0, ctx->stream, ctx->d_spec,
                               ctx->d_gridk, (int64_t)ctx->Mh, gg);
        }
        FSD_HIP(hipGetLastError());
        prof_end(ctx, PROF_GREEN, ev);
        const int rcw = k_wave_contract(ctx, pos, fx);
        if (rcw) return rcw;
        wave = ctx->d_wave;
    }
    if (before_real) {
        bool rebuilt = false;
        const int rc = (*before_real)(&rebuilt);
        if (rc) return rc;
        if (rebuilt) {
            order = slot_order(ctx);
            records();
        }
    }
    RealParams rp;
    rp.b = ctx->box; rp.rcut = ps.rcut; rp.dr = RS_DR; rp.self_x = ps.self_x; rp.self_y = ps.self_y;
    rp.ewald_n = ps.ewald_n;
    rp.x_scale = (float)((double)ps.ewald_n / ((double)ps.rcut - (double)rp.dr));
    rp.inv_dr = 1.0f / rp.dr;
    // the processing order is the neighbour list's cell list (identity without a list, wave part
    // only, or for a box of fewer than three cells per side, whose list is built over all pairs)
    if (!ctx->nlist_valid && (parts & 1)) { ctx->err = "neighbour list not built"; return FSD_E_STATE; }
    const int *snn = ctx->use_cells ? ctx->d_snn : ctx->d_nneigh, *nslot = ctx->use_cells ? ctx->d_nslot : ctx->d_nlist;
    hipEvent_t ev;
    prof_begin(ctx, PROF_REAL, &ev);
    const int G = ctx->tune.real_g, blk = ctx->tune.real_blk;
    const dim3 rg(nblk((int64_t)N * G, blk)), rb(blk);
    const float4 *tab = reinterpret_cast<const float4 *>(ctx->d_ewald);
    const int ur = (parts & 1) ? 1 : 0;
    const int row0 = rs_first_row(ctx), nrows = ctx->ewald_nR - row0;
    const bool lds = ur && real_table_in_lds(ctx);
    auto go = [&](auto plain, auto in_lds) {
        if (lds)
            hipLaunchKernelGGL(in_lds, dim3(256), dim3(1024), 2 * sizeof(float4) * nrows, ctx->stream, rp, rec, tab,
                               row0, nrows, snn, nslot, ctx->maxn, N, wave, addU, gU, order);
        else
            hipLaunchKernelGGL(plain, rg, rb, 0, ctx->stream, rp, rec, tab, snn, nslot, ctx->maxn, N,
                               wave, addU, ur, gU, order);
    };
    if (G == 4) go(realspace_kernel<4>, realspace_lds_kernel<4>);
    else if (G == 8) go(realspace_kernel<8>, realspace_lds_kernel<8>);
    else go(realspace_kernel<16>, realspace_lds_kernel<16>);
    FSD_HIP(hipGetLastError());
    prof_end(ctx, PROF_REAL, ev);
    return 0;
}
