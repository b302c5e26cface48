// Scans of a particle's neighbour list by 16 lanes.
#pragma once
#include "fsd_internal.h"

// ------------------------------------------- pairs of a particle, 16 lanes
// The kernels that scan a particle's neighbour list and work on the pairs inside a
// smaller cutoff (the lubrication operators, the force law, the pruned list) give each
// particle 16 lanes of one wave.  They are bound by latency: a scan is a chain of
// dependent loads (index, then position) and a table lookup is another, so one thread
// per particle leaves 145 waves on 256 CUs at N = 9261 and waits for ~150 of them in
// turn.  The lanes read 16 list entries at a time and append the pairs that pass the
// cutoff, in list order, to a small LDS ring; the pair work (about a third of the list
// at r < 4) then runs on 16 pairs at a time with every lane busy.  At N = 32768 and volume
// fraction 0.45 the lubrication pairs take 42 us (119 with a thread per particle); at N =
// 9261 the pairs, R_FU, R_FE, R_SU and R_SE together 110 us (491).
constexpr int PG = 16;                  // lanes per particle
constexpr int PGB = 256;                // threads per workgroup
struct PairRing {
    float4 d[PGB / PG][2 * PG];         // separation and its square
    int j[PGB / PG][2 * PG];
};

// orders this wave's LDS accesses (a group's lanes are in one wave)
__device__ __forceinline__ void wave_lds_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// particle and lane of this thread: particles in cell order (when there is one), a
// contiguous range of them per XCD; -1 past the end
__device__ __forceinline__ int pg_particle(int N, const int *order, int &lane)
{
    const int gid = xcd_remap(blockIdx.x, gridDim.x) * PGB + threadIdx.x;
    const int slot = gid / PG;
    lane = gid % PG;
    if (slot >= N) return -1;
    return order ? order[slot] : slot;
}

// Calls keep(d2) on every list entry and use(q, j, d) on the entries kept, q their
// ordinal in list order and d = (p_j - p_i, d2).  Returns the number kept.
template <class Keep, class Use>
__device__ __forceinline__ int pg_pairs(PairRing &ring, const float4 *pos, const BoxF &b, float4 pi, const int *row,
                                        int nn, int lane, Keep keep, Use use)
{
    const int grp = threadIdx.x / PG, first = (threadIdx.x & 63) & ~(PG - 1);
    float4 *rd = ring.d[grp];
    int *rj = ring.j[grp];
    int head = 0, tail = 0;
    int jn = lane < nn ? row[lane] : 0;
    for (int k0 = 0; k0 < nn; k0 += PG) {
        const int j = jn;
        const bool in = k0 + lane < nn;
        jn = k0 + PG + lane < nn ? row[k0 + PG + lane] : 0;
        const float4 pj = pos[j];
        float dx = pj.x - pi.x, dy = pj.y - pi.y, dz = pj.z - pi.z;
        box_min_image(b, dx, dy, dz);
        const float d2 = dist2_nc(dx, dy, dz);
        const bool ok = in && keep(d2);
        const unsigned m = (unsigned)(__ballot(ok) >> first) & 0xffffu;
        if (ok) {
            const int q = (tail + __popc(m & ((1u << lane) - 1u))) & (2 * PG - 1);
            rd[q] = make_float4(dx, dy, dz, d2);
            rj[q] = j;
        }
        tail += __popc(m);
        wave_lds_fence();
        if (tail - head >= PG) {
            const int q = (head + lane) & (2 * PG - 1);
            use(head + lane, rj[q], rd[q]);
            head += PG;
            wave_lds_fence();
        }
    }
    if (head + lane < tail) {
        const int q = (head + lane) & (2 * PG - 1);
        use(head + lane, rj[q], rd[q]);
    }
    wave_lds_fence();
    return tail;
}

// the neighbour list's cell order; null for a list built over all pairs (identity order)
inline const int *cell_order(const fsd_ctx *ctx) { return ctx->use_cells ? ctx->d_cell_list : nullptr; }

// the counts of a workgroup's particles (one per group, -1: none): the largest into *most when it
// exceeds the capacity cap, their sum (each at most cap) added to *sum.  Every thread calls it.
__device__ __forceinline__ void pg_block_counts(int *s_cnt, int cap, int *most, int *sum)
{
    __syncthreads();
    if (threadIdx.x == 0) {
        int m = 0, t = 0;
        for (int g = 0; g < PGB / PG; ++g) {
            m = max(m, s_cnt[g]);
            t += max(0, min(s_cnt[g], cap));
        }
        if (m > cap) atomicMax(most, m);
        if (sum) atomicAdd(sum, t);
    }
}
