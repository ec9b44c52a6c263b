// psim_build.hpp -- the per-step cell rebuild (hash, counting sort,
// cell-start table, canonical reorder of the state), kernels shared by the
// single-system engine and the replica ensemble.
//
// Replaces system::hashParticles / sortParticles / clearCells /
// reorderParticles (systemHandling.cpp:33-85): instead of an O(N log N)
// comparison sort of (hash, index) tuples every step, each particle is
// entered in the bin of its new cell during the step, and one kernel (two in
// crowded boxes) turns the bins into a start table and moves the state into cell
// order.  Within a
// cell the order is the previous slot order (a stable counting sort), which
// makes every run reproducible bit for bit.  The scan and scatter kernels
// below serve the rebuilds that start from counts (analysis grid, forces
// without a context).
#pragma once

#include "psim_bins.hpp"
#include "psim_gather.hpp"

namespace psim {
namespace {

constexpr int kScanThreads = 1024;
constexpr int kScanItems = 4;
constexpr int kScanTile = kScanThreads * kScanItems;

// Every particle into its cell's bin, in an arbitrary order (initial build).
__global__ void k_bin_all(Geo g, const double *pos, Bins b)
{
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= g.n) return;
    const int N = g.n;
    const int k = g.c0 + cell_1d(pos[s], g.cell, g.S) + g.S * cell_1d(pos[N + s], g.cell, g.S)
                + g.S2 * cell_1d(pos[2 * N + s], g.cell, g.S);
    bin_particle(b, N, s, k);
}

// Cell hash + atomic count for an arbitrary order.
__global__ void k_hash_count(Geo g, const double *pos, int *key, int *arank, int *count)
{
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= g.n) return;
    const int N = g.n;
    int k = g.c0 + cell_1d(pos[s], g.cell, g.S) + g.S * cell_1d(pos[N + s], g.cell, g.S)
          + g.S2 * cell_1d(pos[2 * N + s], g.cell, g.S);
    key[s] = k;
    arank[s] = wave_aggregated_rank(count, k);
}

// Exclusive scan over a 1024-thread block of one value per thread; *total
// receives the block's sum.
__device__ int block_exclusive_scan(int v, int *total)
{
    __shared__ int wsum[kScanThreads / 64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int x = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        int y = __shfl_up(x, d, 64);
        if (lane >= d) x += y;
    }
    if (lane == 63) wsum[w] = x;
    __syncthreads();
    if (w == 0) {
        int t = lane < kScanThreads / 64 ? wsum[lane] : 0;
#pragma unroll
        for (int d = 1; d < kScanThreads / 64; d <<= 1) {
            int y = __shfl_up(t, d, 64);
            if (lane >= d) t += y;
        }
        if (lane < kScanThreads / 64) wsum[lane] = t;
    }
    __syncthreads();
    int pre = (w > 0 ? wsum[w - 1] : 0) + x - v;
    *total = wsum[kScanThreads / 64 - 1];
    __syncthreads();
    return pre;
}

// The counts of one tile (kScanItems consecutive cells per thread, one
// 16-byte load where the tile is whole).
__device__ __forceinline__ void tile_counts(const int *count, int ncell, int base,
                                            int (&c)[kScanItems])
{
    static_assert(kScanItems == 4, "one int4 per thread");
    if (base + kScanItems <= ncell) {
        const int4 q = *reinterpret_cast<const int4 *>(count + base);
        c[0] = q.x;
        c[1] = q.y;
        c[2] = q.z;
        c[3] = q.w;
    } else {
#pragma unroll
        for (int k = 0; k < kScanItems; ++k) c[k] = (base + k < ncell) ? count[base + k] : 0;
    }
}

// Tile totals: bsum[b] = sum of the counts of tile b.
__global__ __launch_bounds__(kScanThreads) void k_scan_reduce(const int *count, int ncell,
                                                              int *bsum)
{
    int c[kScanItems];
    tile_counts(count, ncell, blockIdx.x * kScanTile + threadIdx.x * kScanItems, c);
    int v = c[0] + c[1] + c[2] + c[3];
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) v += __shfl_xor(v, d, 64);
    __shared__ int wsum[kScanThreads / 64];
    if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        int t = 0;
        for (int w = 0; w < kScanThreads / 64; ++w) t += wsum[w];
        bsum[blockIdx.x] = t;
    }
}

// The tile totals replaced by their exclusive prefix sums (one block, eight
// totals per thread and round).
__global__ __launch_bounds__(kScanThreads) void k_scan_bsum(int *bsum, int nb)
{
    constexpr int kItems = 8;
    int carry = 0;
    for (int b0 = 0; b0 < nb; b0 += kItems * kScanThreads) {
        const int i = b0 + kItems * (int)threadIdx.x;
        int v[kItems], sum = 0;
#pragma unroll
        for (int k = 0; k < kItems; ++k) v[k] = i + k < nb ? bsum[i + k] : 0;
#pragma unroll
        for (int k = 0; k < kItems; ++k) sum += v[k];
        int total;
        int pre = carry + block_exclusive_scan(sum, &total);
#pragma unroll
        for (int k = 0; k < kItems; ++k) {
            if (i + k < nb) bsum[i + k] = pre;
            pre += v[k];
        }
        carry += total;
    }
}

// Cell start table from the counts: block b scans its tile on top of the
// prefix of the tile totals before it, writes the starts and clears the counts for the next step's counting.  With
// RESUM, the block sums the raw totals bsum[0..b) itself (few tiles);
// otherwise bsum already holds the prefixes (k_scan_bsum).
template <bool RESUM>
__global__ __launch_bounds__(kScanThreads) void k_scan_apply(int *count, int ncell,
                                                             const int *bsum,
                                                             int *cstart, int n)
{
    int before;
    if constexpr (RESUM) {
        int v = 0;
        for (int b = threadIdx.x; b < (int)blockIdx.x; b += kScanThreads) v += bsum[b];
        block_exclusive_scan(v, &before);
    } else {
        before = bsum[blockIdx.x];
    }
    const int base = blockIdx.x * kScanTile + threadIdx.x * kScanItems;
    int c[kScanItems];
    tile_counts(count, ncell, base, c);
    int total;
    int pre = block_exclusive_scan(c[0] + c[1] + c[2] + c[3], &total) + before;
    if (base + kScanItems <= ncell) {
        const int4 st = make_int4(pre, pre + c[0], pre + c[0] + c[1], pre + c[0] + c[1] + c[2]);
        *reinterpret_cast<int4 *>(cstart + base) = st;
        *reinterpret_cast<int4 *>(count + base) = make_int4(0, 0, 0, 0);
    } else {
#pragma unroll
        for (int k = 0; k < kScanItems; ++k) {
            if (base + k < ncell) {
                cstart[base + k] = pre;
                count[base + k] = 0;
            }
            pre += c[k];
        }
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) cstart[ncell] = n;
}

// The scan of the cell counts into the start table for grids of more than
// kScanDirectTiles tiles: tile totals, then each tile's scan on top of the
// totals before it, summed by each block itself up to kScanResumTiles tiles
// (two launches), beyond that first turned into prefixes by one block
// (three launches; the re-summing grows with the square of the tile count).
constexpr int kScanResumTiles = 256;
inline void launch_scan3(hipStream_t st, int *count, int ncell, int nscan, int *bsum,
                         int *cstart, int n)
{
    k_scan_reduce<<<nscan, kScanThreads, 0, st>>>(count, ncell, bsum);
    if (nscan <= kScanResumTiles) {
        k_scan_apply<true><<<nscan, kScanThreads, 0, st>>>(count, ncell, bsum, cstart, n);
    } else {
        k_scan_bsum<<<1, kScanThreads, 0, st>>>(bsum, nscan);
        k_scan_apply<false><<<nscan, kScanThreads, 0, st>>>(count, ncell, bsum, cstart, n);
    }
}

// Cell start table in one launch for grids of at most kScanDirectTiles
// tiles: each block sums the counts of the tiles before it itself instead of
// reading k_scan_reduce's tile sums.  The counts stay in place (other blocks
// are still reading them); k_scatter clears them.
// (alone it beats k_scan_reduce + k_scan_apply up to about 32 tiles, 7.0 vs
// 9.6 us at 20; inside a step it does not: at 16 tiles, N = 32768 AO with
// 64000 cells, the two launches make the whole step 3.5 us faster, so the
// direct form is kept for the smallest grids only)
constexpr int kScanDirectTiles = 4;
__global__ __launch_bounds__(kScanThreads) void k_scan_direct(const int *count, int ncell,
                                                              int *cstart, int n)
{
    const int lim = blockIdx.x * kScanTile;   // a multiple of 4, at most ncell
    int before = 0;
    // eight independent 16-byte loads in flight per lane (the sum is
    // latency-bound otherwise)
    constexpr int kStride = kScanThreads * 4;
    for (int i0 = threadIdx.x * 4; i0 < lim; i0 += 8 * kStride) {
        int4 v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int i = i0 + u * kStride;
            v[u] = i < lim ? *reinterpret_cast<const int4 *>(count + i) : make_int4(0, 0, 0, 0);
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) before += v[u].x + v[u].y + v[u].z + v[u].w;
    }
    int before_total;
    block_exclusive_scan(before, &before_total);
    const int base = blockIdx.x * kScanTile + threadIdx.x * kScanItems;
    int c[kScanItems];
    int v = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        c[k] = (base + k < ncell) ? count[base + k] : 0;
        v += c[k];
    }
    int total;
    int pre = block_exclusive_scan(v, &total) + before_total;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        if (base + k < ncell) cstart[base + k] = pre;
        pre += c[k];
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) cstart[ncell] = n;
}

// With clear_count set (after k_scan_direct), also zeroes the ncell counts
// for the next call's counting.
__global__ __launch_bounds__(256) void k_scatter(int n, const int *key, const int *arank,
                                                 const int *cstart, int *perm,
                                                 int *clear_count, int ncell)
{
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (clear_count)
        for (int c = s; c < ncell; c += gridDim.x * blockDim.x) clear_count[c] = 0;
    if (s < n) perm[cstart[key[s]] + arank[s]] = s;
}

// 1 / L of the box that slot t's particle lives in: one box for all; NoBox
// where the pair kernel reads no box fractions.
struct OneBox {
    static constexpr bool kPack = true;
    double inv_L;
    __device__ double operator()(int) const { return inv_L; }
};
struct NoBox {
    static constexpr bool kPack = false;
    __device__ double operator()(int) const { return 0.0; }
};

// Where the rebuild writes the new order.  With cstart2 / pos2 / id2 set, the
// cell table and the new positions and ids are also written there (a record
// of the state, e.g. the adjoint's recomputed trajectory), and with inv2 the
// slot of each original index.
struct Rebuilt {
    int *cstart;
    double *pos;
    int *id, *prev;
    uint4 *upos;
    int *cstart2;
    double *pos2;
    int *id2, *inv2;
};

constexpr int kTileList = 1024;   // members in LDS at a time

// The particle of slot s (position, original id o) to slot dst of cell c.
template <class Box>
__device__ __forceinline__ void put_particle(const Rebuilt &to, int n, int dst, int s, double px,
                                             double py, double pz, int o, int c, const Box &box)
{
    to.pos[dst] = px;
    to.pos[n + dst] = py;
    to.pos[2 * n + dst] = pz;
    if (to.pos2) {
        to.pos2[dst] = px;
        to.pos2[n + dst] = py;
        to.pos2[2 * n + dst] = pz;
    }
    if (Box::kPack) to.upos[dst] = pack_position(px, py, pz, c, box(dst));
    to.id[dst] = o;
    if (to.id2) to.id2[dst] = o;
    if (to.inv2) to.inv2[o] = dst;
    to.prev[dst] = s;
}

// The cell rebuild in one launch: start table, canonical order, positions and
// ids moved into it.
//
// A workgroup owns a tile of 1 << shift consecutive cells, at most kPer per
// thread.  Its first slot is
// the sum of the tile totals before it (prefixed: tile_total already holds
// that sum), the starts of its cells a scan of their counts; the members come
// from the cells' bins, and a member's place in its cell is the number of
// members with a lower slot.  Canonical order within a cell = ascending
// source slot (a stable counting sort).  Only the positions and the original
// ids are gathered into the new order; prev[dst] records the slot each
// particle came from, so the integrator reads the previous positions, forces
// and memory of the last step where it wrote them (at prev[s]) instead of
// every array moving every step.
//
// Bound by latency: three dependent rounds of loads (counts and totals, bins,
// positions) and one of stores.  As separate kernels (counts summed by tile,
// start table, scatter into cell order, move) it was nine such rounds and
// three more launch boundaries: 4.9 + 5.4 + 4.7 + 6.6 us of a 45 us step at
// 262,144 AO particles, now a step of 33.3; 19.1 for 23.0 us at 4,096 (three
// kernels before), 27.4 for 36.0 at 30,011, 829 for 900 at 2,097,152.
//
// Each lane moves up to U particles with their loads together.  A tile with
// more members than U * kTileThreads (a dense spot) is done in batches of
// cells that fit the list, kWide particles per lane; a cell that does not fit
// by itself keeps its members in perm, which has room for them at the cell's
// slots.
//
// split: the kernel stops at the start table and the chains (left in perm), and
// k_place moves the particles, one per lane over the whole grid: see
// shape_bins.
//
// The kernel clears what the next step counts into: the counts of its cells,
// the heads of its chains, and next_total, the other of two arrays of tile
// totals (this step's are still being read).  With ctl set (a step sequence
// whose control lives in device memory) it also ends the step: it advances
// the clock and the next step's flags, which no kernel of this step reads
// after the integrator.  Box::kPack: the new positions' box fractions and
// cells are written to upos too (the thread-per-particle kernels' cull).
template <int U, int kPer, class Box>
__global__ __launch_bounds__(kTileThreads) void k_rebuild(int n, int ncell, Bins b, int prefixed,
                                                          int split, int *next_total, int *perm,
                                                          const double *__restrict__ npos,
                                                          const int *__restrict__ id_in,
                                                          StepCtl *ctl, Box box, Rebuilt to)
{
    constexpr int kDirect = U * kTileThreads;
    __shared__ int start[kPer * kTileThreads + 1];
    __shared__ int list[kTileList];
    __shared__ unsigned short cell_of[kTileList];
    __shared__ int wsum[2][kTileThreads / 64];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    // below the size of U = 4 a tile runs on the XCD whose L2 the integrator
    // left its particles in (xcd_block's order; 34.0 -> 33.3 us a step at
    // 262,144 particles, 7.25 -> 7.07 ms a fit at 32,768; at 2,097,152 they
    // are long gone, and the launch order is 3 us faster)
    const int tile = U < 4 ? xcd_block() : blockIdx.x;
    if (U < 4 && ((long long)tile << b.shift) >= ncell) return;
    const int c0 = tile << b.shift;
    const int cells = min(1 << b.shift, ncell - c0);
    if (ctl && tile == 0 && tid == 0) ctl_advance(ctl);

    // totals of the tiles before this one; this lane's four counts
    int before = 0;
    if (prefixed) {
        if (tid == 0) before = b.tile_total[tile];
    } else {
        for (int i = tid * 4; i < tile; i += kTileThreads * 4) {
            const int4 q = *reinterpret_cast<const int4 *>(b.tile_total + i);
            before += q.x + (i + 1 < tile ? q.y : 0) + (i + 2 < tile ? q.z : 0) +
                      (i + 3 < tile ? q.w : 0);
        }
    }
    const int k0 = tid * kPer;
    int cnt[kPer] = {};
#pragma unroll
    for (int k = 0; k < kPer; k += 4) {
        if (k0 + k + 4 <= cells) {
            int4 *p = reinterpret_cast<int4 *>(b.count + c0 + k0 + k);
            const int4 q = *p;
            cnt[k] = q.x;
            cnt[k + 1] = q.y;
            cnt[k + 2] = q.z;
            cnt[k + 3] = q.w;
            *p = make_int4(0, 0, 0, 0);
        } else {
#pragma unroll
            for (int u = k; u < k + 4; ++u)
                if (k0 + u < cells) {
                    cnt[u] = b.count[c0 + k0 + u];
                    b.count[c0 + k0 + u] = 0;
                }
        }
    }
    if (tid == 0) next_total[tile] = 0;
    int mine = 0;
#pragma unroll
    for (int k = 0; k < kPer; ++k) mine += cnt[k];
    int x = mine;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int y = __shfl_up(x, d, 64);
        if (lane >= d) x += y;
        before += __shfl_xor(before, d, 64);
    }
    if (lane == 63) {
        wsum[0][w] = x;
        wsum[1][w] = before;
    }
    __syncthreads();
    int pre = x - mine, base = 0, m = 0;
#pragma unroll
    for (int v = 0; v < kTileThreads / 64; ++v) {
        if (v < w) pre += wsum[0][v];
        m += wsum[0][v];
        base += wsum[1][v];
    }
    const bool direct = m <= kDirect && !split;
    {
        int st[kPer];
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
            st[k] = pre;
            pre += cnt[k];
            if (k0 + k < cells) {
                start[k0 + k] = st[k];
                if (direct)
                    for (int j = 0; j < cnt[k]; ++j) cell_of[st[k] + j] = (unsigned short)(k0 + k);
            }
        }
#pragma unroll
        for (int k = 0; k < kPer; k += 4) {
            if (k0 + k + 4 <= cells) {
                const int4 q = make_int4(base + st[k], base + st[k + 1], base + st[k + 2],
                                         base + st[k + 3]);
                *reinterpret_cast<int4 *>(to.cstart + c0 + k0 + k) = q;
            } else {
#pragma unroll
                for (int u = k; u < k + 4; ++u)
                    if (k0 + u < cells) to.cstart[c0 + k0 + u] = base + st[u];
            }
        }
        if (to.cstart2) {   // of any alignment
#pragma unroll
            for (int k = 0; k < kPer; ++k)
                if (k0 + k < cells) to.cstart2[c0 + k0 + k] = base + st[k];
        }
    }
    if (tid == 0) {
        start[cells] = m;
        if (c0 + cells == ncell) {
            to.cstart[ncell] = n;
            if (to.cstart2) to.cstart2[ncell] = n;
        }
    }
    __syncthreads();
    if (m == 0) return;

    // chain q of cell i: members cap + q, cap + q + chains, ... to out[0],
    // out[chains], ...
    auto unchain = [&](int i, int q, int *out) {
        int *head = b.over + (size_t)n + (size_t)(c0 + i) * b.chains + q;
        int s = *head;
        *head = -1;
        const int end = start[i + 1] - start[i] - b.cap - q;
        for (int k = 0; k < end && s >= 0; k += b.chains) {
            out[k] = s;
            s = b.over[s];
        }
    };
    if (split) {
        for (int i = tid; i < cells; i += kTileThreads)
            for (int q = 0; q < b.chains && start[i + 1] - start[i] > b.cap + q; ++q)
                unchain(i, q, perm + base + start[i] + b.cap + q);
        return;
    }
    // member j of the tile (cell i, r-th of its bin) to *out; the first members
    // past the row walk the cell's chains
    auto fetch = [&](int j, int i, int *out) {
        const int r = j - start[i];
        if (r < b.cap) {
            const int s = *b.place(c0 + i, r);
            *out = s;
            return s;
        }
        if (r < b.cap + b.chains) unchain(i, r - b.cap, out);
        return -1;
    };
    auto place = [&](int i, int rank, int s, double px, double py, double pz, int o) {
        put_particle(to, n, base + start[i] + rank, s, px, py, pz, o, c0 + i, box);
    };
    // l: the members of cell i
    auto rank_in = [&](const int *l, int i, int s) {
        const int len = start[i + 1] - start[i];
        int rank = 0;
        for (int k = 0; k < len; ++k) rank += l[k] < s;
        return rank;
    };
    if (direct) {
        int i[U], s[U], o[U];
        double p[U][3];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int j = tid + u * kTileThreads;
            i[u] = j < m ? cell_of[j] : 0;
            s[u] = j < m ? fetch(j, i[u], list + j) : -1;
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int j = tid + u * kTileThreads;
            if (s[u] < 0) s[u] = j < m ? list[j] : list[0];
#pragma unroll
            for (int d = 0; d < 3; ++d) p[u][d] = npos[d * n + s[u]];
            o[u] = id_in[s[u]];
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (tid + u * kTileThreads < m)
                place(i[u], rank_in(list + start[i[u]], i[u], s[u]), s[u], p[u][0], p[u][1],
                      p[u][2], o[u]);
        return;
    }
    // Batches of cells whose members fit the list: kWide members per lane, their
    // searches and loads together, and kDeep members of each one's cell at a
    // time for its rank (four and two, or four and four: no faster, 79 and 86
    // VGPRs instead of 50).  A drop of 160,000 LJ particles, 12 to 27 per cell,
    // in 40,000 of vapour: the rebuild takes 38 us, 101 with the members and
    // their order in global memory, 10 to 22 without the drop.
    constexpr int kWide = 2, kDeep = 4;
    auto last_at = [&](int j, int lo, int hi) {   // last of lo..hi that starts at or before j
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (start[mid] <= j) lo = mid; else hi = mid - 1;
        }
        return lo;
    };
    // l: the members of cells i0 .. i1 - 1
    auto batch = [&](int i0, int i1, int *l, bool in_list) __attribute__((always_inline)) {
        const int j0 = start[i0], j1 = start[i1];
        int top = 1;
        while (top < i1 - i0) top *= 2;
        for (int j = j0 + tid; j < j1; j += kWide * kTileThreads) {
            int i[kWide];
#pragma unroll
            for (int u = 0; u < kWide; ++u) i[u] = i0;
            for (int step = top >> 1; step; step >>= 1)
#pragma unroll
                for (int u = 0; u < kWide; ++u) {
                    const int mid = min(i[u] + step, i1 - 1);
                    if (start[mid] <= j + u * kTileThreads) i[u] = mid;
                }
#pragma unroll
            for (int u = 0; u < kWide; ++u) {
                const int q = j + u * kTileThreads;
                if (q < j1) {
                    fetch(q, i[u], l + (q - j0));
                    if (in_list) cell_of[q - j0] = (unsigned short)i[u];
                }
            }
        }
        __syncthreads();
        for (int j = j0 + tid; j < j1; j += kWide * kTileThreads) {
            int s[kWide], o[kWide], at[kWide], len[kWide], rank[kWide], i[kWide], most = 0;
            double p[kWide][3];
#pragma unroll
            for (int u = 0; u < kWide; ++u) {   // (a missing member repeats the last)
                const int q = min(j + u * kTileThreads, j1 - 1) - j0;
                s[u] = l[q];
                i[u] = in_list ? cell_of[q] : i0;
            }
#pragma unroll
            for (int u = 0; u < kWide; ++u) {
#pragma unroll
                for (int d = 0; d < 3; ++d) p[u][d] = npos[d * n + s[u]];
                o[u] = id_in[s[u]];
                at[u] = start[i[u]] - j0;
                len[u] = start[i[u] + 1] - start[i[u]];
                rank[u] = 0;
                most = max(most, len[u]);
            }
            for (int k = 0; k < most; k += kDeep)
#pragma unroll
                for (int u = 0; u < kWide; ++u)
#pragma unroll
                    for (int q = 0; q < kDeep; ++q)
                        rank[u] += (k + q < len[u]) & (l[min(at[u] + k + q, j1 - j0 - 1)] < s[u]);
#pragma unroll
            for (int u = 0; u < kWide; ++u)
                if (j + u * kTileThreads < j1)
                    place(i[u], rank[u], s[u], p[u][0], p[u][1], p[u][2], o[u]);
        }
        __syncthreads();   // the list is free again
    };
    for (int i0 = 0; i0 < cells;) {
        const int i1 = last_at(start[i0] + kTileList, i0, cells);
        if (i1 > i0) {
            batch(i0, i1, list, true);
            i0 = i1;
        } else {
            batch(i0, i0 + 1, perm + base + start[i0], false);
            ++i0;
        }
    }
}

// The other half of a split rebuild: the particle of every slot of the bins'
// order (cell by cell, rows and then chains) to its place in its cell.  Each
// lane finds its cell in the start table.
template <class Box>
__global__ __launch_bounds__(256) void k_place(int n, int ncell, Bins b,
                                               const int *__restrict__ perm,
                                               const double *__restrict__ npos,
                                               const int *__restrict__ id_in, Box box, Rebuilt to)
{
    const int t = xcd_block() * 256 + threadIdx.x;
    if (t >= n) return;
    int c = 0;
    for (int hi = ncell - 1; c < hi;) {
        const int mid = c + (hi - c + 1) / 2;
        if (to.cstart[mid] <= t) c = mid; else hi = mid - 1;
    }
    const int base = to.cstart[c], len = to.cstart[c + 1] - base;
    const int *row = b.place(c, 0);
    const int s = t - base < b.cap ? row[t - base] : perm[t];
    const double x = npos[s], y = npos[n + s], z = npos[2 * n + s];
    const int o = id_in[s];
    // (16 members' loads in flight; a row is a multiple of 16 long here)
    const int in_row = min(len, b.cap);
    int rank = 0;
    for (int r = 0; r < in_row; r += 16) {
        int4 v[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = reinterpret_cast<const int4 *>(row + r)[q];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int k = r + 4 * q;
            rank += (k < in_row && v[q].x < s) + (k + 1 < in_row && v[q].y < s) +
                    (k + 2 < in_row && v[q].z < s) + (k + 3 < in_row && v[q].w < s);
        }
    }
    for (int k = in_row; k < len; ++k) rank += perm[base + k] < s;
    put_particle(to, n, base + rank, s, x, y, z, o, c, box);
}

// A workgroup sums the totals before its tile itself up to this many tiles (16
// loads of 16 bytes per lane); beyond that one block turns them into prefixes
// first.  (10,044 tiles, a step at N = 262,144 in 20.6 million cells: 126.5 us
// with the prefix launch, 115.1 without.)
constexpr int kSelfPrefixTiles = 16384;

template <class Box>
void launch_rebuild(hipStream_t st, int n, int ncell, BinStore &t, const double *npos,
                    const int *id_in, StepCtl *ctl, Box box, const Rebuilt &to)
{
    const int prefixed = t.tiles > kSelfPrefixTiles;
    if (prefixed) k_scan_bsum<<<1, kScanThreads, 0, st>>>(t.b.tile_total, t.tiles);
    auto go = [&](auto lanes, auto per) {
        constexpr int kU = decltype(lanes)::value;
        k_rebuild<kU, decltype(per)::value>
            <<<kU < 4 ? xcd_grid(t.tiles) : t.tiles, kTileThreads, 0, st>>>(
                n, ncell, t.b, prefixed, t.split, t.next_total, t.perm, npos, id_in, ctl, box, to);
    };
    const std::integral_constant<int, 1> one;
    const std::integral_constant<int, 2> two;
    const std::integral_constant<int, 4> four;
    const std::integral_constant<int, 8> eight;
    if (t.per == 8) t.lanes == 4 ? go(four, eight) : t.lanes == 2 ? go(two, eight) : go(one, eight);
    else t.lanes == 4 ? go(four, four) : t.lanes == 2 ? go(two, four) : go(one, four);
    if (t.split)
        k_place<<<xcd_grid((n + 255) / 256), 256, 0, st>>>(n, ncell, t.b, t.perm, npos, id_in, box,
                                                           to);
}

// The lagged arrays (previous positions, last forces, memory, kept in the
// order of the step that wrote them) gathered into the current slot order.
// With pos set, pos0 holds the positions the last step started from and is
// re-imaged against the current positions (util::safeMod0, as the step would
// have stored it).
__global__ void k_settle(int n, const int *__restrict__ prev, const double *__restrict__ pos0,
                         const double *__restrict__ frc, const double *__restrict__ mem,
                         double *__restrict__ pos0_out, double *__restrict__ frc_out,
                         double *__restrict__ mem_out, const double *__restrict__ pos = nullptr,
                         double L = 0.0)
{
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    const int p = prev[s];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const double x0 = pos0[d * n + p];
        pos0_out[d * n + s] = pos ? safe_mod0(x0, pos[d * n + s], L) : x0;
        frc_out[d * n + s] = frc[d * n + p];
        mem_out[d * n + s] = mem[d * n + p];
    }
}

}  // namespace
}  // namespace psim
