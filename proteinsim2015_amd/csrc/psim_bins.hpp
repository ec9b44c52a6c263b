// psim_bins.hpp -- the bins that a step's integrator enters every particle in
// and the cell rebuild (k_rebuild) takes them from: storage and shape.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>

#include "psim_device.hpp"

namespace psim {

constexpr int kTileThreads = 256;

// The bins of a system or a stack of systems, and the shape of their tiles.
struct BinStore {
    Bins b{};
    int *next_total = nullptr, *perm = nullptr;
    int tiles = 0, lanes = 1, per = 4;   // k_rebuild's U and kPer
    bool split = false;         // k_rebuild leaves the particles to k_place
};

// Bins and tiles for n particles in ncell cells of at most cell_volume (in
// cubed particle diameters).
//
// A bin holds what hard particles can pack into a cell, or four times the mean
// and a few (at least 32), whichever is less; a longer chain costs time, not
// correctness.  Bins that would take more than 256 bytes per particle and more
// than 1 GiB (boxes with hardly any particle per cell) are made shorter, down to
// one member, and have one chain per cell instead of four: at 1290^3 cells, the
// most there are, 12 bytes per cell beside the start table.  The bins lie member
// by member (all first members, all second ones, ...): the lines that a dilute
// system touches are full of what its neighbours wrote.  With a row per cell a
// step at N = 1,200,000 in 4.1 million cells took 168 us (now 138), at 2,097,152
// AO in 40 million 531 (488), at 1,200,000 LJ at 1.5 per cell 217 (194); at 15
// per cell there is no difference (2,097,152: 724, 720).
//
// A tile holds the cells of about 1/256 of the particles (a workgroup per
// compute unit), at least 64 and at most 192 per particle of a lane.  Lanes
// move two particles from 131,072 on and four from 1,048,576 (a step in us, one /
// two / four, AO at phi = 0.15: 65,536 19.1 / 20.0 / 24.6, 131,072 29.8 / 30.2 /
// 34.6, 180,000 39.7 / 38.0 / 40.9, 524,288 59.6 / 53.7 / 53.1, 1,048,576 112 /
// 96 / 99, 1,400,000 185 / 159 / 154; 15 per cell, 65,536 40.0 / 40.7 / 42.6,
// 262,144 110 / 106 / 108, 1,048,576 391 / 373 / 368).  Tiles of half or twice as
// many particles: no difference.  It holds at most 1024 cells, or 2048 where
// there are more of those tiles than the chip holds twice over and they are
// nearly empty (2,097,152 AO particles in 40 million cells: 489 / 452 us a step,
// 100,000 in 7.8 million 47.0 / 39.8; at 2 million cells 1.4 us slower).
//
// A tile is four cells at least.  Where that many hold more than its workgroup
// moves at once, a handful of workgroups would do all the work; the particles
// are then moved by a second launch over the whole grid (split), which reads
// whole rows.  The rebuild in us, one launch / two: 64 per cell 8.9 / 11.7 at
// 30,000 particles (one per lane) and 13.0 / 16.7 at 300,000 (two), 80 per cell
// 20.1 / 12.2 at 10,000, 137 per cell 36.3 / 16.5 at 100,000 and 38.7 / 19.4 at
// 300,000; at 4 cells a side, 10,000 particles 32.7 / 13.7, 100,000 2191 / 50.
inline void shape_bins(int n, int ncell, double cell_volume, BinStore &t)
{
    const double occ = (double)n / ncell;
    t.lanes = n >= (1 << 20) ? 4 : n >= (1 << 17) ? 2 : 1;
    t.per = occ < 0.15 && ncell > (4 << 20) ? 8 : 4;
    t.split = 4.0 * occ > 0.9 * kTileThreads * t.lanes;
    const double packed = fmin(1.25 * cell_volume + 1.0, fmax(4.0 * occ + 8.0, 32.0));
    const double most = fmin(fmax(packed, 2.0 * occ + 2.0), (double)n);
    t.b.cap = t.split ? 16 : 4;   // (rows are read 16 at a time)
    while (t.b.cap < most) t.b.cap *= 2;
    t.b.chains = 4;
    const double room = fmax(256.0 * n, 1073741824.0);
    while (t.b.cap > 1 && 4.0 * ncell * t.b.cap > room) {
        t.b.cap /= 2;
        t.b.chains = 1;
    }
    t.b.cell_step = t.split ? t.b.cap : 1;
    t.b.member_step = t.split ? 1 : ncell;
    const double members = t.lanes > 1 ? 192.0 * t.lanes : fmin(fmax(n / 256.0, 64.0), 192.0);
    t.b.shift = 2;
    while ((2 << t.b.shift) <= t.per * kTileThreads && (2 << t.b.shift) * occ <= members) ++t.b.shift;
    t.tiles = (int)(((long long)ncell + (1 << t.b.shift) - 1) >> t.b.shift);
}

// Device memory of the bins: alloc(int **, count) for each array.
template <class Alloc>
int alloc_bins(int n, int ncell, BinStore &t, Alloc alloc)
{
    int rc = alloc(&t.b.count, (size_t)ncell);
    if (!rc) rc = alloc(&t.b.tab, (size_t)ncell * t.b.cap);
    if (!rc) rc = alloc(&t.b.over, (size_t)n + (size_t)ncell * t.b.chains);
    if (!rc) rc = alloc(&t.b.tile_total, (size_t)t.tiles + 3);   // read by fours
    if (!rc) rc = alloc(&t.next_total, (size_t)t.tiles + 3);
    if (!rc) rc = alloc(&t.perm, (size_t)n);
    return rc;
}

inline void free_bins(BinStore &t)
{
    for (int *p : {t.b.count, t.b.tab, t.b.over, t.b.tile_total, t.next_total, t.perm})
        if (p) (void)hipFree(p);
}

// Empty bins.
inline hipError_t clear_bins(hipStream_t st, int n, int ncell, const BinStore &t)
{
    const size_t tb = sizeof(int) * ((size_t)t.tiles + 3);
    hipError_t e = hipMemsetAsync(t.b.count, 0, sizeof(int) * ncell, st);
    if (e == hipSuccess) e = hipMemsetAsync(t.b.over + n, 0xff, sizeof(int) * t.b.chains * ncell, st);
    if (e == hipSuccess) e = hipMemsetAsync(t.b.tile_total, 0, tb, st);
    if (e == hipSuccess) e = hipMemsetAsync(t.next_total, 0, tb, st);
    return e;
}

}  // namespace psim
