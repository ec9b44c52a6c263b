// psim_bins.hpp -- the bins that a step's integrator enters every particle in
// and the cell rebuild (k_rebuild) takes them from: storage and shape.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>

#include "psim_device.hpp"

namespace psim {

constexpr int kTileCells = 1024;   // most cells of a tile: four per thread of k_rebuild

// The bins of a system or a stack of systems, and the shape of their tiles.
struct BinStore {
    Bins b{};
    int *next_total = nullptr, *perm = nullptr;
    int tiles = 0, lanes = 1;   // lanes: k_rebuild's U
};

// Row length and tiles for n particles in ncell cells of at most
// cell_volume (in cubed particle diameters).  A row holds what hard particles
// can pack into a cell or four times the mean and a few, whichever is less: a
// longer chain costs time, not correctness.  A tile holds the cells of about
// 1/256 of the particles (a workgroup per compute unit), at least 64 and at
// most 192 per particle of a lane.  Lanes move two particles from 131,072 on
// (a step at 262,144: one 35.4 us, two 33.9, four 33.9; at 32,768 two are
// 10 % slower than one) and four from 1,048,576 (2,097,152: one 861 us, two
// 841, four 829).  Tiles of half or twice as many particles: no difference.
inline void shape_bins(int n, int ncell, double cell_volume, BinStore &t)
{
    const double occ = (double)n / ncell;
    const double most = fmin(fmin(1.25 * cell_volume + 1.0, 4.0 * occ + 8.0), (double)n);
    t.b.cap = 4;
    while (t.b.cap < most) t.b.cap *= 2;
    t.lanes = n >= (1 << 20) ? 4 : n >= (1 << 17) ? 2 : 1;
    const double members = t.lanes > 1 ? 192.0 * t.lanes : fmin(fmax(n / 256.0, 64.0), 192.0);
    t.b.shift = 2;
    while ((2 << t.b.shift) <= kTileCells && (2 << t.b.shift) * occ <= members) ++t.b.shift;
    t.tiles = (int)(((long long)ncell + (1 << t.b.shift) - 1) >> t.b.shift);
}

// Device memory of the bins: alloc(int **, count) for each array.
template <class Alloc>
int alloc_bins(int n, int ncell, BinStore &t, Alloc alloc)
{
    int rc = alloc(&t.b.count, (size_t)ncell);
    if (!rc) rc = alloc(&t.b.tab, (size_t)ncell * t.b.cap);
    if (!rc) rc = alloc(&t.b.over, (size_t)n + ncell);
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
    if (e == hipSuccess) e = hipMemsetAsync(t.b.over + n, 0xff, sizeof(int) * ncell, st);
    if (e == hipSuccess) e = hipMemsetAsync(t.b.tile_total, 0, tb, st);
    if (e == hipSuccess) e = hipMemsetAsync(t.next_total, 0, tb, st);
    return e;
}

}  // namespace psim
