// psim_pairs.hpp -- particle sources, cell tables and the x-run walk shared by
// the pair kernels.
//
// The 27 neighbour cells of the reference's stencil (LJPotential.cpp:154-177)
// are visited as 9 runs along x: for each (dy, dz), y outer and z inner, the
// cells x-1, x, x+1 of that row hold consecutive slots, so the run is one
// slot range (two where the row wraps the periodic boundary, each with its
// own image), candidates in slot order.
#pragma once

#include "psim_device.hpp"

namespace psim {

// Positions in the engine's slot-ordered SoA ([3][N]) with one radius.
struct SoAPos {
    const double *__restrict__ p;
    int N;
    double radius;
    // 32-bit byte offsets (3 x 2^26 doubles stay below 4 GiB)
    __device__ double at(unsigned k) const { return *(const double *)((const char *)p + 8u * k); }
    __device__ double x(int j) const { return at((unsigned)j); }
    __device__ double y(int j) const { return at((unsigned)(N + j)); }
    __device__ double z(int j) const { return at((unsigned)(2 * N + j)); }
    __device__ double rad(int) const { return radius; }
};

// The reference's sortedParticles layout (x,y,z,r per sorted index,
// systemHandling.cpp:79-83).
struct AoS4Pos {
    const double *__restrict__ p;
    __device__ double x(int j) const { return p[4 * (size_t)j]; }
    __device__ double y(int j) const { return p[4 * (size_t)j + 1]; }
    __device__ double z(int j) const { return p[4 * (size_t)j + 2]; }
    __device__ double rad(int j) const { return p[4 * (size_t)j + 3]; }
};

// Engine cell table: start offsets, cell c = [cs[c], cs[c+1]).
struct StartTab {
    const int *__restrict__ cs;
    __device__ void range(int h, int &b, int &e) const
    {
        b = cs[h];
        e = cs[h + 1];
    }
    // slots of the consecutive cells row + lo .. row + hi - 1
    __device__ void row_range(unsigned row, size_t lo, size_t hi, int &b, int &e) const
    {
        const int *__restrict__ r = cs + row;
        b = r[lo];
        e = r[hi];
    }
};

// The reference's cellStartEnd: (start, end) pairs, -1 for empty
// (system.h:166, systemHandling.cpp:60-75).
struct PairTab {
    const int *__restrict__ se;
    __device__ void range(int h, int &b, int &e) const
    {
        b = se[2 * h];
        e = se[2 * h + 1];
        if (b < 0 || e < b) {
            b = 0;
            e = 0;
        }
    }
    // cells are stored in cell order, so consecutive non-empty cells are
    // adjacent: the row's slots run from the first start to the last end
    __device__ void row_range(unsigned row, size_t lo, size_t hi, int &b, int &e) const
    {
        b = 0;
        e = 0;
        for (size_t h = row + lo; h < row + hi; ++h) {
            int hb, he;
            range((int)h, hb, he);
            if (he > hb) {
                if (e == 0) b = hb;
                e = he;
            }
        }
    }
};

// The neighbour cells x-1, x, x+1 (cell x = cx) of row `row` as at most two
// slot segments in stencil order dx = -1, 0, +1: a wrapped end cell is a
// segment of its own with image code 1 (dx = -1 at cx = 0: image +L) or 2
// (dx = +1 at cx = S-1: image -L).  Segment 1 is empty unless the row wraps.
struct XRun {
    int b0, e0, k0, b1, e1, k1;
};

template <class Tab>
__device__ __forceinline__ XRun x_run(const Tab &tab, int row, int cx, int S)
{
    const bool lw = cx == 0, rw = cx == S - 1;
    XRun r;
    tab.row_range((unsigned)row, lw ? S - 1 : cx - 1, lw || rw ? S : cx + 2, r.b0, r.e0);
    r.k0 = lw ? 1 : 0;
    if (lw || rw) {
        tab.row_range((unsigned)row, 0, lw ? 2 : 1, r.b1, r.e1);
    } else {
        r.b1 = 0;   // an interior row is one segment (no table reads for the second)
        r.e1 = 0;
    }
    r.k1 = lw ? 0 : 2;
    return r;
}

// Original particle index of a slot (for error reports).
struct Orig {
    const int *__restrict__ p;
    int stride;
    int off;
    __device__ int operator()(int j) const { return p[stride * j + off]; }
};

__device__ inline double shifted(double xi, int k, double L)
{
    return k == 0 ? xi : (k == 1 ? xi + L : xi - L);
}

}  // namespace psim
