// psim_gather.hpp -- the thread-per-particle pair gather as a wave-wide
// pipeline: candidate lists, a fixed-point cull and balanced pair evaluation.
//
// One lane (or SPLIT lanes) per particle.  A lane's work differs from its
// neighbours' at every level: its 27 cells (LJPotential.cpp:154-177) hold
// between none and dozens of candidates, and between none and a dozen of
// them lie inside the cutoff.  Walked cell by cell, a wave pays the longest
// of its 64 lanes' loops at each cell and one dependent load per candidate.
// Here the stages are separated:
//   1. ranges   the slot ranges of the x-runs (psim_pairs.hpp x_run), three
//               runs (twelve table reads) at a time;
//   2. list     the candidates' slots appended to the lane's column in LDS
//               (no memory access besides LDS);
//   3. cull     the column read four entries at a time, their four positions
//               in flight together, survivors compacted in place.  Positions
//               are the 32-bit box fractions of `upos` (16 bytes per particle
//               with its cell), so one load brings a candidate, the
//               difference of two fractions wraps to the minimum image by
//               itself and needs no image code;
//   4. pairs    the wave's survivors packed into one list and evaluated 64 at
//               a time, whichever lane they belong to: every evaluation runs
//               on a full wave (all but the last), instead of as many rounds
//               as the fullest lane has pairs.  fNet / r and the displacement
//               go through LDS back to the pair's lane, which accumulates
//               them in list order: the sum does not depend on how the pairs
//               were dealt out, and is that of a walk pair by pair.
//
// What bounds it: at 0.4 particles per cell (AO, N = 262,144) a wave issues
// 971 VALU instructions (1,871 with the integrator), against 1,337 for the
// cell-by-cell walk, and waits for a chain of about ten loads; VALU issue (54 %
// of the launch) and the chain share the time.
// Measured on MI355X, the walk first, this second: the pair kernel of the
// 128-replica AO ensemble (1.34 M particles, one launch per class) 4 x 41 us
// and 4 x 22 us, its whole step 220 and 154 us; the N = 262,144 step kernel
// (with the integrator) 34 and 24 us; N = 32,768 (four lanes per particle)
// 14.4 and 11.9 us.  Measured equal or slower: the next three runs' table reads in
// flight during the list stage (39.4 against 39.2 us per step), 5 or 6 waves
// per SIMD with shorter columns (39.5; 6 waves spill), 64 pairs per round.
//
// Neighbour sets are bit-exact with the reference: the cull accepts with a
// margin that covers the fixed-point and FP32 rounding, and the FP64 r^2 of
// every survivor near or beyond the cutoff is re-tested with util::pbcDist's
// own arithmetic (utilities.cpp:79-104) against the strict r^2 < rc^2 of
// LJPotential.cpp:82.
//
// Fractions and the nearest image stand for the walk over the cells only where
// both positions lie in the box.  A pair with one that does not (or is NaN or
// infinite) takes the image that the walk meets it in (walk_image), so that
// it is accepted and evaluated as in the kernels that move positions by cell.
#pragma once

#include "psim_pairs.hpp"

namespace psim {

// Box fraction of a coordinate in 2^-32 (modulo one box).
__device__ __forceinline__ unsigned box_fraction(double x, double inv_L)
{
    return (unsigned)(__builtin_amdgcn_fract(x * inv_L) * 4294967296.0);
}

// The cull's copy of a particle: box fractions and the (global) cell index,
// below 2^31.  Bit 31 of the cell: so many boxes away (or not finite) that the
// fractions, of 53 bits less those of the number of boxes, are no bound.
constexpr unsigned kFarAway = 0x80000000u;
__device__ __forceinline__ uint4 pack_position(double x, double y, double z, int cell,
                                               double inv_L)
{
    const bool near = fabs(x * inv_L) + fabs(y * inv_L) + fabs(z * inv_L) < 65536.0;
    return make_uint4(box_fraction(x, inv_L), box_fraction(y, inv_L), box_fraction(z, inv_L),
                      (unsigned)cell | (near ? 0u : kFarAway));
}

// True for every position that is not in [0, L)^3, with a NaN or an infinity
// too; also for a few that are (-0.0, and x with the high word of L).
__device__ __forceinline__ unsigned high_word(double x) { return (unsigned)__double2hiint(x); }
__device__ __forceinline__ bool maybe_outside(double xi, double yi, double zi, double xj,
                                              double yj, double zj, double L)
{
    return max(max(max(high_word(xi), high_word(yi)), high_word(zi)),
               max(max(high_word(xj), high_word(yj)), high_word(zj))) >= high_word(L);
}

// The particle at (x, y, z), moved to the image in which the walk over its 27
// cells meets slot j.
template <class Tab>
__device__ inline void walk_image(const Geo &g, const Tab &tab, int j, double &x, double &y,
                                  double &z)
{
    const int S = g.S;
    const int cx = cell_1d(x, g.cell, S), cy = cell_1d(y, g.cell, S), cz = cell_1d(z, g.cell, S);
#pragma unroll 1
    for (int m = 0; m < 9; ++m) {
        int ry = cy + m / 3 - 1, rz = cz + m % 3 - 1, ky = 0, kz = 0;
        if (ry < 0) { ry += S; ky = 1; } else if (ry >= S) { ry -= S; ky = 2; }
        if (rz < 0) { rz += S; kz = 1; } else if (rz >= S) { rz -= S; kz = 2; }
        const XRun r = x_run(tab, g.c0 + S * ry + g.S2 * rz, cx, S);
        const bool first = j >= r.b0 && j < r.e0;
        if (first || (j >= r.b1 && j < r.e1)) {
            x = shifted(x, first ? r.k0 : r.k1, g.L);
            y = shifted(y, ky, g.L);
            z = shifted(z, kz, g.L);
            return;
        }
    }
}

// upos[j] by a 32-bit byte offset (16 bytes x 2^26 slots)
__device__ __forceinline__ uint4 upos_at(const uint4 *__restrict__ upos, unsigned j)
{
    return *(const uint4 *)((const char *)upos + (j << 4));
}

// Rows of a lane's candidate column, and pairs evaluated per round.  A wave's
// share of LDS is 256 (rows + 3) + 32 pairs bytes: 10 KiB, 16 waves per CU.
#ifndef PSIM_LIST_ROWS
#define PSIM_LIST_ROWS 21
#endif
#ifndef PSIM_ROUND_PAIRS
#define PSIM_ROUND_PAIRS 128
#endif
constexpr int kListRows = PSIM_LIST_ROWS;
constexpr int kRoundPairs = PSIM_ROUND_PAIRS;
static_assert(kRoundPairs % 64 == 0, "whole waves of pairs");

struct WaveLists {
    unsigned list[(kListRows + 3) * 64];   // [row][lane]; 3 rows of padding
    // the round's pairs: lane << 26 | slot, then (over it, written by the
    // lane that has read it) fNet / r, and the displacement
    union {
        unsigned flat;
        double fr;
    } pair[kRoundPairs];
    double dx[kRoundPairs], dy[kRoundPairs], dz[kRoundPairs];
};

// LDS written by some lanes of the wave is read by others after this.
__device__ __forceinline__ void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Inclusive sum over the lanes of the wave (all 64 active).
__device__ __forceinline__ int wave_inclusive_sum(int x)
{
    x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);   // row_shr:1
    x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);   // row_shr:2
    x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);   // row_shr:4
    x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);   // row_shr:8
    x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);   // row_bcast:15
    x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);   // row_bcast:31
    return x;
}

// One pair of the evaluation stage: fNet / r of particle j on particle i and
// the displacement (FP64 positions), or with statistics the acceptance (fr)
// and the partner's hash (dx).  All are 0 for a pair that is not accepted.
template <int MASK, class ST, class Tab, class Orig_>
__device__ __forceinline__ void eval_pair(const Geo &g, const Pot &p, const Cull &q,
                                          const Tab &tab, double xi,
                                          double yi, double zi, double xj, double yj, double zj,
                                          double size, int si, int j, DevErr *err,
                                          const Orig_ &orig, double &fr, double &dx, double &dy,
                                          double &dz)
{
    fr = dx = dy = dz = 0.0;
    double ex = xj - xi, ey = yj - yi, ez = zj - zi;
    double r2, r, rinv;
    if (!g.exact_mi) {
        // the home position moved to the partner's image (by 0 or +-L, exact
        // product), then the difference
        double hx = fma(rint(ex * q.inv_L), g.L, xi), hy = fma(rint(ey * q.inv_L), g.L, yi),
               hz = fma(rint(ez * q.inv_L), g.L, zi);
        // (this test is 1 % of a step at 262,144 AO particles, 32.0 -> 32.4 us)
        if (maybe_outside(xi, yi, zi, xj, yj, zj, g.L)) {
            hx = xi;
            hy = yi;
            hz = zi;
            walk_image(g, tab, j, hx, hy, hz);
        }
        ex = xj - hx;
        ey = yj - hy;
        ez = zj - hz;
        r2 = fma(ex, ex, fma(ey, ey, ez * ez));
        if (!(r2 < p.rc2_lo)) {
            const double r2x = pbc_dist_ref(xi, yi, zi, xj, yj, zj, g.L, g.half_pbc);
            if (!(r2 < p.rc2_hi && r2x < p.rc2)) return;
        }
        rinv = rsqrt_nr(r2);
        r = r2 * rinv;
    } else {
        // the reference's own arithmetic throughout (S == 3 boxes)
        r2 = pbc_dist_ref(xi, yi, zi, xj, yj, zj, g.L, g.half_pbc);
        if (!(r2 < p.rc2)) return;
        r = sqrt(r2);
        rinv = 1.0 / r;
        ex = min_image_uv(ex, g.L, g.half_uv);
        ey = min_image_uv(ey, g.L, g.half_uv);
        ez = min_image_uv(ez, g.L, g.half_uv);
    }
    if constexpr (ST::kOn) {
        fr = 1.0;
        dx = __longlong_as_double((long long)nbr_hash((unsigned)orig(j)));
        return;
    }
    const double ov = p.ov_factor * size;
    if (r2 < ov * ov * (1.0 + p.ov_band)) {
        const double r2x = pbc_dist_ref(xi, yi, zi, xj, yj, zj, g.L, g.half_pbc);
        if (sqrt(r2x) < ov) report_error(err, 7704, orig(si), orig(j));
    }
    bool nan_ao = false;
    fr = pair_fr<MASK>(p, rinv, r, size, &nan_ao);
    dx = ex;
    dy = ey;
    dz = ez;
    if (nan_ao) report_error(err, 7705, orig(si), orig(j));
}

// Force on the particle of this lane (slot s), shared by SPLIT consecutive
// lanes: lane `sub` gathers the x-runs sub, sub + SPLIT,
// ... of the 9 and gets its partial force (the caller sums the partials).
// Every lane of the wave calls it; `valid` is false on lanes without a
// particle (their s must still be a slot of the system).  upos: box
// fractions and cells of all slots.  With ST = NbrStats the accepted pairs
// are recorded in st instead.
template <int MASK, int SPLIT, class Src, class Tab, class ST = NoStats>
__device__ __forceinline__ void wave_gather(const Geo &g, const Pot &p, const Cull &q,
                                            const Src &src, const Tab &tab,
                                            const uint4 *__restrict__ upos, bool valid, int s,
                                            WaveLists &w, double &fx, double &fy, double &fz,
                                            DevErr *err, const Orig &orig, int sub,
                                            ST *st = nullptr)
{
    const int lane = (int)__lane_id();
    const int S = g.S;
    const int s0 = __builtin_amdgcn_readfirstlane(s);   // slot of lane 0
    const uint4 u = upos_at(upos, (unsigned)s);
    // cell coordinates from the cell index: (c + 1/2) / S^2 is at least
    // 1 / (2 S^2) away from a whole number, far above the rounding of the
    // product (S <= 1290)
    const int c = (int)(u.w & ~kFarAway) - g.c0;
    const int cz = (int)(((double)c + 0.5) * q.inv_S2);
    const int cyx = c - __mul24(cz, g.S2);
    const int cy = (int)(((float)cyx + 0.5f) * q.inv_S);
    const int cx = cyx - __mul24(cy, S);
    // (a particle too far away for the cull takes every candidate; one in the
    // box and one that far away are no pair)
    const float ucut2 = u.w & kFarAway ? INFINITY : q.ucut2;
    unsigned *col = w.list + lane;

    // The cells x-1, x, x+1 of a row as two segments [a0, a1) and [0, b1) of
    // its cells; the second is empty unless the row wraps.  (A lane without a
    // particle has two empty ones: every lane loads the same four table
    // entries per row, with no branch between the loads.)
    const bool lw = cx == 0, rw = cx == S - 1;
    const unsigned a0 = lw ? S - 1 : cx - 1;
    const unsigned a1 = !valid ? a0 : lw || rw ? S : cx + 2;
    const unsigned b1 = !valid ? 0 : lw ? 2 : rw ? 1 : 0;
    // first cell of the home row, and the steps to the rows around it
    const int row0 = g.c0 + __mul24(cy, S) + __mul24(cz, g.S2);
    const int ylo = cy == 0 ? g.S2 - S : -S, yhi = cy == S - 1 ? S - g.S2 : S;
    const int zlo = cz == 0 ? g.ncell - g.S2 : -g.S2, zhi = cz == S - 1 ? g.S2 - g.ncell : g.S2;
    struct Run { int b0, e0, b1, e1; };
    constexpr int kGroups = (9 + 3 * SPLIT - 1) / (3 * SPLIT);
    auto runs = [=](int grp, Run (&r)[3]) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            // run m: y row m / 3, z row m % 3 (SPLIT == 1: group = y row)
            const int m = min(sub + SPLIT * (3 * grp + k), 8);
            const int qy = SPLIT == 1 ? grp : (m * 11) >> 5, qz = SPLIT == 1 ? k : m - 3 * qy;
            const int row = row0 + (qy == 0 ? ylo : 0) + (qy == 2 ? yhi : 0)
                          + (qz == 0 ? zlo : 0) + (qz == 2 ? zhi : 0);
            tab.row_range((unsigned)row, a0, a1, r[k].b0, r[k].e0);
            tab.row_range((unsigned)row, 0, b1, r[k].b1, r[k].e1);
            if (SPLIT > 1 && sub + SPLIT * (3 * grp + k) > 8) r[k] = Run{0, 0, 0, 0};
        }
    };

    int n = 0, nh = 0;   // column length; survivors at its front
    Run cur[3];
    runs(0, cur);
    for (int grp = 0;;) {
        // ---- candidates of the group, as many as the column holds
        bool more = false;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
#pragma unroll
            for (int sg = 0; sg < 2; ++sg) {
                int &b = sg ? cur[k].b1 : cur[k].b0;
                const int e = sg ? cur[k].e1 : cur[k].e0;
                // (a host's table with cells out of row order: b past e)
                const int take = max(0, min(e - b, kListRows - n)), to = b + take;
                // two entries at a time (an odd last one spills into the
                // next free row)
                unsigned *at = col + n * 64;
#pragma unroll 1
                for (; b < to; b += 2, at += 128) {
                    at[0] = (unsigned)b;
                    at[64] = (unsigned)(b + 1);
                }
                n += take;
                b = to;
                more |= b < e;
            }
        }
        const bool again = __any(more);
        if (!again && grp + 1 < kGroups) {
            runs(++grp, cur);
            continue;
        }
        // ---- cull the new entries; the particle itself pads the column (it
        // is skipped as any other copy of itself)
        col[n * 64] = (unsigned)s;
        col[(n + 1) * 64] = (unsigned)s;
        col[(n + 2) * 64] = (unsigned)s;
#pragma unroll 1
        for (int k = nh; k < n; k += 4) {
            unsigned e[4];
            uint4 v[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) e[t] = col[(k + t) * 64];
#pragma unroll
            for (int t = 0; t < 4; ++t) v[t] = upos_at(upos, e[t]);
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const float dx = (float)(int)(v[t].x - u.x), dy = (float)(int)(v[t].y - u.y),
                            dz = (float)(int)(v[t].z - u.z);
                const float r2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
                const bool hit = r2 < ucut2 && e[t] != (unsigned)s;
                col[nh * 64] = e[t];   // rows up to k + t have been read
                nh += hit ? 1 : 0;
            }
        }
        n = nh;
        if (again && !__any(nh > kListRows / 2)) continue;
        // ---- the wave's survivors, kRoundPairs at a time
        const int incl = wave_inclusive_sum(nh);
        const int off = incl - nh;
        const int total = __builtin_amdgcn_readlane(incl, 63);
        for (int t0 = 0; t0 < total; t0 += kRoundPairs) {
            const int lo = max(off, t0), hi = min(off + nh, t0 + kRoundPairs);
#pragma unroll 1
            for (int t = lo; t < hi; ++t)
                w.pair[t - t0].flat = col[(t - off) * 64] | ((unsigned)lane << kIdxBits);
            wave_lds_sync();
            const int cnt = min(total - t0, kRoundPairs);
            for (int b = 0; b < cnt; b += 64) {
                const int t = b + lane;
                const bool act = t < cnt;
                const unsigned e = act ? w.pair[t].flat : ((unsigned)lane << kIdxBits);
                const int i = (int)(e >> kIdxBits), j = (int)(e & kIdxMask);
                const int si = s0 + i / SPLIT;
                if (act) {
                    double fr, dx, dy, dz;
                    eval_pair<MASK, ST>(g, p, q, tab, src.x(si), src.y(si), src.z(si), src.x(j),
                                        src.y(j), src.z(j), src.rad(si) + src.rad(j), si, j, err,
                                        orig, fr, dx, dy, dz);
                    w.pair[t].fr = fr;
                    w.dx[t] = dx;
                    w.dy[t] = dy;
                    w.dz[t] = dz;
                }
            }
            wave_lds_sync();
#pragma unroll 1
            for (int t = lo - t0; t < hi - t0; ++t) {
                if constexpr (ST::kOn) {
                    const bool in = w.pair[t].fr != 0.0;
                    st->count += in ? 1 : 0;
                    st->hash += in ? (unsigned long long)__double_as_longlong(w.dx[t]) : 0ull;
                } else {
                    const double fr = w.pair[t].fr;
                    fx = fma(fr, w.dx[t], fx);
                    fy = fma(fr, w.dy[t], fy);
                    fz = fma(fr, w.dz[t], fz);
                }
            }
            wave_lds_sync();
        }
        n = nh = 0;
        if (!again) break;
    }
}

}  // namespace psim
