// psim_cells.hpp -- wave-per-cell pair kernel for a few particles per cell.
//
// The cell-per-workgroup kernel (psim_dense.hpp) spends 256 lanes, four
// barriers and a pass over 256 partial sums on every cell.  At three
// particles per cell that is some 80 candidates and 38 pairs: most lanes have
// one candidate, one in six of them a pair.  Here a wave owns the cell: it
// stages the candidates, culls them for every home particle with one ballot
// each, evaluates the surviving pairs of the whole cell 64 at a time, and adds
// them up in the order of the other kernel, so the forces are the same bits.
//
// That order: candidate k of a cell with n_i home particles belongs to lane
// group k mod G, G = 256 / n_i; a group's pairs are chained by FMA from its
// last candidate down, the groups g = q mod 4 are added in order for q = 0..3,
// and the four sums in order.  The candidates are therefore staged sorted by
// (g mod 4, g, -k), and the pairs of a home particle come out of the ballots
// in the order in which they are added.
//
// Bound by its instructions, 870 VALU and 650 scalar per wave at 3 per cell, half
// of them spent whatever the cell holds; six waves per SIMD (80 VGPRs, 25 KiB of LDS per
// workgroup) against five at the compiler's own choice: 137 / 151 us a step at
// N = 200,000, three per cell.  The workgroup kernel: 210.
//
// With ST = NbrStats the accepted pairs are recorded instead (the acceptance
// code of the forces).
//
// Cells it is not made for (more than kCellHome particles, fewer than 4 or
// more than kCellCap candidates, more than kCellPairs pairs) are left to the
// workgroup, which does them the other kernel's way afterwards.
#pragma once

#include "psim_dense.hpp"
#include "psim_gather.hpp"

namespace psim {

constexpr int kCellHome = 16;
constexpr int kCellCap = 128;
constexpr int kCellPairs = 128;
constexpr int kCellMasks = (kCellCap + 63) / 64;
static_assert(kDenseThreads == 256, "the order of the sums");

// flags of an entry of the pair list
constexpr int kNewGroup = 0x8000;   // not the group of the pair before
constexpr int kNoPair = 0x4000;     // not inside the cutoff (statistics)

struct CellShared {
    double s[3][kCellCap];    // candidates, shifted to the home cell's image
    double h[3][kCellHome];   // home particles
    double fr[kCellPairs];
    unsigned long long mask[kCellHome][kCellMasks];
    int slot[kCellCap];
    int first[4 * kCellHome + 1];   // first pair of home particle i, q: [4 i + q]
    unsigned short group[kCellCap], self[kCellHome];
    unsigned short list[kCellPairs];   // home particle << 8 | candidate; kNewGroup
    unsigned short cell[kCellCap];     // of candidate k
};

// Forces on the home particles of cell c by one wave; epi(slot, fx, fy, fz)
// takes them, or with statistics *so.  False, with nothing done, where the cell
// does not fit.
template <int MASK, int LJN, class ST, class Epi>
__device__ bool cell_forces(const Geo &g, const Pot &p, double radius,
                            const double *__restrict__ pos, const int *__restrict__ cstart,
                            const int *__restrict__ id, DevErr *err, int c, CellShared &sh,
                            const double *etab, Epi epi, const NbrStatsOut *so)
{
    const int N = g.n, S = g.S;
    const int lane = threadIdx.x & 63;
    const int cl = c - g.c0;
    const int cx = cl % S, cy = (cl / S) % S, cz = cl / g.S2;
    int b = 0, cnt = 0;
    double ex = 0.0, ey = 0.0, ez = 0.0;
    if (lane < 27) {
        int rx = cx + lane / 9 - 1, ry = cy + (lane / 3) % 3 - 1, rz = cz + lane % 3 - 1;
        if (rx < 0) { rx += S; ex = -g.L; } else if (rx >= S) { rx -= S; ex = g.L; }
        if (ry < 0) { ry += S; ey = -g.L; } else if (ry >= S) { ry -= S; ey = g.L; }
        if (rz < 0) { rz += S; ez = -g.L; } else if (rz >= S) { rz -= S; ez = g.L; }
        const int q = g.c0 + rx + S * ry + g.S2 * rz;
        b = cstart[q];
        cnt = cstart[q + 1] - b;
    }
    const int home0 = __builtin_amdgcn_readlane(b, 13);
    const int ni = __builtin_amdgcn_readlane(cnt, 13);
    if (ni == 0) return true;
    if (ni > kCellHome) return false;
    int incl = cnt;
#pragma unroll
    for (int d = 1; d < 32; d <<= 1) {
        const int y = __shfl_up(incl, d, 64);
        if (lane >= d) incl += y;
    }
    const int M = __builtin_amdgcn_readlane(incl, 26);
    if (M < 4 || M > kCellCap) return false;

    // the place of candidate k in the order of the sums: group, and with t =
    // k / G its turn from the group's end; groups below r have nmax members,
    // the others one less
    const int G = kDenseThreads / ni;
    const float inv_G = 1.0f / (float)G;
    const int nmax = (M + G - 1) / G, r = M - (nmax - 1) * G;
    auto longer = [&](int q) { return max(r - q + 3, 0) >> 2; };   // of groups q mod 4
    int qs[4];
    qs[0] = 0;
#pragma unroll
    for (int q = 0; q < 3; ++q) qs[q + 1] = qs[q] + ((G - q + 3) >> 2) * (nmax - 1) + longer(q);

    for (int t = 0; t < cnt; ++t) sh.cell[incl - cnt + t] = (unsigned short)lane;
    wave_lds_sync();
    for (int k0 = 0; k0 < M; k0 += 64) {
        const int k = k0 + lane;
        const int q27 = sh.cell[min(k, M - 1)];
        const int t = k - __shfl(incl - cnt, q27, 64);
        const int slot = __shfl(b, q27, 64) + t;
        const double sx = __shfl(ex, q27, 64), sy = __shfl(ey, q27, 64),
                     sz = __shfl(ez, q27, 64);
        if (k < M) {
            const double x = pos[slot] + sx, y = pos[N + slot] + sy, z = pos[2 * N + slot] + sz;
            const int turn = (int)(((float)k + 0.5f) * inv_G);
            const int gk = k - turn * G, q = gk & 3, m = gk >> 2;
            const int v = (q == 0 ? qs[0] : q == 1 ? qs[1] : q == 2 ? qs[2] : qs[3]) +
                          m * (nmax - 1) + min(m, longer(q)) + nmax - (gk >= r) - 1 - turn;
            sh.s[0][v] = x;
            sh.s[1][v] = y;
            sh.s[2][v] = z;
            sh.slot[v] = slot;
            sh.group[v] = (unsigned short)gk;
            if (q27 == 13) {
                sh.h[0][t] = x;
                sh.h[1][t] = y;
                sh.h[2][t] = z;
                sh.self[t] = (unsigned short)v;
            }
        }
    }
    wave_lds_sync();
    // ---- cull: a bit per candidate and home particle
    for (int v0 = 0; v0 < M; v0 += 64) {
        const int v = min(v0 + lane, M - 1);
        const bool in = v0 + lane < M;
        const double x = sh.s[0][v], y = sh.s[1][v], z = sh.s[2][v];
        for (int i = 0; i < ni; ++i) {
            const double dx = x - sh.h[0][i], dy = y - sh.h[1][i], dz = z - sh.h[2][i];
            const double r2 = fma(dx, dx, fma(dy, dy, dz * dz));
            const unsigned long long m = __ballot(in && r2 < p.rc2_hi && v != sh.self[i]);
            if (lane == 0) sh.mask[i][v0 >> 6] = m;
        }
    }
    wave_lds_sync();
    // ---- the pairs as a list, and where each run of it starts
    int total = 0;
    for (int i = 0; i < ni; ++i)
        for (int ch = 0; ch * 64 < M; ++ch) {
            const unsigned long long mv = sh.mask[i][ch];
            const unsigned long long m =
                (unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane((int)mv) |
                (unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane((int)(mv >> 32)) << 32;
            const int here = __popcll(m);
            if (total + here > kCellPairs) return false;
            if ((m >> lane) & 1ull)
                sh.list[total + __popcll(m & ((1ull << lane) - 1ull))] =
                    (unsigned short)(i << 8 | (ch * 64 + lane));
            if (lane < 4) {
                const int q0 = lane == 0 ? qs[0] : lane == 1 ? qs[1] : lane == 2 ? qs[2] : qs[3];
                if (q0 >> 6 == ch)
                    sh.first[4 * i + lane] = total + __popcll(m & ((1ull << (q0 & 63)) - 1ull));
            }
            total += here;
        }
    if (lane == 0) sh.first[4 * ni] = total;
    wave_lds_sync();
    // ---- evaluate, 64 pairs at a time
    const double size = 2.0 * radius;
    const double ov = p.ov_factor * size;
    const double ov2_hi = ov * ov * (1.0 + p.ov_band);
    for (int e = lane; e < total; e += 64) {
        const int ent = sh.list[e];
        const int i = ent >> 8, v = ent & 255;
        if constexpr (!ST::kOn) {
            const int gp = e ? sh.group[sh.list[e - 1] & 255] : -1;
            if (gp != sh.group[v]) sh.list[e] = (unsigned short)(ent | kNewGroup);
        }
        const double xi = sh.h[0][i], yi = sh.h[1][i], zi = sh.h[2][i];
        const double dx = sh.s[0][v] - xi, dy = sh.s[1][v] - yi, dz = sh.s[2][v] - zi;
        const double r2 = fma(dx, dx, fma(dy, dy, dz * dz));
        bool in = true;
        if (r2 >= p.rc2_lo || r2 < ov2_hi) {
            const int sj = sh.slot[v];
            const double r2x = pbc_dist_ref(xi, yi, zi, pos[sj], pos[N + sj], pos[2 * N + sj],
                                            g.L, g.half_pbc);
            in = !(r2 >= p.rc2_lo) || r2x < p.rc2;
            if (!ST::kOn && in && sqrt(r2x) < p.ov_factor * size)
                report_error(err, 7704, id[home0 + i], id[sj]);
        }
        if constexpr (ST::kOn) {
            sh.fr[e] = __longlong_as_double(
                (long long)(in ? nbr_hash((unsigned)id[sh.slot[v]]) : 0ull));
            if (!in) sh.list[e] = (unsigned short)(ent | kNoPair);
            continue;
        }
        const double rinv = rsqrt_nr(r2);
        bool nan_ao = false;
        const double fr = pair_fr<MASK, true, LJN>(p, rinv, r2 * rinv, size, &nan_ao, etab);
        if (in && nan_ao) report_error(err, 7705, id[home0 + i], id[sh.slot[v]]);
        sh.fr[e] = in ? fr : 0.0;
    }
    wave_lds_sync();
    if constexpr (ST::kOn) {
        if (lane < ni) {
            int pairs = 0;
            unsigned long long hash = 0;
            for (int e = sh.first[4 * lane]; e < sh.first[4 * lane + 4]; ++e) {
                pairs += sh.list[e] & kNoPair ? 0 : 1;
                hash += (unsigned long long)__double_as_longlong(sh.fr[e]);
            }
            const int o = id[home0 + lane];
            so->count[o] = pairs;
            so->hash[o] = hash;
        }
        return true;
    }
    // ---- add: three lanes (dimensions) per home particle and q, the four q
    // of a particle side by side
    for (int w0 = 0; w0 < 4 * ni; w0 += 20) {
        const int d = lane % 3, w = w0 + lane / 3;
        const bool act = lane < 60 && w < 4 * ni;
        double sum = 0.0;
        if (act) {
            const double xi = sh.h[d][w >> 2];
            double part = 0.0;
            const int e1 = sh.first[w + 1];
            int e = sh.first[w];
            int ent = sh.list[min(e, kCellPairs - 1)];
            while (e < e1) {
                const int v = ent & 255;
                const double f = sh.fr[e], dx = sh.s[d][v] - xi;
                if (ent & kNewGroup) {
                    sum += part;
                    part = 0.0;
                }
                ++e;
                ent = sh.list[min(e, kCellPairs - 1)];
                part = fma(f, dx, part);
            }
            sum += part;
        }
        const double s1 = __shfl(sum, lane + 3, 64), s2 = __shfl(sum, lane + 6, 64),
                     s3 = __shfl(sum, lane + 9, 64);
        const double F = ((sum + s1) + s2) + s3;
        const double Fy = __shfl(F, lane + 1, 64), Fz = __shfl(F, lane + 2, 64);
        if (act && d == 0 && (w & 3) == 0) epi(home0 + (w >> 2), F, Fy, Fz);
    }
    return true;
}

constexpr int kCellBlock = 256;
// Waves per SIMD the registers are held to: six, as many as the LDS allows; LJ
// with AO would spill.
constexpr int cell_waves(int mask) { return (mask & F_LJ) && (mask & F_AO) ? 5 : 6; }
union CellsShared {
    CellShared w[kCellBlock / 64];
    DenseShared d;
};

// The cells of one workgroup, one per wave, then those that did not fit by
// the whole workgroup.
template <int MASK, int LJN, class ST = NoStats, class Epi>
__device__ __forceinline__ void cells_forces(const Geo &g, const Pot &p, double radius,
                                             const double *__restrict__ pos,
                                             const int *__restrict__ cstart,
                                             const int *__restrict__ id, DevErr *err, int per_xcd,
                                             Epi epi, const NbrStatsOut *so = nullptr)
{
    __shared__ CellsShared sh;
    __shared__ double etab[64];
    __shared__ int left[kCellBlock / 64];
    if (threadIdx.x < 64) etab[threadIdx.x] = kExp2Tab[threadIdx.x];
    __syncthreads();
    const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int c = xcd_cell(blockIdx.x, per_xcd) * (kCellBlock / 64) + w;
    const bool done = c >= g.ncell ||
                      cell_forces<MASK, LJN, ST>(g, p, radius, pos, cstart, id, err, c, sh.w[w],
                                                 etab, epi, so);
    if ((threadIdx.x & 63) == 0) left[w] = done ? -1 : c;
    __syncthreads();
    for (int k = 0; k < kCellBlock / 64; ++k) {
        const int q = left[k];
        if (q < 0) continue;
        const int home0 = cstart[q];
        dense_cell_forces<MASK, kDenseThreads, LJN, ST>(
            g, p, radius, pos, cstart, id, err, q, sh.d,
            [=](int i, double fx, double fy, double fz) { epi(home0 + i, fx, fy, fz); }, so);
    }
}

}  // namespace psim
