// psim_step.hpp -- the step kernels of one system: pair forces (both
// kernel paths), the G&B integrator epilogue and force-only evaluations.
#pragma once

#include <algorithm>
#include <cmath>

#include "psim_brick.hpp"
#include "psim_cells.hpp"
#include "psim_dense.hpp"
#include "psim_gather.hpp"
#include "psim_gpu.h"
#include "psim_pairs.hpp"
#include "psim_stage.hpp"

namespace psim {
namespace {

// Mean particles per cell from which the cell kernels are used.
constexpr double kDenseMinOccupancy = 2.0;
// Below this many particles per cell a wave takes a cell instead of a
// workgroup, in systems of this size: a workgroup's time is mostly the same
// for every cell, a wave's grows with the cell's pairs and is the longer one
// where there are too few cells to fill the chip.  Whole steps (workgroup /
// wave, us) at 2.2 per cell: N = 30,011 54 / 38, 200,000 277 / 141; at 3.0:
// 10,000 26.1 / 26.9, 16,000 32.4 / 28.6, 30,011 45 / 38, 200,000 210 / 137;
// at 3.9: 30,011 38 / 45, 60,000 58 / 59; at 4.8: 200,000 139 / 183.
constexpr double kCellsMaxOccupancy = 3.5;
constexpr int kCellsMin = 12288;
// below this many particles the thread-per-particle kernels use 64-lane
// blocks (256-lane blocks would leave CUs idle: 256 CUs x 4 blocks)
constexpr int kSmallSystem = 256 * 1024;
#ifndef PSIM_SMALL_SPLIT
#define PSIM_SMALL_SPLIT 4
#endif
constexpr int kSmallSplit = PSIM_SMALL_SPLIT;   // lanes per particle below kSmallSystem
// home particles per brick, as a fraction of the lane groups of one workgroup
#ifndef PSIM_BRICK_TARGET
#define PSIM_BRICK_TARGET 0.8
#endif
constexpr double kBrickTarget = PSIM_BRICK_TARGET;

// Checks of a psim_params shared by every entry point that takes one.
inline int check_params(const psim_params &P)
{
    if (P.n_particles <= 0 || P.n_particles >= (1 << kIdxBits)) return PSIM_E_ARG;
    // the 27-cell stencil repeats cells for S < 3 (double counting in the
    // reference, LJPotential.cpp:154-169)
    if (P.cells_per_dim < 3 || P.cells_per_dim > 1290) return PSIM_E_UNSUPPORTED;
    if (P.kernel_path < 0 || P.kernel_path > 3) return PSIM_E_ARG;
    if (!(P.box > 0) || !(P.cell_size > 0) || !(P.cutoff > 0) || !(P.dt > 0) ||
        !(P.mass > 0) || P.force_mask <= 0 || P.force_mask > 7)
        return PSIM_E_ARG;
    if ((P.force_mask & PSIM_FORCE_LJ) && !(P.debye_length > 0)) return PSIM_E_ARG;
    return 0;
}

// Pair-kernel path of a system: the cell kernels need S >= 4 (shifted image =
// minimum image) and pay off once cells hold a few particles, a wave per cell
// first, then a workgroup; below that, one thread per particle (bricks of cells per
// workgroup, path 3, give the same bits but measured slower at every sparse
// density).
struct PathChoice {
    bool dense;
    bool cells;    // a wave per cell instead of a workgroup (the same bits)
    bool brick;
    int brick_g;   // lanes per particle of the brick step kernel
    BrickGeo bg;
};
inline PathChoice choose_path(const psim_params &P, const Geo &g)
{
    PathChoice c{};
    const double occupancy = (double)g.n / g.ncell;
    if (P.kernel_path == 1 || P.kernel_path == 3)
        c.dense = false;
    else if (P.kernel_path == 2)
        c.dense = g.S >= 4;
    else
        c.dense = g.S >= 4 && occupancy >= kDenseMinOccupancy;
    c.cells = c.dense && occupancy < kCellsMaxOccupancy && g.n >= kCellsMin;
    c.brick = P.kernel_path == 3;
    c.brick_g = g.n < kSmallSystem ? kSmallSplit : 1;
    c.bg = brick_shape(g.S, occupancy, kBrickTarget * kBrickThreads / c.brick_g);
    return c;
}


struct StepArgs {
    const double *pos, *pos0, *frc, *mem;
    const uint4 *upos;   // box fractions and cells of pos (thread-per-particle kernels)
    const int *id, *cstart;
    const int *prev;     // slot of each particle in pos0 / frc / mem (null: the same slot)
    int x0_raw;          // pos0 holds the positions the last step started from (re-imaged
                         // here against the current ones); npos0 is then not written
    double *npos, *npos0, *nfrc, *nmem;
    double *vel;         // [3][N] by original index
    Bins bins;
    DevErr *err;
    const double *noise; // [6][N] by original index, or null -> Philox
    unsigned long long seed, step;
    int first, do_vel;
    const StepCtl *ctl;  // when set, step / first / do_vel are read from it
    int *pbc;            // [3][N] periodic crossings by original index, or null
};

// G&B epilogue for the particle in slot s with total force F
// (brownianIntegrator.cpp:191-356, particle.cpp:61-99); writes the next state
// at slot s and enters it in its new cell's bin.
// (o = id[s] and ps = prev[s] may be read by the caller ahead of the force
// loop, so that their latency overlaps it: pass them as o_pre / ps_pre.)
template <bool WRITE_F>
__device__ __forceinline__ void integrate_one(const Geo &g, const GB &gb, const StepArgs &a, int s,
                              double fx, double fy, double fz, int o_pre = -1, int ps_pre = -1)
{
    const int N = g.n;
    const int o = o_pre >= 0 ? o_pre : a.id[s];
    const int first = a.ctl ? a.ctl->first : a.first;
    const int do_vel = a.ctl ? a.ctl->do_vel : a.do_vel;
    double z[6];
    if (a.noise) {
#pragma unroll
        for (int k = 0; k < 6; ++k) z[k] = a.noise[(size_t)k * N + o];
    } else {
        philox_normals6(a.seed, a.ctl ? a.ctl->step : a.step, (uint32_t)o, z);
    }
    const double xc[3] = {a.pos[s], a.pos[N + s], a.pos[2 * N + s]};
    const double F[3] = {fx, fy, fz};
    // the previous position, force and memory where the last step left them
    const int ps = ps_pre >= 0 ? ps_pre : (a.prev ? a.prev[s] : s);
    double x0c[3], xn[3], M[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) x0c[d] = a.pos0[d * N + ps];
    if (a.x0_raw) {
        // what the last step would have stored: util::safeMod0 of its start
        // position against its end position, which is this step's start
#pragma unroll
        for (int d = 0; d < 3; ++d) x0c[d] = safe_mod0(x0c[d], xc[d], g.L);
    }
    if (first) {
        // firstStep :200-218
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            M[d] = z[3 + d];
            double v = a.vel[(size_t)d * N + o];
            xn[d] = xc[d] + (v * gb.coeff1 * gb.dt)
                  + (F[d] * gb.coeff3 * gb.dt * gb.dt * gb.m) + (gb.sig1 * M[d]);
        }
    } else {
        // normalStep :238-274
        double Mo[3], Fo[3], Cr[3];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            Mo[d] = a.mem[d * N + ps];
            Fo[d] = a.frc[d * N + ps];
            Cr[d] = gb.sig2 * ((gb.corr * Mo[d]) + (gb.dev * z[d]));
            M[d] = z[3 + d];
        }
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            double q = (gb.c0 * xc[d]);
            q -= (gb.coeff0 * x0c[d]);
            q += (gb.c1 * F[d]);
            q += (gb.c2 * (F[d] - Fo[d]));
            q += (gb.sig1 * M[d]) + (gb.coeff0 * Cr[d]);
            xn[d] = q;
        }
        if (do_vel) {
            // velocityStep :305-354
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                double dx0 = xc[d] - x0c[d];
                double xN = safe_mod(xn[d], g.L);
                double x0 = safe_mod0(xc[d], xN, g.L);
                double dx = xN - x0;
                double vv = dx + dx0;
                vv += (gb.g2 * F[d]);
                vv -= (gb.g3 * (F[d] - Fo[d]));
                vv += (Cr[d] - gb.sig1 * M[d]);
                vv *= gb.g4;
                a.vel[(size_t)d * N + o] = vv;
            }
        }
    }
    bool bad = false;
    double xw[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        xw[d] = safe_mod(xn[d], g.L);
        double x0n = safe_mod0(xc[d], xw[d], g.L);
        bad |= (xw[d] < 0.0) || (xw[d] >= g.L);
        if (a.pbc) {
            // analysisManager::updateParticlePBC (analysisTracker.cpp:38-56):
            // the re-imaged previous position leaves the box exactly when the
            // particle crossed a face this step
            if (x0n < 0)
                a.pbc[(size_t)d * N + o] += 1;
            else if (x0n > g.L)
                a.pbc[(size_t)d * N + o] -= 1;
        }
        a.npos[d * N + s] = xw[d];
        if (!a.x0_raw) a.npos0[d * N + s] = x0n;
        if (WRITE_F) a.nfrc[d * N + s] = F[d];
        a.nmem[d * N + s] = M[d];
    }
    if (bad) report_error(a.err, 7703, o, -1);
    int k = g.c0 + cell_1d(xw[0], g.cell, g.S) + g.S * cell_1d(xw[1], g.cell, g.S)
          + g.S2 * cell_1d(xw[2], g.cell, g.S);
    bin_particle(a.bins, N, s, k);
}

// integrate_one<true> with four consecutive lanes per particle: lane sub =
// 0..2 makes one Box-Muller pair and takes one dimension, with that component
// f of the force; lane 3 only takes part in the exchanges.  The operations on
// a value are integrate_one's, so the results are the same bits.
// The epilogue is some thousand FP64 instructions, most of them noise; on one
// lane in four every wave still issues them all.  A step before -> after:
// 30,011 LJ 26.7 -> 24.5 us, 60,000 AO 19.6 -> 18.1; a fit iteration at 32,768
// AO 7.05 -> 6.78 ms.  (The separate integrator of the dense path gains
// nothing from it: it waits for memory.  4,096 LJ+CAL 18.8 -> 18.25, 2,000
// and 16,500 no difference, a single step of 1,000 0.9 us slower.)
__device__ __forceinline__ void integrate_quad(const Geo &g, const GB &gb, const StepArgs &a,
                                               int s, bool valid, int sub, int o, int ps,
                                               double f)
{
    const int N = g.n;
    const int first = a.ctl ? a.ctl->first : a.first;
    const int do_vel = a.ctl ? a.ctl->do_vel : a.do_vel;
    const int d = sub < 3 ? sub : 2;
    const bool mine = valid && sub < 3;
    const double xc = a.pos[d * N + s];
    double x0c = a.pos0[d * N + ps];
    const double Mo = a.mem[d * N + ps], Fo = a.frc[d * N + ps];
    double zc, M;   // normals d and 3 + d of the particle
    if (a.noise) {
        zc = a.noise[(size_t)d * N + o];
        M = a.noise[(size_t)(3 + d) * N + o];
    } else {
        double za, zb;   // normals 2 sub and 2 sub + 1
        philox_pair(a.seed, a.ctl ? a.ctl->step : a.step, (uint32_t)o, d, za, zb);
        const int base = (int)(threadIdx.x & 63u) & ~3;
        // 0, 1, 2 come from lanes 0, 0, 1; 3, 4, 5 from lanes 1, 2, 2
        const double ca = __shfl(za, base + (d >> 1), 64), cb = __shfl(zb, base, 64);
        const double ma = __shfl(za, base + 2, 64), mb = __shfl(zb, base + 1 + (d >> 1), 64);
        zc = d == 1 ? cb : ca;
        M = d == 1 ? ma : mb;
    }
    if (a.x0_raw) x0c = safe_mod0(x0c, xc, g.L);
    double xn;
    if (first) {
        const double v = a.vel[(size_t)d * N + o];
        xn = xc + (v * gb.coeff1 * gb.dt) + (f * gb.coeff3 * gb.dt * gb.dt * gb.m) +
             (gb.sig1 * M);
    } else {
        const double Cr = gb.sig2 * ((gb.corr * Mo) + (gb.dev * zc));
        xn = (gb.c0 * xc);
        xn -= (gb.coeff0 * x0c);
        xn += (gb.c1 * f);
        xn += (gb.c2 * (f - Fo));
        xn += (gb.sig1 * M) + (gb.coeff0 * Cr);
        if (do_vel) {
            const double xN = safe_mod(xn, g.L);
            const double dx = xN - safe_mod0(xc, xN, g.L);
            double vv = dx + (xc - x0c);
            vv += (gb.g2 * f);
            vv -= (gb.g3 * (f - Fo));
            vv += (Cr - gb.sig1 * M);
            vv *= gb.g4;
            if (mine) a.vel[(size_t)d * N + o] = vv;
        }
    }
    const double xw = safe_mod(xn, g.L);
    const double x0n = safe_mod0(xc, xw, g.L);
    int k = cell_1d(xw, g.cell, g.S) * (d == 0 ? 1 : d == 1 ? g.S : g.S2);
    k = sub < 3 ? k : g.c0;
    k += __shfl_xor(k, 1, 64);
    k += __shfl_xor(k, 2, 64);
    if (mine) {
        if (a.pbc) {
            if (x0n < 0)
                a.pbc[(size_t)d * N + o] += 1;
            else if (x0n > g.L)
                a.pbc[(size_t)d * N + o] -= 1;
        }
        a.npos[d * N + s] = xw;
        if (!a.x0_raw) a.npos0[d * N + s] = x0n;
        a.nfrc[d * N + s] = f;
        a.nmem[d * N + s] = M;
        if ((xw < 0.0) || (xw >= g.L)) report_error(a.err, 7703, o, -1);
    }
    if (valid && sub == 0) bin_particle(a.bins, N, s, k);
}

// Thread-per-particle step (sparse systems and S < 4); with SPLIT > 1,
// SPLIT lanes per particle share its 27 neighbour cells (small systems,
// where one lane per particle leaves most SIMDs idle and each lane waits
// on 27 dependent cell lookups).
template <int MASK, int BLOCK, int SPLIT = 1>
__global__ __launch_bounds__(BLOCK) void k_step(Geo g, Pot p, Cull q, GB gb,
                                                double radius, StepArgs a)
{
    static_assert(SPLIT == 1 || SPLIT == 4, "lane groups");
    __shared__ WaveLists lists[BLOCK / 64];
    const int t = xcd_block() * BLOCK + threadIdx.x;
    const int sub = t % SPLIT;
    int s = t / SPLIT;
    if (__builtin_amdgcn_readfirstlane(s) >= g.n) return;   // whole waves
    const bool valid = s < g.n;
    s = valid ? s : g.n - 1;
    const int N = g.n;
    // the integrator's index loads, in flight during the force loop
    const int o = a.id[s], ps = a.prev ? a.prev[s] : s;
    double fx = 0.0, fy = 0.0, fz = 0.0;
    wave_gather<MASK, SPLIT>(g, p, q, SoAPos{a.pos, N, radius}, StartTab{a.cstart}, a.upos, valid,
                             s, lists[threadIdx.x >> 6], fx, fy, fz, a.err, Orig{a.id, 1, 0},
                             sub);
    if constexpr (SPLIT == 4) {
        fx = split_sum<SPLIT>(fx);
        fy = split_sum<SPLIT>(fy);
        fz = split_sum<SPLIT>(fz);
        integrate_quad(g, gb, a, s, valid, sub, o, ps, sub == 0 ? fx : sub == 1 ? fy : fz);
        return;
    }
    if (sub != 0 || !valid) return;
    integrate_one<true>(g, gb, a, s, fx, fy, fz, o, ps);
}

// Brick-per-workgroup step (sparse systems): G lanes per home particle, the
// G&B epilogue fused as in k_step (same result as k_step<MASK, *, G>).
template <int MASK, int G>
__global__ __launch_bounds__(kBrickThreads) void k_step_brick(Geo g, Pot p, GB gb,
                                                              double radius, BrickGeo bg,
                                                              int per_xcd, StepArgs a)
{
    __shared__ BrickShared sh;
    const int b = xcd_cell(blockIdx.x, per_xcd);
    if (b >= bg.nbricks) return;
    auto epi = [&](int s, double fx, double fy, double fz) {
        integrate_one<true>(g, gb, a, s, fx, fy, fz);
    };
    if (g.exact_mi)
        brick_forces<MASK, true, G>(g, p, radius, a.pos, a.cstart, a.id, a.err, bg, b, sh, epi);
    else
        brick_forces<MASK, false, G>(g, p, radius, a.pos, a.cstart, a.id, a.err, bg, b, sh, epi);
}

// Cell-per-workgroup forces for the step (dense systems, S >= 4): the total
// force on each particle goes to nfrc[slot], where k_integrate picks it up.
// (Fusing the G&B epilogue here would run it on n_i of the workgroup's lanes,
// latency-bound; the separate kernel runs it at full occupancy.)
template <int MASK, int LJN>
__global__ __launch_bounds__(kDenseThreads)
__attribute__((amdgpu_waves_per_eu(dense_waves(MASK, LJN)))) void k_step_dense(
    Geo g, Pot p, double radius, const double *pos, const int *id, const int *cstart,
    double *nfrc, DevErr *err, int per_xcd)
{
    __shared__ DenseShared sh;
    const int c = xcd_cell(blockIdx.x, per_xcd);
    if (c >= g.ncell) return;
    const int home0 = cstart[c];
    const int N = g.n;
    dense_cell_forces<MASK, kDenseThreads, LJN>(g, p, radius, pos, cstart, id, err, c, sh,
                            [=](int i, double Fx, double Fy, double Fz) {
                                const int s = home0 + i;
                                nfrc[s] = Fx;
                                nfrc[N + s] = Fy;
                                nfrc[2 * N + s] = Fz;
                            });
}

// Wave-per-cell forces for the step (the same bits as k_step_dense).
template <int MASK, int LJN>
__global__ __launch_bounds__(kCellBlock)
__attribute__((amdgpu_waves_per_eu(cell_waves(MASK)))) void k_step_cells(Geo g, Pot p, double radius,
                                                           const double *pos, const int *id,
                                                           const int *cstart, double *nfrc,
                                                           DevErr *err, int per_xcd)
{
    const int N = g.n;
    cells_forces<MASK, LJN>(g, p, radius, pos, cstart, id, err, per_xcd,
                            [=](int s, double Fx, double Fy, double Fz) {
                                nfrc[s] = Fx;
                                nfrc[N + s] = Fy;
                                nfrc[2 * N + s] = Fz;
                            });
}

// G&B step for every slot with the force already in nfrc (dense path).
__global__ __launch_bounds__(256) void k_integrate(Geo g, GB gb, StepArgs a)
{
    const int s = blockIdx.x * 256 + threadIdx.x;
    if (s >= g.n) return;
    const int N = g.n;
    integrate_one<false>(g, gb, a, s, a.nfrc[s], a.nfrc[N + s], a.nfrc[2 * N + s]);
}

// Forces only at the current state, written by original index (N x 3).
template <int MASK, int BLOCK, int SPLIT>
__global__ __launch_bounds__(BLOCK) void k_forces(Geo g, Pot p, Cull q, double radius,
                                                   const double *pos, const uint4 *upos,
                                                   const int *id, const int *cstart,
                                                   double *fout, DevErr *err)
{
    __shared__ WaveLists lists[BLOCK / 64];
    const int t = xcd_block() * BLOCK + threadIdx.x;
    const int sub = t % SPLIT;
    int s = t / SPLIT;
    if (__builtin_amdgcn_readfirstlane(s) >= g.n) return;   // whole waves
    const bool valid = s < g.n;
    s = valid ? s : g.n - 1;
    const int N = g.n;
    double fx = 0.0, fy = 0.0, fz = 0.0;
    wave_gather<MASK, SPLIT>(g, p, q, SoAPos{pos, N, radius}, StartTab{cstart}, upos, valid, s,
                             lists[threadIdx.x >> 6], fx, fy, fz, err, Orig{id, 1, 0}, sub);
    fx = split_sum<SPLIT>(fx);
    fy = split_sum<SPLIT>(fy);
    fz = split_sum<SPLIT>(fz);
    if (sub == 0 && valid) store_aos(fout, id[s], fx, fy, fz);
}

// Forces only, brick per workgroup (same result as k_forces with SPLIT = G).
template <int MASK, int G>
__global__ __launch_bounds__(kBrickThreads) void k_forces_brick(Geo g, Pot p, double radius,
                                                                BrickGeo bg, int per_xcd,
                                                                const double *pos,
                                                                const int *id,
                                                                const int *cstart,
                                                                double *fout, DevErr *err)
{
    __shared__ BrickShared sh;
    const int b = xcd_cell(blockIdx.x, per_xcd);
    if (b >= bg.nbricks) return;
    auto epi = [&](int s, double fx, double fy, double fz) {
        store_aos(fout, id[s], fx, fy, fz);
    };
    if (g.exact_mi)
        brick_forces<MASK, true, G>(g, p, radius, pos, cstart, id, err, bg, b, sh, epi);
    else
        brick_forces<MASK, false, G>(g, p, radius, pos, cstart, id, err, bg, b, sh, epi);
}

template <int MASK, int LJN>
__global__ __launch_bounds__(kDenseThreads)
__attribute__((amdgpu_waves_per_eu(dense_waves(MASK, LJN)))) void k_forces_dense(
    Geo g, Pot p, double radius, const double *pos, const int *id, const int *cstart,
    double *fout, DevErr *err, int per_xcd)
{
    __shared__ DenseShared sh;
    const int c = xcd_cell(blockIdx.x, per_xcd);
    if (c >= g.ncell) return;
    const int home0 = cstart[c];
    dense_cell_forces<MASK, kDenseThreads, LJN>(g, p, radius, pos, cstart, id, err, c, sh,
                            [=](int i, double Fx, double Fy, double Fz) {
                                store_aos(fout, id[home0 + i], Fx, Fy, Fz);
                            });
}

// Forces only, wave per cell (the same bits as k_forces_dense).
template <int MASK, int LJN>
__global__ __launch_bounds__(kCellBlock)
__attribute__((amdgpu_waves_per_eu(cell_waves(MASK)))) void k_forces_cells(Geo g, Pot p, double radius,
                                                             const double *pos, const int *id,
                                                             const int *cstart, double *fout,
                                                             DevErr *err, int per_xcd)
{
    cells_forces<MASK, LJN>(g, p, radius, pos, cstart, id, err, per_xcd,
                            [=](int s, double Fx, double Fy, double Fz) {
                                store_aos(fout, id[s], Fx, Fy, Fz);
                            });
}

// Grid of the wave-per-cell kernels and its per_xcd.
inline int cells_per_xcd(int ncell)
{
    constexpr int kWaves = kCellBlock / 64;
    return ((ncell + kWaves - 1) / kWaves + 7) / 8;
}

// ---------------------------------------------------------------------------
// Neighbour-set statistics of the pair kernels: the launch shapes and the
// acceptance code of the step kernels (k_step with BLOCK / SPLIT,
// k_step_dense, k_step_cells, k_step_brick with G), each accepted pair recorded in an
// NbrStats instead of evaluated; counts and partner hashes by original index.
// ---------------------------------------------------------------------------
template <int BLOCK, int SPLIT>
__global__ __launch_bounds__(BLOCK) void k_stats(Geo g, Pot p, Cull q, double radius,
                                                 const double *pos, const uint4 *upos,
                                                 const int *id, const int *cstart,
                                                 NbrStatsOut so)
{
    __shared__ WaveLists lists[BLOCK / 64];
    const int t = xcd_block() * BLOCK + threadIdx.x;
    const int sub = t % SPLIT;
    int s = t / SPLIT;
    if (__builtin_amdgcn_readfirstlane(s) >= g.n) return;   // whole waves
    const bool valid = s < g.n;
    s = valid ? s : g.n - 1;
    const int N = g.n;
    double fx = 0.0, fy = 0.0, fz = 0.0;
    NbrStats st;
    wave_gather<F_CAL, SPLIT>(g, p, q, SoAPos{pos, N, radius}, StartTab{cstart}, upos, valid, s,
                              lists[threadIdx.x >> 6], fx, fy, fz, nullptr, Orig{id, 1, 0}, sub,
                              &st);
    split_stats<SPLIT>(st);
    if (sub == 0 && valid) {
        so.count[id[s]] = st.count;
        so.hash[id[s]] = st.hash;
    }
}

__global__ __launch_bounds__(kDenseThreads)
__attribute__((amdgpu_waves_per_eu(dense_waves(F_CAL)))) void k_stats_dense(
    Geo g, Pot p, double radius, const double *pos, const int *id, const int *cstart,
    NbrStatsOut so, int per_xcd)
{
    __shared__ DenseShared sh;
    const int c = xcd_cell(blockIdx.x, per_xcd);
    if (c >= g.ncell) return;
    dense_cell_forces<F_CAL, kDenseThreads, 0, NbrStats>(
        g, p, radius, pos, cstart, id, nullptr, c, sh, [](int, double, double, double) {}, &so);
}

__global__ __launch_bounds__(kCellBlock)
__attribute__((amdgpu_waves_per_eu(cell_waves(F_CAL)))) void k_stats_cells(
    Geo g, Pot p, double radius, const double *pos, const int *id, const int *cstart,
    NbrStatsOut so, int per_xcd)
{
    cells_forces<F_CAL, 0, NbrStats>(g, p, radius, pos, cstart, id, nullptr, per_xcd,
                                     [](int, double, double, double) {}, &so);
}

template <int G>
__global__ __launch_bounds__(kBrickThreads) void k_stats_brick(Geo g, Pot p, double radius,
                                                               BrickGeo bg, int per_xcd,
                                                               const double *pos, const int *id,
                                                               const int *cstart, NbrStatsOut so)
{
    __shared__ BrickShared sh;
    const int b = xcd_cell(blockIdx.x, per_xcd);
    if (b >= bg.nbricks) return;
    auto epi = [](int, double, double, double) {};
    if (g.exact_mi)
        brick_forces<F_CAL, true, G, NbrStats>(g, p, radius, pos, cstart, id, nullptr, bg, b, sh,
                                               epi, &so);
    else
        brick_forces<F_CAL, false, G, NbrStats>(g, p, radius, pos, cstart, id, nullptr, bg, b,
                                                sh, epi, &so);
}

// The cull's copy of the reference's sortedParticles.
__global__ void k_pack_table(Geo g, double inv_L, const double *sorted4, uint4 *upos)
{
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= g.n) return;
    const AoS4Pos src{sorted4};
    const double x = src.x(s), y = src.y(s), z = src.z(s);
    upos[s] = pack_position(x, y, z,
                            cell_1d(x, g.cell, g.S) + g.S * cell_1d(y, g.cell, g.S)
                                + g.S2 * cell_1d(z, g.cell, g.S), inv_L);
}

// Forces from the reference's host arrays (IForce::getAcceleration over the
// whole system): sorted4, particleHashIndex (hash, orig), cellStartEnd.
template <int MASK, int BLOCK, int SPLIT>
__global__ __launch_bounds__(BLOCK) void k_forces_table(Geo g, Pot p, Cull q, const double *sorted4,
                                                        const uint4 *upos,
                                                        const int *hash_index, const int *cse,
                                                        double *fout, DevErr *err)
{
    __shared__ WaveLists lists[BLOCK / 64];
    const int t = xcd_block() * BLOCK + threadIdx.x;
    const int sub = t % SPLIT;
    int s = t / SPLIT;
    if (__builtin_amdgcn_readfirstlane(s) >= g.n) return;   // whole waves
    const bool valid = s < g.n;
    s = valid ? s : g.n - 1;
    const AoS4Pos src{sorted4};
    const Orig orig{hash_index, 2, 1};
    double fx = 0.0, fy = 0.0, fz = 0.0;
    wave_gather<MASK, SPLIT>(g, p, q, src, PairTab{cse}, upos, valid, s, lists[threadIdx.x >> 6],
                             fx, fy, fz, err, orig, sub);
    fx = split_sum<SPLIT>(fx);
    fy = split_sum<SPLIT>(fy);
    fz = split_sum<SPLIT>(fz);
    if (sub != 0 || !valid) return;
    const int o = orig(s);
    store_aos(fout, o, fx, fy, fz);   // particleForce[3*orig + k] (LJPotential.cpp:179-181)
}


}  // namespace
}  // namespace psim
