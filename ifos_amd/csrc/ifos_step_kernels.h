// ifos_step_kernels.h -- fused time-step kernels of the native engine.  Each
// stencil order is compiled in a file of its own (ifos_order1.hip ..
// ifos_order6.hip); ifos_step.hip holds the launch entry points.
//
// One time step is two kernels:
//   k_vel_step   velocity update (src/update_v_PML.c) + the point forces or
//                adjoint residual injection that follow it (:553-578) + the
//                acceleration snapshot (forward) or the adjoint vxp1 update
//   k_str_step   stress update (src/update_s_*_PML.c) + explosive source
//                (src/psource.c) + free surface (src/surface_*_PML.c) +
//                snapshot store (src/IFOS2D.c:1805-1871) or zero-lag
//                correlation (:2381-2419) + receiver sampling
//                (src/seismo_ssg.c) + stability probe
// Each launch advances every active shot slot (one shot of the same model per
// slot).  Work items are (tile, group of spb slots) pairs; a thread owns one
// cell of a 64x8 tile and loops over the slots of its group, loading the
// cell's materials once.  Point sources and receivers are looked up by cell
// (PointMap), in tiles that hold any.  The free surface needs the new
// stresses of rows 2..N+1 of its column: tiles are 8 rows high and N <= 6, so
// the top tile row holds them; they are exchanged through LDS after a barrier.
// The arithmetic is the per-cell code of ifos_cellmath.h, bit-identical to
// the reference.
#pragma once
#include <algorithm>

#include "ifos_stepdev.h"

namespace ifos {

static int step_flags(const StepArgs &a, int k)
{
    const int D = a.DTINV > 0 ? a.DTINV : 1;
    int f = 0;
    if (a.sw == 0 && (a.snap[0] || a.snap16[0]) && (a.base ? k % D == 0 : (k - 1) % D == 0)) f |= kSnapStep;
    if (a.sw == 1 && (a.base ? (k + 1) % D == 0 : (a.NT - k) % D == 0)) f |= kCorrStep;
    if (a.sw == 0) f |= kForward;
    if (a.sw == 1 && a.VELOCITY == 0) f |= kAdjInt;
    if (a.wacc || a.wacc64) f |= kEnergy;
    return f;
}

// a step whose kernels need no more than the update, the sources and the
// receivers: most steps of a run (every step but each DTINV-th of the
// forward run with snapshots and of the adjoint run with VELOCITY 1)
static bool lean_step(int flags) { return (flags & ~kForward) == 0; }

// velocity step of one cell of slot s
template <int N>
__device__ __forceinline__ void vel_cell(const StepArgs &a, int s, int blk, int i, int j, bool live, long c, long e,
                                         int nt, int flags, float rip, float rjp, float (*s_red)[kTileY])
{
    const StepGeom &g = a.g;
    const int P = g.pitch;
    const long wo = (long)s * a.ws, po = (long)s * a.pss;
    const auto vxs = gmem(a.vx) + wo, vys = gmem(a.vy) + wo;
    float sxx_x = 0.0f, sxy_x = 0.0f, sxy_y = 0.0f, syy_y = 0.0f, vx0 = 0.0f, vy0 = 0.0f;
    if (live) {
        stress_derivs<N>(g.hc, a.sxx + wo + c, a.syy + wo + c, a.sxy + wo + c, P, sxx_x, sxy_x, sxy_y, syy_y);
        cpml_velocity(g, j, i, a.psi_sxx_x + po, a.psi_sxy_x + po, a.psi_syy_y + po, a.psi_sxy_y + po, sxx_x, sxy_x,
                      sxy_y, syy_y);
        vx0 = vxs[c];
        vy0 = vys[c];
    }
    const int p0 = live ? first_point(a, a.inj, s, e, tile_has(a.inj, s, a.nbx * a.nby, blk)) : -1;
    if (flags & kForward) {
        if (flags & kSnapStep) {
            const float val[2] = {vel_rate(rip, sxx_x + sxy_y, g.DH), vel_rate(rjp, sxy_x + syy_y, g.DH)};
            snap_store<2>(a, s, 0, (nt - 1) / a.DTINV, e, blk, live, val, s_red);
        }
    } else if (!live) {
    } else if (flags & kAdjInt) {
        gmem(a.vxp1)[wo + c] += vx0 * g.DT;
        gmem(a.vyp1)[wo + c] += vy0 * g.DT;
    } else if (flags & kCorrStep) {
        gmem(a.vxp1)[wo + c] = vx0;
        gmem(a.vyp1)[wo + c] = vy0;
    }
    if (!live) return;
    float vx = vel_new(vx0, g.DT, rip, sxx_x + sxy_y, g.DH);
    float vy = vel_new(vy0, g.DT, rjp, sxy_x + syy_y, g.DH);

    // point forces (forward) / residual injection (adjoint) at this cell, in order
    for (int l = p0; l >= 0; l = gmem(a.inj.next)[l]) inject(a, l, nt, rip, rjp, vx, vy);
    vxs[c] = vx;
    vys[c] = vy;
    if (g.BOUNDARY) wrap_pair<N>(g, vys, vxs, c, i, vy, vx);
    // energy of the new particle velocities (eprecond, src/eprecond.c:8-21)
    if (flags & kEnergy) {
        if (a.wacc64) {
            const auto W = gmem(a.wacc64) + (long)s * a.wacs;
            W[e] += ((double)vx * (double)vx) + ((double)vy * (double)vy);
        } else {
            const auto W = gmem(a.wacc) + (long)s * a.wacs;
            W[e] += ((vx * vx) + (vy * vy));
        }
    }
}

// velocity step of the R vertically adjacent cells (rows j .. j+R-1) of an
// R-row thread, slot s; the same arithmetic as vel_cell for each cell.  All
// loads of the R cells issue before any store, so their memory latencies
// overlap; live[r] implies live[r-1].
// Derivs(sxx_x, sxy_x, sxy_y, syy_y) fills the stress derivatives of the R
// cells (called only when live[0]): from global memory (vel_cell_rows) or
// from the workgroup's LDS copy of the tile (k_vel_step_lds).
template <int N, int R, typename Derivs>
__device__ __forceinline__ void vel_rows_with(const StepArgs &a, int s, int blk, int i, int j, const bool (&live)[R],
                                              long c, long e, int nt, int flags, const float (&rip)[R],
                                              const float (&rjp)[R], float (*s_red)[kTileY], Derivs derivs)
{
    const StepGeom &g = a.g;
    const int P = g.pitch, NX = g.NX;
    const long wo = (long)s * a.ws, po = (long)s * a.pss;
    const auto vxs = gmem(a.vx) + wo, vys = gmem(a.vy) + wo;
    float sxx_x[R], sxy_x[R], sxy_y[R], syy_y[R], vx0[R], vy0[R];
#pragma unroll
    for (int r = 0; r < R; r++) sxx_x[r] = sxy_x[r] = sxy_y[r] = syy_y[r] = vx0[r] = vy0[r] = 0.0f;
    if (live[0]) {
        derivs(sxx_x, sxy_x, sxy_y, syy_y);
#pragma unroll
        for (int r = 0; r < R; r++)
            if (live[r]) {
                vx0[r] = vxs[c + r * P];
                vy0[r] = vys[c + r * P];
            }
#pragma unroll
        for (int r = 0; r < R; r++)
            if (live[r])
                cpml_velocity(g, j + r, i, a.psi_sxx_x + po, a.psi_sxy_x + po, a.psi_syy_y + po, a.psi_sxy_y + po,
                              sxx_x[r], sxy_x[r], sxy_y[r], syy_y[r]);
    }
    if (flags & kForward) {
        if (flags & kSnapStep) {
            float val[R][2];
#pragma unroll
            for (int r = 0; r < R; r++) {
                val[r][0] = vel_rate(rip[r], sxx_x[r] + sxy_y[r], g.DH);
                val[r][1] = vel_rate(rjp[r], sxy_x[r] + syy_y[r], g.DH);
            }
            snap_store_rows<2, R>(a, s, 0, (nt - 1) / a.DTINV, e, blk, live, val, s_red);
        }
    } else if (flags & kAdjInt) {
#pragma unroll
        for (int r = 0; r < R; r++)
            if (live[r]) {
                gmem(a.vxp1)[wo + c + r * P] += vx0[r] * g.DT;
                gmem(a.vyp1)[wo + c + r * P] += vy0[r] * g.DT;
            }
    } else if (flags & kCorrStep) {
#pragma unroll
        for (int r = 0; r < R; r++)
            if (live[r]) {
                gmem(a.vxp1)[wo + c + r * P] = vx0[r];
                gmem(a.vyp1)[wo + c + r * P] = vy0[r];
            }
    }
    if (!live[0]) return;
    float vx[R], vy[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        vx[r] = vel_new(vx0[r], g.DT, rip[r], sxx_x[r] + sxy_y[r], g.DH);
        vy[r] = vel_new(vy0[r], g.DT, rjp[r], sxy_x[r] + syy_y[r], g.DH);
    }
    // point forces / residual injection of these cells, in order
    if (tile_has(a.inj, s, a.nbx * a.nby, blk)) {
#pragma unroll
        for (int r = 0; r < R; r++)
            if (live[r])
                for (int l = first_point(a, a.inj, s, e + r * NX, true); l >= 0; l = gmem(a.inj.next)[l])
                    inject(a, l, nt, rip[r], rjp[r], vx[r], vy[r]);
    }
#pragma unroll
    for (int r = 0; r < R; r++)
        if (live[r]) {
            vxs[c + r * P] = vx[r];
            vys[c + r * P] = vy[r];
            if (g.BOUNDARY) wrap_pair<N>(g, vys, vxs, c + r * P, i, vy[r], vx[r]);
        }
    if (flags & kEnergy) {
        if (a.wacc64) {
            const auto W = gmem(a.wacc64) + (long)s * a.wacs;
#pragma unroll
            for (int r = 0; r < R; r++)
                if (live[r])
                    W[e + r * NX] += ((double)vx[r] * (double)vx[r]) + ((double)vy[r] * (double)vy[r]);
        } else {
            const auto W = gmem(a.wacc) + (long)s * a.wacs;
#pragma unroll
            for (int r = 0; r < R; r++)
                if (live[r]) W[e + r * NX] += ((vx[r] * vx[r]) + (vy[r] * vy[r]));
        }
    }
}

template <int N, int R>
__device__ __forceinline__ void vel_cell_rows(const StepArgs &a, int s, int blk, int i, int j, const bool (&live)[R],
                                              long c, long e, int nt, int flags, const float (&rip)[R],
                                              const float (&rjp)[R], float (*s_red)[kTileY])
{
    const StepGeom &g = a.g;
    const long wo = (long)s * a.ws;
    vel_rows_with<N, R>(a, s, blk, i, j, live, c, e, nt, flags, rip, rjp, s_red,
                        [&](float(&sxx_x)[R], float(&sxy_x)[R], float(&sxy_y)[R], float(&syy_y)[R]) {
                            // the padded grid holds rows 1-H .. NY+H with H = N+1; with
                            // j <= NY, R = 2 reads up to row NY+N+1 and larger R clamp to it
                            stress_derivs_rows<N, R>(g.hc, a.sxx + wo + c, a.syy + wo + c, a.sxy + wo + c, g.pitch,
                                                     g.NY + N + 1 - j, sxx_x, sxy_x, sxy_y, syy_y);
                        });
}

// RY = 1: a 64x8 block, one cell per thread.  RY = 2 or 4: a 64x(8/RY)
// block, each thread owns rows RY*ty .. RY*ty+RY-1 of the 64x8 tile
// (vel_cell_rows).
template <int N, int SPB, int RY, bool LEAN>
__global__ __launch_bounds__(512) void k_vel_step(const StepArgs *__restrict__ pa, int k, int persistent, int flags_)
{
    // LEAN: a step with no snapshot, correlation, adjoint integration or
    // energy sum (lean_step), compiled without that code and its registers
    const int flags = LEAN ? (flags_ & kForward) : flags_;
    const StepArgs &a = *pa;
    __shared__ float s_red[2][kTileY];
    const StepGeom &g = a.g;
    const ItemMap m = item_map(a);
    const int nt = step_number(a, k);
    int first, end, stride;
    work_range(m, m.ntiles * m.ngroups, persistent != 0, first, end, stride);
    for (int it = first; it < end; it += stride) {
        int blk, s0;
        item_of(m, it, SPB, blk, s0);
        // uniform across the workgroup: keep them in scalar registers
        blk = __builtin_amdgcn_readfirstlane(blk);
        s0 = __builtin_amdgcn_readfirstlane(s0);
        const int by = (int)fdiv(blk, m.nbx_mul, m.nbx_sh), bx = blk - by * m.nbx;
        const int i = bx * kTileX + threadIdx.x + 1;
        const int j = by * kTileY + RY * threadIdx.y + 1;
        const long c = (long)j * g.pitch + i;
        const long e = (long)(j - 1) * g.NX + (i - 1);
        if constexpr (RY == 1) {
            const bool live = i <= g.NX && j <= g.NY;
            const float rip = live ? gmem(a.rip)[c] : 0.0f, rjp = live ? gmem(a.rjp)[c] : 0.0f;
#pragma unroll
            for (int u = 0; u < SPB; u++)
                if (s0 + u < m.nslots) vel_cell<N>(a, s0 + u, blk, i, j, live, c, e, nt, flags, rip, rjp, s_red);
        } else {
            bool live[RY];
            float rip[RY], rjp[RY];
#pragma unroll
            for (int r = 0; r < RY; r++) {
                live[r] = i <= g.NX && j + r <= g.NY;
                // unconditional loads, then a select: live lanes read their
                // own cell, the others cell (1, 1), which every grid has (no
                // per-lane branch, so the pointers are loaded once)
                const long ci = live[r] ? c + r * g.pitch : (long)g.pitch + 1;
                const float vr = gmem(a.rip)[ci], vj = gmem(a.rjp)[ci];
                rip[r] = live[r] ? vr : 0.0f;
                rjp[r] = live[r] ? vj : 0.0f;
            }
#pragma unroll
            for (int u = 0; u < SPB; u++)
                if (s0 + u < m.nslots)
                    vel_cell_rows<N, RY>(a, s0 + u, blk, i, j, live, c, e, nt, flags, rip, rjp, s_red);
        }
    }
}

// Velocity step with the tile's stresses staged in LDS: a 64x4 workgroup of
// two-row threads first copies, for its 64x8 tile, sxx (rows j0..j0+7,
// columns i0-N..i0+63+N), sxy (rows j0-N..j0+7+N, same columns) and syy (rows
// j0-N..j0+7+N, columns i0..i0+63) from HBM into LDS with row-contiguous
// loads, then every stencil value comes from LDS.  Coordinates outside the
// padded grid are clamped to its edge; they only feed cells outside the
// model, which are not stored.  Same arithmetic as vel_cell.
template <int N>
struct VelTile {
    static constexpr int W = kTileX + 2 * N;  // LDS column x <-> grid column i0 - N + x
    static constexpr int H = kTileY + 2 * N;  // LDS row y <-> grid row j0 - N + y (sxy, syy)
    float sxx[kTileY][W];                     // LDS row y <-> grid row j0 + y
    float sxy[H][W];
    float syy[H][kTileX];                     // LDS column x <-> grid column i0 + x
};

template <int N>
__device__ __forceinline__ void stage_tile(VelTile<N> &t, const float *sxx_, const float *sxy_, const float *syy_,
                                           int P, int i0, int j0, int NX, int NY)
{
    constexpr int W = VelTile<N>::W, H = VelTile<N>::H;
    const auto sxx = gmem(sxx_), sxy = gmem(sxy_), syy = gmem(syy_);
    const int lo_i = -N, hi_i = NX + N + 1, lo_j = -N, hi_j = NY + N + 1;  // inside the padded grid
    const int tid = threadIdx.y * kTileX + threadIdx.x, nth = kTileX * (kTileY / 2);
    for (int q = tid; q < kTileY * W; q += nth) {
        const int y = q / W, x = q - y * W;
        const int ii = min(max(i0 - N + x, lo_i), hi_i), jj = min(j0 + y, hi_j);
        t.sxx[y][x] = sxx[(long)jj * P + ii];
    }
    for (int q = tid; q < H * W; q += nth) {
        const int y = q / W, x = q - y * W;
        const int ii = min(max(i0 - N + x, lo_i), hi_i), jj = min(max(j0 - N + y, lo_j), hi_j);
        t.sxy[y][x] = sxy[(long)jj * P + ii];
    }
    for (int q = tid; q < H * kTileX; q += nth) {
        const int y = q / kTileX, x = q - y * kTileX;
        const int ii = min(i0 + x, hi_i), jj = min(max(j0 - N + y, lo_j), hi_j);
        t.syy[y][x] = syy[(long)jj * P + ii];
    }
}

template <int N, int SPB>
__global__ __launch_bounds__(256) void k_vel_step_lds(const StepArgs *__restrict__ pa, int k, int persistent,
                                                      int flags)
{
    constexpr int R = 2;
    const StepArgs &a = *pa;
    __shared__ float s_red[2][kTileY];
    __shared__ VelTile<N> t;
    const StepGeom &g = a.g;
    const ItemMap m = item_map(a);
    const int nt = step_number(a, k);
    int first, end, stride;
    work_range(m, m.ntiles * m.ngroups, persistent != 0, first, end, stride);
    for (int it = first; it < end; it += stride) {
        int blk, s0;
        item_of(m, it, SPB, blk, s0);
        blk = __builtin_amdgcn_readfirstlane(blk);
        s0 = __builtin_amdgcn_readfirstlane(s0);
        const int by = (int)fdiv(blk, m.nbx_mul, m.nbx_sh), bx = blk - by * m.nbx;
        const int i0 = bx * kTileX + 1, j0 = by * kTileY + 1;
        const int tx = threadIdx.x, jr = R * threadIdx.y;  // this thread's rows: j0 + jr, j0 + jr + 1
        const int i = i0 + tx, j = j0 + jr;
        const long c = (long)j * g.pitch + i;
        const long e = (long)(j - 1) * g.NX + (i - 1);
        bool live[R];
        float rip[R], rjp[R];
#pragma unroll
        for (int r = 0; r < R; r++) {
            live[r] = i <= g.NX && j + r <= g.NY;
            rip[r] = live[r] ? gmem(a.rip)[c + r * g.pitch] : 0.0f;
            rjp[r] = live[r] ? gmem(a.rjp)[c + r * g.pitch] : 0.0f;
        }
#pragma unroll 1
        for (int u = 0; u < SPB; u++) {
            const int sl = s0 + u;
            if (sl >= m.nslots) break;  // uniform: the whole workgroup leaves together
            const long wo = (long)sl * a.ws;
            __syncthreads();  // the previous item's or slot's reads of t are done
            stage_tile<N>(t, a.sxx + wo, a.sxy + wo, a.syy + wo, g.pitch, i0, j0, g.NX, g.NY);
            __syncthreads();
            vel_rows_with<N, R>(a, sl, blk, i, j, live, c, e, nt, flags, rip, rjp, s_red,
                                [&](float(&sxx_x)[R], float(&sxy_x)[R], float(&sxy_y)[R], float(&syy_y)[R]) {
                                    const float *hc = g.hc;
#pragma unroll
                                    for (int r = 0; r < R; r++) {
                                        const float *sx = &t.sxx[jr + r][tx + N];
                                        const float *sy = &t.sxy[jr + r + N][tx + N];
                                        const float *cy = &t.sxy[jr + r + N][tx + N];
                                        const float *cs = &t.syy[jr + r + N][tx];
                                        constexpr int Wd = VelTile<N>::W;
                                        sxx_x[r] = hc[1] * (sx[1] - sx[0]);
                                        sxy_x[r] = hc[1] * (sy[0] - sy[-1]);
                                        sxy_y[r] = hc[1] * (cy[0] - cy[-Wd]);
                                        syy_y[r] = hc[1] * (cs[kTileX] - cs[0]);
#pragma unroll
                                        for (int mm = 2; mm <= N; mm++) {
                                            sxx_x[r] = sxx_x[r] + hc[mm] * (sx[mm] - sx[1 - mm]);
                                            sxy_x[r] = sxy_x[r] + hc[mm] * (sy[mm - 1] - sy[-mm]);
                                            sxy_y[r] = sxy_y[r] + hc[mm] * (cy[(mm - 1) * Wd] - cy[-mm * Wd]);
                                            syy_y[r] = syy_y[r] + hc[mm] * (cs[mm * kTileX] - cs[(1 - mm) * kTileX]);
                                        }
                                    }
                                });
        }
    }
}

// ---------------------------------------------------------------------------
// per-cell material values of the stress step, loaded once per work item
template <int L>
struct StressMat {
    float fe, ge, fipjp;  // elastic
    ViscCell vc;          // viscoelastic
};

// stress step of one cell of slot s
template <int N, int L>
__device__ __forceinline__ void str_cell(const StepArgs &a, int s, int blk, int i, int j, bool live, bool top, long c,
                                         long e, int nt, int flags, const StressMat<L> &M, float (*s_syy)[kTileX],
                                         float (*s_sxy)[kTileX], float (*s_red)[kTileY])
{
    const StepGeom &g = a.g;
    const int tx = threadIdx.x, ty = threadIdx.y;
    const int P = g.pitch;
    const long wo = (long)s * a.ws, po = (long)s * a.pss;
    const auto vxs = gmem(a.vx) + wo, vys = gmem(a.vy) + wo;
    const bool snap_step = (flags & kSnapStep) != 0;
    const bool corr_step = (flags & kCorrStep) != 0;
    const bool rates = snap_step && a.VELOCITY == 1;
    float sxx = 0.0f, syy = 0.0f, sxy = 0.0f, ux = 0.0f, uy = 0.0f, uxy = 0.0f;
    float rr[L > 0 ? L : 1], pp[L > 0 ? L : 1], qq[L > 0 ? L : 1];
    if (live) {
        float vxx, vyx, vxy, vyy;
        const float scale = L ? (float)(1.0 / (double)g.DH) : g.DT / g.DH;
        velocity_derivs<N>(g.hc, a.vx + wo + c, a.vy + wo + c, P, scale, vxx, vyx, vxy, vyy);
        cpml_stress(g, j, i, a.psi_vxx + po, a.psi_vyx + po, a.psi_vyy + po, a.psi_vxy + po, vxx, vyx, vxy, vyy);
        sxx = gmem(a.sxx)[wo + c];
        syy = gmem(a.syy)[wo + c];
        sxy = gmem(a.sxy)[wo + c];
        if (L == 0) {
            if (rates) rates_elastic(M.fe, M.ge, M.fipjp, g.DT, vxx, vyx, vxy, vyy, ux, uy, uxy);
            stress_elastic(2.0f * M.fe, M.ge, M.fipjp, vxx, vyx, vxy, vyy, sxx, syy, sxy);
        } else {
#pragma unroll
            for (int l = 0; l < L; l++) {
                rr[l] = gmem(a.r)[wo + mv_index(c, l, 3 * L)];
                pp[l] = gmem(a.r)[wo + mv_index(c, L + l, 3 * L)];
                qq[l] = gmem(a.r)[wo + mv_index(c, 2 * L + l, 3 * L)];
            }
            ViscUpdate<(L > 0 ? L : 1)> vu;
            visc_update(M.vc, a.eta, vu);
            stress_visc(vu, a.bip, a.bjm, a.cip, a.cjm, g.DT / 2.0, g.DT, vxx, vyx, vxy, vyy, sxx, syy, sxy, rr, pp, qq, rates,
                        ux, uy, uxy);
        }
        // explosive sources of this cell, applied after the stress update
        // and before the free surface (src/IFOS2D.c:1758-1773)
        // the look-ups of points come last: a tile without any (nearly all) would
        // wait for their scalar loads before it issued its stencil loads (stress
        // step of 2000x800, L=2: 27.6 us with them first, 26.4 so)
        if (flags & kForward) {
            const int ex = first_point(a, a.exp, s, e, tile_has(a.exp, s, a.nbx * a.nby, blk) && cmem(a.explosive)[s]);
            for (int l = ex; l >= 0; l = gmem(a.exp.next)[l]) {
                const float amp = explosive_amp(a.exp.sig + (long)l * a.NT - 1, nt, a.NT, g.DH);
                sxx = add_half(sxx, amp);
                syy = add_half(syy, amp);
            }
        }
    }
    if (top) {
        // the free surface of column i reads the new syy of rows 2..N+1 and
        // sxy of rows 1..N; they come from the other threads of this tile
        s_syy[ty][tx] = live ? syy : 0.0f;
        s_sxy[ty][tx] = live ? sxy : 0.0f;
        __syncthreads();
        if (live && j == 1) {
            syy = 0.0f;
            if (rates) uy = 0.0f;
            if (L) {
#pragma unroll
                for (int l = 0; l < L; l++) qq[l] = 0.0f;
            }
#pragma unroll
            for (int m = 1; m <= N; m++) {
                gmem(a.syy)[wo + c - (long)m * P] = -s_syy[m][tx];
                gmem(a.sxy)[wo + c - (long)m * P] = -s_sxy[m - 1][tx];
            }
            float vxx, vyy;
            surface_derivs<N>(g, i, a.vx + wo + c, a.vy + wo + c, P, a.psi_vxxs + po, vxx, vyy);
            if (L == 0) {
                surface_elastic_update((float)((double)M.fe * 2.0), M.ge, g.DT, vxx, vyy, sxx, rates, ux);
            } else {
                surface_visc_update<(L > 0 ? L : 1)>(M.vc.mu, M.vc.pi, M.vc.taus, M.vc.taup, a.eta, g.DT, vxx, vyy,
                                                     sxx, pp, rates, ux);
            }
        }
        __syncthreads();  // the exchange rows are reused by the next slot
    }
    if (snap_step) {
        const float val[3] = {a.VELOCITY ? ux : sxx, a.VELOCITY ? uy : syy, a.VELOCITY ? uxy : sxy};
        snap_store<3>(a, s, 2, (nt - 1) / a.DTINV, e, blk, live, val, s_red);
    }
    if (!live) return;
    gmem(a.sxx)[wo + c] = sxx;
    gmem(a.syy)[wo + c] = syy;
    gmem(a.sxy)[wo + c] = sxy;
    if (g.BOUNDARY) wrap_pair<N>(g, gmem(a.sxx) + wo, gmem(a.sxy) + wo, c, i, sxx, sxy);
    if (L) {
#pragma unroll
        for (int l = 0; l < L; l++) {
            gmem(a.r)[wo + mv_index(c, l, 3 * L)] = rr[l];
            gmem(a.r)[wo + mv_index(c, L + l, 3 * L)] = pp[l];
            gmem(a.r)[wo + mv_index(c, 2 * L + l, 3 * L)] = qq[l];
        }
    }
    if (corr_step) {
        const long ks = (a.NT - nt) / a.DTINV, wco = (long)s * a.wcs;
        float wr = gmem(a.wc_rho)[wco + e], w = gmem(a.wc)[wco + e], wu = gmem(a.wc_u)[wco + e];
        correlate_cell(gmem(a.vxp1)[wo + c], gmem(a.vyp1)[wo + c], sxx, syy, sxy, snap_load(a, s, 0, ks, e, blk),
                       snap_load(a, s, 1, ks, e, blk), snap_load(a, s, 2, ks, e, blk),
                       snap_load(a, s, 3, ks, e, blk), snap_load(a, s, 4, ks, e, blk), gmem(a.muss)[e],
                       gmem(a.lamss)[e], gmem(a.vs_i)[e] > 0.0f, wr, w, wu);
        gmem(a.wc_rho)[wco + e] = wr;
        gmem(a.wc)[wco + e] = w;
        gmem(a.wc_u)[wco + e] = wu;
    }
    if (flags & kForward) {
        const int rc = first_point(a, a.rec, s, e, tile_has(a.rec, s, a.nbx * a.nby, blk));
        for (int t = rc; t >= 0; t = gmem(a.rec.next)[t]) {
            gmem(a.seis_vx)[(long)t * a.NT + nt - 1] = vxs[c];
            gmem(a.seis_vy)[(long)t * a.NT + nt - 1] = vys[c];
        }
    }
    if (a.nan_flag && j == g.NY / 2 && i == g.NX / 2) {
        const float v = vys[c];
        if (isnan(v) && *gmem(a.nan_flag) == 0) *gmem(a.nan_flag) = nt;
    }
}

template <int N, int L, int SPB, bool LEAN>
__global__ __launch_bounds__(512) void k_str_step(const StepArgs *__restrict__ pa, int k, int persistent, int flags_)
{
    const int flags = LEAN ? (flags_ & kForward) : flags_;  // as in k_vel_step
    const StepArgs &a = *pa;
    __shared__ float s_syy[kTileY][kTileX];
    __shared__ float s_sxy[kTileY][kTileX];
    __shared__ float s_red[3][kTileY];
    const StepGeom &g = a.g;
    const ItemMap m = item_map(a);
    const int nt = step_number(a, k);
    int first, end, stride;
    work_range(m, m.ntiles * m.ngroups, persistent != 0, first, end, stride);
    for (int it = first; it < end; it += stride) {
        int blk, s0;
        item_of(m, it, SPB, blk, s0);
        // uniform across the workgroup: keep them in scalar registers
        blk = __builtin_amdgcn_readfirstlane(blk);
        s0 = __builtin_amdgcn_readfirstlane(s0);
        const int by = (int)fdiv(blk, m.nbx_mul, m.nbx_sh), bx = blk - by * m.nbx;
        const int i = bx * kTileX + threadIdx.x + 1;
        const int j = by * kTileY + threadIdx.y + 1;
        const bool live = i <= g.NX && j <= g.NY;
        const bool top = by == 0 && g.FREE_SURF;
        const long c = (long)j * g.pitch + i;
        const long e = (long)(j - 1) * g.NX + (i - 1);
        StressMat<L> M;
        M.fe = M.ge = M.fipjp = 0.0f;
        M.vc = ViscCell{};
        if (live) {
            if (L == 0) {
                M.fe = gmem(a.f)[c];
                M.ge = gmem(a.gl)[c];
                M.fipjp = gmem(a.uipjp)[c];
            } else {
                visc_coeffs(L, g.DT, gmem(a.mu)[c], gmem(a.pi)[c], gmem(a.muipjp)[c], gmem(a.taus)[c], gmem(a.taup)[c], gmem(a.tausipjp)[c], M.vc);
            }
        }
#pragma unroll
        for (int u = 0; u < SPB; u++)
            if (s0 + u < m.nslots)
                str_cell<N, L>(a, s0 + u, blk, i, j, live, top, c, e, nt, flags, M, s_syy, s_sxy, s_red);
    }
}

// ---------------------------------------------------------------------------
// One time step in one kernel.  A workgroup owns a 64x8 tile.  It first
// stages the old stresses it needs in LDS, computes the new velocities of the
// tile and of an N-cell rim around it (the rim's values are what the
// neighbouring tiles compute for their own cells, from the same inputs and
// the same arithmetic, so they are the same bits), then updates the tile's
// stresses from those velocities.  Wavefields and the velocity-side CPML
// memory are read from one buffer and written to the other (the buffers swap
// every step), because a tile reads its neighbours' old values while they
// write their new ones.  Per cell and step this moves one read and one write
// of vx, vy, sxx, syy, sxy instead of the two kernels' two reads of the
// stresses and of the velocities.
template <int N>
struct FusedLds {
    static constexpr int VX = kTileX + 2 * N, VY = kTileY + 2 * N;  // velocity region
    static constexpr int AX = kTileX + 4 * N - 1, SY = kTileY + 4 * N - 1;
    float sxx[VY][AX];   // rows j0+1-N .., columns i0+2-2N ..
    float syy[SY][VX];   // rows j0+2-2N .., columns i0+1-N ..
    float sxy[SY][AX];   // rows j0+1-2N .., columns i0+1-2N ..
    float vx[VY][VX];    // new velocities, rows j0+1-N .., columns i0+1-N ..
    float vy[VY][VX];
    float acc[2][kTileY][kTileX];  // accelerations of the tile's cells (forward snapshot steps)
};

// velocity-side CPML (the arithmetic of cpml_velocity) reading the memory of
// the previous step from the *_r arrays and, when `own`, writing the new
// memory to the *_w arrays
__device__ __forceinline__ void cpml_velocity_rw(const StepGeom &g, int j, int i, bool own, const float *rxx,
                                                 const float *rxy, const float *ryy, const float *ryx, float *wxx,
                                                 float *wxy, float *wyy, float *wyx, float &sxx_x, float &sxy_x,
                                                 float &sxy_y, float &syy_y)
{
    const Cpml &pm = g.pml;
    auto side_x = [&](int h) {
        const long o = (long)(j - 1) * g.px + h;
        const float p1 = cmem(pm.b_xh)[h] * gmem(rxx)[o] + cmem(pm.a_xh)[h] * sxx_x;
        sxx_x = divK(sxx_x, pm.K_xh, h, g.K_one) + p1;
        const float p2 = cmem(pm.b_x)[h] * gmem(rxy)[o] + cmem(pm.a_x)[h] * sxy_x;
        sxy_x = divK(sxy_x, pm.K_x, h, g.K_one) + p2;
        if (own) {
            gmem(wxx)[o] = p1;
            gmem(wxy)[o] = p2;
        }
    };
    auto side_y = [&](int h) {
        const long o = (long)h * g.py + (i - 1);
        const float p1 = cmem(pm.b_yh)[h] * gmem(ryy)[o] + cmem(pm.a_yh)[h] * syy_y;
        syy_y = divK(syy_y, pm.K_yh, h, g.K_one) + p1;
        const float p2 = cmem(pm.b_y)[h] * gmem(ryx)[o] + cmem(pm.a_y)[h] * sxy_y;
        sxy_y = divK(sxy_y, pm.K_y, h, g.K_one) + p2;
        if (own) {
            gmem(wyy)[o] = p1;
            gmem(wyx)[o] = p2;
        }
    };
    if (!g.BOUNDARY && i <= g.FW) side_x(i - 1);
    if (!g.BOUNDARY && i >= g.NX - g.FW + 1) side_x(i - g.NX + 2 * g.FW - 1);
    if (!g.FREE_SURF && j <= g.FW) side_y(j - 1);
    if (j >= g.NY - g.FW + 1) side_y(j - g.NY + 2 * g.FW - 1);
}

template <int N, int L>
__global__ __launch_bounds__(512) void k_fused_step(const StepArgs *__restrict__ pa, int k, int persistent,
                                                     int flags)
{
    using T = FusedLds<N>;
    constexpr int VX = T::VX, VY = T::VY, AX = T::AX, SY = T::SY;
    const StepArgs &a = *pa;
    __shared__ T st;
    __shared__ float s_syy[kTileY][kTileX];
    __shared__ float s_sxy[kTileY][kTileX];
    __shared__ float s_red[3][kTileY];
    const StepGeom &g = a.g;
    const ItemMap m = item_map(a);
    const int nt = step_number(a, k);
    const int tid = threadIdx.y * kTileX + threadIdx.x, tx = threadIdx.x, ty = threadIdx.y;
    const int P = g.pitch, NX = g.NX, NY = g.NY, H = N + 1;
    // buffers: step nt reads set (nt - 1) & 1 and writes set nt & 1
    const bool odd = (nt & 1) != 0;
    const float *rvx = odd ? a.vx : a.vx2, *rvy = odd ? a.vy : a.vy2;
    const float *rsxx = odd ? a.sxx : a.sxx2, *rsyy = odd ? a.syy : a.syy2, *rsxy = odd ? a.sxy : a.sxy2;
    float *wvx = odd ? a.vx2 : a.vx, *wvy = odd ? a.vy2 : a.vy;
    float *wsxx = odd ? a.sxx2 : a.sxx, *wsyy = odd ? a.syy2 : a.syy, *wsxy = odd ? a.sxy2 : a.sxy;
    const float *rp_xx = odd ? a.psi_sxx_x : a.psi2_sxx_x, *rp_xy = odd ? a.psi_sxy_x : a.psi2_sxy_x;
    const float *rp_yy = odd ? a.psi_syy_y : a.psi2_syy_y, *rp_yx = odd ? a.psi_sxy_y : a.psi2_sxy_y;
    float *wp_xx = odd ? a.psi2_sxx_x : a.psi_sxx_x, *wp_xy = odd ? a.psi2_sxy_x : a.psi_sxy_x;
    float *wp_yy = odd ? a.psi2_syy_y : a.psi_syy_y, *wp_yx = odd ? a.psi2_sxy_y : a.psi_sxy_y;
    const bool snap_step = (flags & kSnapStep) != 0, corr_step = (flags & kCorrStep) != 0;
    const bool fwd = (flags & kForward) != 0;
    const bool rates = snap_step && a.VELOCITY == 1;
    int first, end, stride;
    work_range(m, m.ntiles * m.ngroups, persistent != 0, first, end, stride);
    for (int it = first; it < end; it += stride) {
        int blk, s;
        item_of(m, it, 1, blk, s);
        blk = __builtin_amdgcn_readfirstlane(blk);
        s = __builtin_amdgcn_readfirstlane(s);
        const int by = (int)fdiv(blk, m.nbx_mul, m.nbx_sh), bx = blk - by * m.nbx;
        const int i0 = bx * kTileX, j0 = by * kTileY;
        const long wo = (long)s * a.ws, po = (long)s * a.pss;
        // ---- stage the old stresses (zero outside the padded grid, where
        // they only feed velocities of cells outside the model)
        auto stage = [&](const float *src, float *dst, int rows, int cols, int jr, int ic) {
            const auto sg = gmem(src) + wo;
            for (int q = tid; q < rows * cols; q += kTileX * kTileY) {
                const int r = q / cols, cc = q - r * cols;
                const int gj = jr + r, gi = ic + cc;
                const bool in = gj >= 1 - H && gj <= NY + H && gi >= -15 && gi <= P - 16;
                dst[q] = in ? sg[(long)gj * P + gi] : 0.0f;
            }
        };
        __syncthreads();  // the previous item's readers are done with the LDS
        stage(rsxx, &st.sxx[0][0], VY, AX, j0 + 1 - N, i0 + 2 - 2 * N);
        stage(rsyy, &st.syy[0][0], SY, VX, j0 + 2 - 2 * N, i0 + 1 - N);
        stage(rsxy, &st.sxy[0][0], SY, AX, j0 + 1 - 2 * N, i0 + 1 - 2 * N);
        __syncthreads();
        // ---- velocities of the tile and its rim
        for (int q = tid; q < VX * VY; q += kTileX * kTileY) {
            const int ry = q / VX, rx = q - ry * VX;
            const int gj = j0 + 1 - N + ry, gi = i0 + 1 - N + rx;
            float vx = 0.0f, vy = 0.0f;
            if (gj >= 1 && gj <= NY && gi >= 1 && gi <= NX) {
                const bool own = rx >= N && rx < N + kTileX && ry >= N && ry < N + kTileY;
                const float *X = &st.sxx[ry][rx + N - 1];
                const float *Y = &st.syy[ry + N - 1][rx];
                const float *S = &st.sxy[ry + N][rx + N];
                float sxx_x = g.hc[1] * (X[1] - X[0]);
                float sxy_x = g.hc[1] * (S[0] - S[-1]);
                float sxy_y = g.hc[1] * (S[0] - S[-AX]);
                float syy_y = g.hc[1] * (Y[VX] - Y[0]);
#pragma unroll
                for (int mm = 2; mm <= N; mm++) {
                    sxx_x = sxx_x + g.hc[mm] * (X[mm] - X[1 - mm]);
                    sxy_x = sxy_x + g.hc[mm] * (S[mm - 1] - S[-mm]);
                    sxy_y = sxy_y + g.hc[mm] * (S[(mm - 1) * AX] - S[-mm * AX]);
                    syy_y = syy_y + g.hc[mm] * (Y[mm * VX] - Y[(1 - mm) * VX]);
                }
                cpml_velocity_rw(g, gj, gi, own, rp_xx + po, rp_xy + po, rp_yy + po, rp_yx + po, wp_xx + po,
                                 wp_xy + po, wp_yy + po, wp_yx + po, sxx_x, sxy_x, sxy_y, syy_y);
                const long c = (long)gj * P + gi;
                const float vx0 = gmem(rvx)[wo + c], vy0 = gmem(rvy)[wo + c];
                const float rip = gmem(a.rip)[c], rjp = gmem(a.rjp)[c];
                if (own) {
                    if (fwd) {
                        if (snap_step) {
                            st.acc[0][ry - N][rx - N] = vel_rate(rip, sxx_x + sxy_y, g.DH);
                            st.acc[1][ry - N][rx - N] = vel_rate(rjp, sxy_x + syy_y, g.DH);
                        }
                    } else if (flags & kAdjInt) {
                        gmem(a.vxp1)[wo + c] += vx0 * g.DT;
                        gmem(a.vyp1)[wo + c] += vy0 * g.DT;
                    } else if (corr_step) {
                        gmem(a.vxp1)[wo + c] = vx0;
                        gmem(a.vyp1)[wo + c] = vy0;
                    }
                }
                vx = vel_new(vx0, g.DT, rip, sxx_x + sxy_y, g.DH);
                vy = vel_new(vy0, g.DT, rjp, sxy_x + syy_y, g.DH);
                // point forces / residual injection at this cell, in order
                for (int l = first_point(a, a.inj, s, (long)(gj - 1) * NX + (gi - 1), true); l >= 0;
                     l = gmem(a.inj.next)[l])
                    inject(a, l, nt, rip, rjp, vx, vy);
                if (own) {
                    gmem(wvx)[wo + c] = vx;
                    gmem(wvy)[wo + c] = vy;
                }
            }
            st.vx[ry][rx] = vx;
            st.vy[ry][rx] = vy;
        }
        __syncthreads();
        // ---- the tile's cells: one per thread
        const int i = i0 + 1 + tx, j = j0 + 1 + ty;
        const bool live = i <= NX && j <= NY;
        const bool top = by == 0 && g.FREE_SURF;
        const long c = (long)j * P + i, e = (long)(j - 1) * NX + (i - 1);
        const float nvx = st.vx[ty + N][tx + N], nvy = st.vy[ty + N][tx + N];
        if (fwd && snap_step) {
            const float val[2] = {st.acc[0][ty][tx], st.acc[1][ty][tx]};
            snap_store<2>(a, s, 0, (nt - 1) / a.DTINV, e, blk, live, val, s_red);
        }
        if ((flags & kEnergy) && live) {
            if (a.wacc64) {
                const auto W = gmem(a.wacc64) + (long)s * a.wacs;
                W[e] += ((double)nvx * (double)nvx) + ((double)nvy * (double)nvy);
            } else {
                const auto W = gmem(a.wacc) + (long)s * a.wacs;
                W[e] += ((nvx * nvx) + (nvy * nvy));
            }
        }
        int ex = -1, rc = -1;
        if (fwd && live) {
            ex = first_point(a, a.exp, s, e, cmem(a.explosive)[s] && tile_has(a.exp, s, m.ntiles, blk));
            rc = first_point(a, a.rec, s, e, tile_has(a.rec, s, m.ntiles, blk));
        }
        float sxx = 0.0f, syy = 0.0f, sxy = 0.0f, ux = 0.0f, uy = 0.0f, uxy = 0.0f;
        float rr[L > 0 ? L : 1], pp[L > 0 ? L : 1], qq[L > 0 ? L : 1];
        StressMat<L> M;
        M.fe = M.ge = M.fipjp = 0.0f;
        M.vc = ViscCell{};
        const float *V = &st.vx[ty + N][tx + N], *Wv = &st.vy[ty + N][tx + N];
        if (live) {
            if (L == 0) {
                M.fe = gmem(a.f)[c];
                M.ge = gmem(a.gl)[c];
                M.fipjp = gmem(a.uipjp)[c];
            } else {
                visc_coeffs(L, g.DT, gmem(a.mu)[c], gmem(a.pi)[c], gmem(a.muipjp)[c], gmem(a.taus)[c],
                            gmem(a.taup)[c], gmem(a.tausipjp)[c], M.vc);
            }
            const float scale = L ? (float)(1.0 / (double)g.DH) : g.DT / g.DH;
            float vxx = g.hc[1] * (V[0] - V[-1]);
            float vyx = g.hc[1] * (Wv[1] - Wv[0]);
            float vxy = g.hc[1] * (V[VX] - V[0]);
            float vyy = g.hc[1] * (Wv[0] - Wv[-VX]);
#pragma unroll
            for (int mm = 2; mm <= N; mm++) {
                vxx = vxx + g.hc[mm] * (V[mm - 1] - V[-mm]);
                vyx = vyx + g.hc[mm] * (Wv[mm] - Wv[1 - mm]);
                vxy = vxy + g.hc[mm] * (V[mm * VX] - V[(1 - mm) * VX]);
                vyy = vyy + g.hc[mm] * (Wv[(mm - 1) * VX] - Wv[-mm * VX]);
            }
            vxx = vxx * scale;
            vyx = vyx * scale;
            vxy = vxy * scale;
            vyy = vyy * scale;
            cpml_stress(g, j, i, a.psi_vxx + po, a.psi_vyx + po, a.psi_vyy + po, a.psi_vxy + po, vxx, vyx, vxy, vyy);
            sxx = st.sxx[ty + N][tx + 2 * N - 1];
            syy = st.syy[ty + 2 * N - 1][tx + N];
            sxy = st.sxy[ty + 2 * N][tx + 2 * N];
            if (L == 0) {
                if (rates) rates_elastic(M.fe, M.ge, M.fipjp, g.DT, vxx, vyx, vxy, vyy, ux, uy, uxy);
                stress_elastic(2.0f * M.fe, M.ge, M.fipjp, vxx, vyx, vxy, vyy, sxx, syy, sxy);
            } else {
#pragma unroll
                for (int l = 0; l < L; l++) {
                    rr[l] = gmem(a.r)[wo + mv_index(c, l, 3 * L)];
                    pp[l] = gmem(a.r)[wo + mv_index(c, L + l, 3 * L)];
                    qq[l] = gmem(a.r)[wo + mv_index(c, 2 * L + l, 3 * L)];
                }
                ViscUpdate<(L > 0 ? L : 1)> vu;
                visc_update(M.vc, a.eta, vu);
                stress_visc(vu, a.bip, a.bjm, a.cip, a.cjm, g.DT / 2.0, g.DT, vxx, vyx, vxy, vyy, sxx, syy, sxy, rr, pp, qq,
                            rates, ux, uy, uxy);
            }
            for (int l = ex; l >= 0; l = gmem(a.exp.next)[l]) {
                const float amp = explosive_amp(a.exp.sig + (long)l * a.NT - 1, nt, a.NT, g.DH);
                sxx = add_half(sxx, amp);
                syy = add_half(syy, amp);
            }
        }
        if (top) {
            s_syy[ty][tx] = live ? syy : 0.0f;
            s_sxy[ty][tx] = live ? sxy : 0.0f;
            __syncthreads();
            if (live && j == 1) {
                syy = 0.0f;
                if (rates) uy = 0.0f;
                if (L) {
#pragma unroll
                    for (int l = 0; l < L; l++) qq[l] = 0.0f;
                }
#pragma unroll
                for (int mm = 1; mm <= N; mm++) {
                    gmem(wsyy)[wo + c - (long)mm * P] = -s_syy[mm][tx];
                    gmem(wsxy)[wo + c - (long)mm * P] = -s_sxy[mm - 1][tx];
                }
                // surface_derivs on the new velocities of row 1 (from LDS)
                float vxx = 0.0f, vyy = 0.0f;
#pragma unroll
                for (int mm = 1; mm <= N; mm++) {
                    vxx += g.hc[mm] * (V[mm - 1] - V[-mm]);
                    vyy += g.hc[mm] * (Wv[(mm - 1) * VX] - Wv[-mm * VX]);
                }
                const float dh24 = 1.0 / (double)g.DH;
                vxx *= dh24;
                vyy *= dh24;
                const Cpml &pm = g.pml;
                auto surf = [&](int h) {
                    auto ps = gmem(a.psi_vxxs + po) + h;
                    *ps = cmem(pm.b_x)[h] * *ps + cmem(pm.a_x)[h] * vxx;
                    vxx = divK(vxx, pm.K_x, h, g.K_one) + *ps;
                };
                if (!g.BOUNDARY && i <= g.FW) surf(i - 1);
                if (!g.BOUNDARY && i >= g.NX - g.FW + 1) surf(i - g.NX + 2 * g.FW - 1);
                if (L == 0) {
                    surface_elastic_update((float)((double)M.fe * 2.0), M.ge, g.DT, vxx, vyy, sxx, rates, ux);
                } else {
                    surface_visc_update<(L > 0 ? L : 1)>(M.vc.mu, M.vc.pi, M.vc.taus, M.vc.taup, a.eta, g.DT, vxx,
                                                         vyy, sxx, pp, rates, ux);
                }
            }
        }
        if (snap_step) {
            const float val[3] = {a.VELOCITY ? ux : sxx, a.VELOCITY ? uy : syy, a.VELOCITY ? uxy : sxy};
            snap_store<3>(a, s, 2, (nt - 1) / a.DTINV, e, blk, live, val, s_red);
        }
        if (!live) continue;
        gmem(wsxx)[wo + c] = sxx;
        gmem(wsyy)[wo + c] = syy;
        gmem(wsxy)[wo + c] = sxy;
        if (L) {
#pragma unroll
            for (int l = 0; l < L; l++) {
                gmem(a.r)[wo + mv_index(c, l, 3 * L)] = rr[l];
                gmem(a.r)[wo + mv_index(c, L + l, 3 * L)] = pp[l];
                gmem(a.r)[wo + mv_index(c, 2 * L + l, 3 * L)] = qq[l];
            }
        }
        if (corr_step) {
            const long ks = (a.NT - nt) / a.DTINV, wco = (long)s * a.wcs;
            float wr = gmem(a.wc_rho)[wco + e], w = gmem(a.wc)[wco + e], wu = gmem(a.wc_u)[wco + e];
            correlate_cell(gmem(a.vxp1)[wo + c], gmem(a.vyp1)[wo + c], sxx, syy, sxy,
                           snap_load(a, s, 0, ks, e, blk), snap_load(a, s, 1, ks, e, blk),
                           snap_load(a, s, 2, ks, e, blk), snap_load(a, s, 3, ks, e, blk),
                           snap_load(a, s, 4, ks, e, blk), gmem(a.muss)[e], gmem(a.lamss)[e],
                           gmem(a.vs_i)[e] > 0.0f, wr, w, wu);
            gmem(a.wc_rho)[wco + e] = wr;
            gmem(a.wc)[wco + e] = w;
            gmem(a.wc_u)[wco + e] = wu;
        }
        for (int t = rc; t >= 0; t = gmem(a.rec.next)[t]) {
            gmem(a.seis_vx)[(long)t * a.NT + nt - 1] = nvx;
            gmem(a.seis_vy)[(long)t * a.NT + nt - 1] = nvy;
        }
        if (a.nan_flag && j == NY / 2 && i == NX / 2) {
            if (isnan(nvy) && *gmem(a.nan_flag) == 0) *gmem(a.nan_flag) = nt;
        }
    }
}

// ---------------------------------------------------------------------------
static int grid_of(const StepArgs &a, const LaunchShape &ls, int grid)
{
    const int nitems = a.nbx * a.nby * ((a.nslots + ls.spb - 1) / ls.spb);
    if (grid > 0) return std::min(grid, (nitems + 7) / 8 * 8);
    if (!a.swizzle) return nitems;
    int widest = 0;  // one workgroup per item of the largest XCD run
    for (int x = 0; x < 8; x++) widest = std::max(widest, a.xlo[x + 1] - a.xlo[x]);
    return 8 * widest;
}

template <int N, int SPB, bool LEAN>
static void vel_launch_rows(const StepArgs &a, const StepArgs *da, const LaunchShape &ls, int k, int flags, int gr,
                            hipStream_t s)
{
    const int pers = ls.grid_v > 0 ? 1 : 0;
    if (ls.rows_v == 4)
        hipLaunchKernelGGL((k_vel_step<N, SPB, 4, LEAN>), dim3(gr), dim3(kTileX, kTileY / 4), 0, s, da, k, pers,
                           flags);
    else if (ls.rows_v == 2)
        hipLaunchKernelGGL((k_vel_step<N, SPB, 2, LEAN>), dim3(gr), dim3(kTileX, kTileY / 2), 0, s, da, k, pers,
                           flags);
    else
        hipLaunchKernelGGL((k_vel_step<N, SPB, 1, LEAN>), dim3(gr), dim3(kTileX, kTileY), 0, s, da, k, pers, flags);
}

template <int N, int SPB>
static void vel_launch(const StepArgs &a, const StepArgs *da, const LaunchShape &ls, int k, hipStream_t s)
{
    const int gr = grid_of(a, ls, ls.grid_v);
    const int flags = step_flags(a, k);
    if (ls.lds_v)
        hipLaunchKernelGGL((k_vel_step_lds<N, SPB>), dim3(gr), dim3(kTileX, kTileY / 2), 0, s, da, k,
                           ls.grid_v > 0 ? 1 : 0, flags);
    else if (lean_step(flags))
        vel_launch_rows<N, SPB, true>(a, da, ls, k, flags, gr, s);
    else
        vel_launch_rows<N, SPB, false>(a, da, ls, k, flags, gr, s);
}

template <int N>
void vel_n(const StepArgs &a, const StepArgs *da, const LaunchShape &ls, int k, hipStream_t s)
{
    switch (ls.spb) {
    case 1: vel_launch<N, 1>(a, da, ls, k, s); break;
    case 2: vel_launch<N, 2>(a, da, ls, k, s); break;
    case 4: vel_launch<N, 4>(a, da, ls, k, s); break;
    default: break;
    }
}

template <int N, int L, int SPB>
static void str_launch(const StepArgs &a, const StepArgs *da, const LaunchShape &ls, int k, hipStream_t s)
{
    const int gr = grid_of(a, ls, ls.grid);
    const int flags = step_flags(a, k);
    if (lean_step(flags))
        hipLaunchKernelGGL((k_str_step<N, L, SPB, true>), dim3(gr), dim3(kTileX, kTileY), 0, s, da, k,
                           ls.grid > 0 ? 1 : 0, flags);
    else
        hipLaunchKernelGGL((k_str_step<N, L, SPB, false>), dim3(gr), dim3(kTileX, kTileY), 0, s, da, k,
                           ls.grid > 0 ? 1 : 0, flags);
}

template <int N, int L>
static void str_nl(const StepArgs &a, const StepArgs *da, const LaunchShape &ls, int k, hipStream_t s)
{
    switch (ls.spb) {
    case 1: str_launch<N, L, 1>(a, da, ls, k, s); break;
    case 2: str_launch<N, L, 2>(a, da, ls, k, s); break;
    case 4: str_launch<N, L, 4>(a, da, ls, k, s); break;
    default: break;
    }
}

template <int N>
void str_n(const StepArgs &a, const StepArgs *da, const LaunchShape &ls, int k, hipStream_t s)
{
    switch (a.L) {
    case 0: str_nl<N, 0>(a, da, ls, k, s); break;
    case 1: str_nl<N, 1>(a, da, ls, k, s); break;
    case 2: str_nl<N, 2>(a, da, ls, k, s); break;
    case 3: str_nl<N, 3>(a, da, ls, k, s); break;
    case 4: str_nl<N, 4>(a, da, ls, k, s); break;
    case 5: str_nl<N, 5>(a, da, ls, k, s); break;
    default: break;
    }
}

template <int N, int L>
static void fused_launch(const StepArgs &a, const StepArgs *da, const LaunchShape &ls, int k, hipStream_t s)
{
    const int gr = grid_of(a, ls, ls.grid);
    hipLaunchKernelGGL((k_fused_step<N, L>), dim3(gr), dim3(kTileX, kTileY), 0, s, da, k, ls.grid > 0 ? 1 : 0,
                       step_flags(a, k));
}

template <int N>
void fused_n(const StepArgs &a, const StepArgs *da, const LaunchShape &ls, int k, hipStream_t s)
{
    switch (a.L) {
    case 0: fused_launch<N, 0>(a, da, ls, k, s); break;
    case 1: fused_launch<N, 1>(a, da, ls, k, s); break;
    case 2: fused_launch<N, 2>(a, da, ls, k, s); break;
    case 3: fused_launch<N, 3>(a, da, ls, k, s); break;
    case 4: fused_launch<N, 4>(a, da, ls, k, s); break;
    case 5: fused_launch<N, 5>(a, da, ls, k, s); break;
    default: break;
    }
}

}  // namespace ifos
