// ifos_step.hip -- launch entry points of the fused time-step kernels
// (ifos_step_kernels.h), whose instantiations for each stencil order sit in
// ifos_order1.hip .. ifos_order6.hip.
#include <algorithm>
#include <vector>

#include "ifos_resident.h"
#include "ifos_step.h"

namespace ifos {

template <int N>
void vel_n(const StepArgs &a, const StepArgs *da, const LaunchShape &ls, int k, hipStream_t s);
template <int N>
void str_n(const StepArgs &a, const StepArgs *da, const LaunchShape &ls, int k, hipStream_t s);
template <int N>
void fused_n(const StepArgs &a, const StepArgs *da, const LaunchShape &ls, int k, hipStream_t s);
template <int N>
size_t resident_lds(int L, int rows);
template <int N>
hipError_t resident_n(int L, const ResidentArgs &r, const ResidentPlan &p, hipStream_t s);

__global__ void k_tick(int *base, int by)
{
    if (threadIdx.x == 0 && blockIdx.x == 0) *base += by;
}

// ---------------------------------------------------------------------------
// multiplier and shift of fdiv for divisor d >= 1 (the round-up method for
// unsigned division by an invariant: l = ceil(log2 d),
// mul = floor(2^32 (2^l - d) / d) + 1, shift l - 1)
static void make_div(uint32_t d, uint32_t &mul, uint32_t &sh)
{
    if (d <= 1) {
        mul = 0;
        sh = 0;
        return;
    }
    uint32_t l = 0;
    while ((1ull << l) < d) l++;
    mul = (uint32_t)((((1ull << 32) * ((1ull << l) - d)) / d) + 1);
    sh = l - 1;
}

// the launcher's copy of the argument block with the per-shape fields set
StepArgs shaped_args(const StepArgs &a0, const LaunchShape &ls)
{
    StepArgs a = a0;
    a.ngroups = (a.nslots + ls.spb - 1) / ls.spb;
    a.slot_major = ls.order ? 1 : 0;
    make_div((uint32_t)a.nbx, a.nbx_mul, a.nbx_sh);
    make_div((uint32_t)a.ngroups, a.ng_mul, a.ng_sh);
    make_div((uint32_t)(a.nbx * a.nby), a.nt_mul, a.nt_sh);
    // XCD runs of equal estimated cost: a tile in an absorbing strip costs
    // 1 + cpml_weight (its cells update the CPML memory and divide by K);
    // the tiles of the bottom strip would otherwise all fall to the last XCD
    const StepGeom &g = a.g;
    const int ntiles = a.nbx * a.nby, nitems = ntiles * a.ngroups;
    auto in_cpml = [&](int blk) {
        const int by = blk / a.nbx, bx = blk - by * a.nbx;
        const int i0 = bx * kTileX + 1, i1 = i0 + kTileX - 1, j0 = by * kTileY + 1, j1 = j0 + kTileY - 1;
        return (!g.BOUNDARY && (i0 <= g.FW || i1 >= g.NX - g.FW + 1)) || (!g.FREE_SURF && j0 <= g.FW) ||
               j1 >= g.NY - g.FW + 1;
    };
    std::vector<double> cum(nitems + 1, 0.0);
    for (int it = 0; it < nitems; it++) {
        const int blk = a.slot_major ? it % ntiles : it / a.ngroups;
        cum[it + 1] = cum[it] + 1.0 + (in_cpml(blk) ? (double)ls.cpml_weight : 0.0);
    }
    a.xlo[0] = 0;
    for (int x = 1; x < 8; x++) {
        const double target = cum[nitems] * x / 8.0;
        a.xlo[x] = (int)(std::lower_bound(cum.begin(), cum.end(), target) - cum.begin());
        a.xlo[x] = std::max(a.xlo[x], a.xlo[x - 1]);
    }
    a.xlo[8] = nitems;
    return a;
}

void launch_vel_step(const StepArgs &a, const StepArgs *da, const LaunchShape &ls, int k, hipStream_t s)
{
    switch (a.g.N) {
    case 1: vel_n<1>(a, da, ls, k, s); break;
    case 2: vel_n<2>(a, da, ls, k, s); break;
    case 3: vel_n<3>(a, da, ls, k, s); break;
    case 4: vel_n<4>(a, da, ls, k, s); break;
    case 5: vel_n<5>(a, da, ls, k, s); break;
    case 6: vel_n<6>(a, da, ls, k, s); break;
    default: break;
    }
}

void launch_str_step(const StepArgs &a, const StepArgs *da, const LaunchShape &ls, int k, hipStream_t s)
{
    switch (a.g.N) {
    case 1: str_n<1>(a, da, ls, k, s); break;
    case 2: str_n<2>(a, da, ls, k, s); break;
    case 3: str_n<3>(a, da, ls, k, s); break;
    case 4: str_n<4>(a, da, ls, k, s); break;
    case 5: str_n<5>(a, da, ls, k, s); break;
    case 6: str_n<6>(a, da, ls, k, s); break;
    default: break;
    }
}

void launch_fused_step(const StepArgs &a, const StepArgs *da, const LaunchShape &ls, int k, hipStream_t s)
{
    switch (a.g.N) {
    case 1: fused_n<1>(a, da, ls, k, s); break;
    case 2: fused_n<2>(a, da, ls, k, s); break;
    case 3: fused_n<3>(a, da, ls, k, s); break;
    case 4: fused_n<4>(a, da, ls, k, s); break;
    case 5: fused_n<5>(a, da, ls, k, s); break;
    case 6: fused_n<6>(a, da, ls, k, s); break;
    default: break;
    }
}

static size_t lds_of(int N, int L, int rows)
{
    switch (N) {
    case 1: return resident_lds<1>(L, rows);
    case 2: return resident_lds<2>(L, rows);
    case 3: return resident_lds<3>(L, rows);
    case 4: return resident_lds<4>(L, rows);
    case 5: return resident_lds<5>(L, rows);
    default: return resident_lds<6>(L, rows);
    }
}

// One workgroup per compute unit at most, all of them resident at once.  The
// tile is as low as that allows (the steps of a small grid cost latency, not
// throughput: more workgroups, less work in each), at least as high as the
// stencil reaches, and on the free surface as the rows mirrored above it.
ResidentPlan resident_plan(const StepGeom &g, int L, int nslots, int snap_prec, int ncu, size_t lds_max)
{
    ResidentPlan p;
    const int most = resident_max_rows(g.N, L), nbx = (g.NX + kTileX - 1) / kTileX;
    // periodic sides wrap the halo, which may span two tiles there
    if (g.BOUNDARY || most == 0 || nslots < 1 || (long)nbx * nslots > ncu) return p;
    const int across = ncu / (nbx * nslots);  // tile rows per slot that fit
    int th = std::max((g.NY + across - 1) / across, g.N + (g.FREE_SURF ? 1 : 0));
    const int line = 2 * (2 * g.N - 1);
    while (line * (kTileX + th) > kWordsPerThread * kTileX * th) th++;
    for (int rows = 1; rows <= most; rows++) {
        int ty = (th + rows - 1) / rows;
        // the scales of 16-bit snapshots belong to 64x8 tiles, which are formed whole
        while (snap_prec && ty * rows % kTileY) ty++;
        if (ty > kResidentThreads / kTileX) continue;
        p.ty = ty;
        p.cells = th;
        p.th = ty * rows;
        p.tiles_y = (g.NY + p.th - 1) / p.th;
        p.nwg = nbx * p.tiles_y * nslots;
        p.words = (2 * g.N - 1) * 2 * (kTileX + p.th);
        p.lds = lds_of(g.N, L, rows);
        if (p.lds + 64 <= lds_max && resident_pays(g.N, L, rows, th)) p.rows = rows;
        return p;
    }
    return p;
}

hipError_t launch_resident(const StepArgs &a, ResidentArgs r, const ResidentPlan &p, hipStream_t s)
{
    r.words = p.words;
    r.th = p.th;
    r.ty = p.ty;
    r.tiles_y = p.tiles_y;
    r.ntile = a.nbx * p.tiles_y;
    r.nwg = p.nwg;
    r.per = (p.nwg + 7) / 8;
    switch (a.g.N) {
    case 1: return resident_n<1>(a.L, r, p, s);
    case 2: return resident_n<2>(a.L, r, p, s);
    case 3: return resident_n<3>(a.L, r, p, s);
    case 4: return resident_n<4>(a.L, r, p, s);
    case 5: return resident_n<5>(a.L, r, p, s);
    case 6: return resident_n<6>(a.L, r, p, s);
    default: return hipErrorInvalidValue;
    }
}

void launch_tick(int *base, int by, hipStream_t s) { hipLaunchKernelGGL(k_tick, dim3(1), dim3(1), 0, s, base, by); }

}  // namespace ifos
