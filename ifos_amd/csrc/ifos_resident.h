// ifos_resident.h -- the time loop as one launch (k_resident): argument block
// and plan.
//
// Each workgroup owns a tile of 64 columns x th rows for the whole run.  The
// wavefields of the tile and the halo its stencils read sit in LDS, the
// memory variables and materials in registers.  After each half step a
// workgroup hands the N edge lines its neighbours read to their inboxes in
// device memory and waits for theirs; nothing else synchronises the tiles.
//
// What bounds it: on small grids the latency of the two exchanges per step
// (about 2 us each: a write-through store, then the neighbour's polling load),
// on larger ones the arithmetic of the tile.  The per-step kernels pay two
// launches a step, each with its ramp, drain and cold loads.  Time per step,
// per-step kernels and this, FDORDER 8, L=2 (us): 1024x128 11.0 / 6.8,
// 1024x256 13.2 / 8.1, 1024x512 20.0 / 13.8; elastic FDORDER 4: 1024x128
// 9.4 / 5.5, 1024x768 17.5 / 11.4.
#pragma once
#include "ifos_step.h"

namespace ifos {

constexpr int kResidentThreads = 1024;  // largest workgroup: 64 columns x 16 rows of threads

// Rows of cells per thread the kernel is compiled for, by the number of
// relaxation mechanisms (0: not compiled).  1024 threads share a compute unit's
// registers, 128 each; beyond these counts so much of a tile spills to scratch
// that the per-step kernels win: 1700x350, L=2, FDORDER 8 (three rows) took
// 77 ms a shot gradient of 1500 steps against their 75 ms, 1024x1024 elastic
// (four rows) 23.4 us a step against 24.4 and no gain over a gradient.
constexpr int resident_max_rows(int L) { return L == 0 ? 3 : L <= 3 ? 2 : 0; }

// A line of the inbox is one word per cell: the value in the low half, the
// step it belongs to in the high half, written and read as one 64-bit atomic,
// so that a word whose tag matches carries its value (no separate flag, no
// fence).  Inbox of a workgroup and half step: M = 2N - 1 lines from each
// side; from below and from above [line][64], then from the right and from
// the left [row][line].
struct ResidentArgs {
    const StepArgs *a;       // argument block in device memory
    unsigned long long *inbox;  // [workgroup][2][words]: stresses, then velocities
    int *stop;               // nonzero: a workgroup gave up waiting, all leave
    int words;               // inbox words per workgroup and half step
    int th, ty;              // tile rows, rows of threads
    int tiles_y, ntile;      // tile rows of the grid, tiles per slot
    int nwg, per;            // workgroups at work, and per XCD
    unsigned long long limit;  // longest wait for a neighbour, ticks of the 100 MHz clock
};

// launch shape of a resident run, decided on the host (resident_plan)
struct ResidentPlan {
    int rows = 0;            // rows per thread, 0: not eligible
    int ty = 0, th = 0, tiles_y = 0, nwg = 0, words = 0;
    size_t lds = 0;
};

// the plan for nslots shots of a grid on a device of ncu compute units with
// lds_max bytes of LDS per workgroup; rows 0 when the run does not fit
ResidentPlan resident_plan(const StepGeom &g, int L, int nslots, int snap_prec, int ncu, size_t lds_max);
// one run of NT steps, fields zero at the start; r: a, inbox, stop and limit set
hipError_t launch_resident(const StepArgs &a, ResidentArgs r, const ResidentPlan &p, hipStream_t s);

}  // namespace ifos
