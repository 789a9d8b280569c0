// ifos_resident.h -- the time loop as one launch (k_resident): argument block
// and plan.
//
// Each workgroup owns a tile of 64 columns x th rows for the whole run.  The
// wavefields of the tile and the halo its stencils read sit in LDS, the
// memory variables and materials in registers.  After each half step a
// workgroup hands the N edge lines its neighbours read to their inboxes in
// device memory and waits for theirs; nothing else synchronises the tiles.
//
// What bounds it: with one row of cells per thread the latency of a half step,
// a chain of instructions more than of memory (400x200 elastic, FDORDER 4,
// 3.7 us a step: 1.7 update, 0.7 polling and unpacking, 0.8 sending, 0.3 waiting
// for the write-through stores that the polling loads queue behind, 0.2 for
// neighbours), so the loop keeps divisions, address arithmetic and anything rare
// out of its registers and its path; with more rows the instructions issued.
// The per-step kernels pay two launches a step, each with its ramp, drain and
// cold loads.  Time per forward step, those and this (us): FDORDER 8, L=2:
// 1024x256 13.2 / 5.6, 1024x512 20.0 / 13.0, 1024x768 26.5 / 21.4; elastic:
// 1200x600 FDORDER 8 18.9 / 11.4, 1024x256 FDORDER 4 10.2 / 5.1.
#pragma once
#include "ifos_step.h"

namespace ifos {

constexpr int kResidentThreads = 1024;  // largest workgroup: 64 columns x 16 rows of threads

// Rows of cells per thread the kernel is compiled for, by the number of
// relaxation mechanisms (0: not compiled).  1024 threads share a compute unit's
// registers, 128 each; with these counts at most a few dozen values spill and
// the run is faster than the per-step kernels' (us per forward step of a full
// chip, FDORDER 8: elastic, four rows 25.1 / 17.3, L=2, three rows 26.5 / 21.4,
// L=3, two rows 22.0 / 16.4).
constexpr int resident_max_rows(int L) { return L == 0 ? 4 : L <= 2 ? 3 : L <= 3 ? 2 : 0; }

constexpr int kWordsPerThread = 3;  // inbox words a thread polls, one row per thread

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
