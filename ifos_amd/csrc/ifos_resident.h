// ifos_resident.h -- the time loop as one launch (k_resident): argument block
// and plan.
//
// Each workgroup owns a tile of 64 columns x th rows for the whole run.  The
// wavefields of the tile and the halo its stencils read sit in LDS, the
// memory variables in registers, the update coefficients in registers with one
// row of cells per thread, else in LDS as far as they fit.  After each half step a
// workgroup hands the N edge lines its neighbours read to their inboxes in
// device memory and waits for theirs; nothing else synchronises the tiles.
//
// What bounds it: with one row of cells per thread the latency of a half step,
// a chain of instructions more than of memory (400x200 elastic, FDORDER 4,
// 3.7 us a step: 1.7 update, 0.7 polling and unpacking, 0.8 sending, 0.3 waiting
// for the write-through stores that the polling loads queue behind, 0.2 for
// neighbours), so the loop keeps divisions, address arithmetic and anything rare
// out of its registers and its path.  With more rows vector instructions fill about
// half of a SIMD's cycles (1024x768 elastic: 834 per wavefront and step, four
// wavefronts a SIMD, 4 cycles each, of 26 k); LDS, the exchange and reloads of spilled
// values take the rest.
// The per-step kernels pay two launches a step, each with its ramp, drain and
// cold loads.  Time per forward step, those and this (us): FDORDER 8, L=2:
// 1024x256 12.7 / 5.9, 1024x512 18.7 / 9.7, 1024x768 25.2 / 17.8; elastic:
// 1024x768 FDORDER 8 19.5 / 11.6, 1024x256 FDORDER 4 10.1 / 5.0.
#pragma once
#include "ifos_step.h"

namespace ifos {

constexpr int kResidentThreads = 1024;  // largest workgroup: 64 columns x 16 rows of threads

// Rows of cells per thread the kernel is compiled for, by the stencil reach and
// the number of relaxation mechanisms (0: not compiled).  1024 threads share a
// compute unit's registers, 128 each, and its LDS.  us per forward step of a full
// chip, per-step kernels and this, FDORDER 8: elastic, four rows 23.7 / 13.8, six
// 32.9 / 27.7; L=1, four 27.6 / 21.8; L=2, three 25.3 / 17.8, four 30.0 / 26.7;
// L=3, three 27.0 / 24.5.  Four rows with L=2 spill too much beyond FDORDER 8
// (FDORDER 12, 56 rows of cells: 32.0 / 34.5, 64 34.2 / 33.0).  Six rows of FDORDER 12
// exceed the LDS.
constexpr int resident_max_rows(int N, int L)
{
    return L == 0 ? (N <= 5 ? 6 : 5) : L == 1 || (L == 2 && N <= 4) ? 4 : L <= 3 ? 3 : 0;
}

// Where the registers spill most the tiles have to be nearly full: a tile just
// over the height of one row fewer takes as long as a full one.  FDORDER 8, a
// gradient's pair of steps (us), per-step kernels and this: L=2, 49 rows of cells 57.8
// / 59.0, 52 60.3 / 60.4, 56 63.8 / 59.0; L=3, 33 rows 48.4 / 46.7 (a forward step
// 21.2 / 21.3, FDORDER 12 53.4 / 55.0), 40 55.0 / 51.5; elastic with a snapshot every
// step, 82 rows, FP32 forward 36.5 / 37.5, BF16 adjoint 53.1 / 56.9, 88 rows 38.8 / 37.6
// and 57.1 / 58.1.  Elastic tiles of five rows are faster from their lowest height on:
// 65 rows 55.2 / 48.3, FDORDER 12 63.9 / 58.1.
constexpr bool resident_pays(int N, int L, int rows, int th)
{
    const bool crowded = N >= 4 && rows >= (L == 0 ? 6 : L == 3 ? 3 : 4) && L != 1;
    return !crowded || th >= 16 * rows - 8;
}

// A step that stores 16-bit snapshots costs more here than in the per-step kernels
// (the values wait in memory for the scale of their tile, behind a barrier; tiles
// round up to multiples of eight rows), so with three and more rows per thread such
// a forward run has to fill more of the tile the more often it stores: this many
// percent of the 16 * rows rows of cells, by the stencil's reach.  Forward runs, BF16,
// how many times as fast as the per-step kernels at DTINV 1 and 8: elastic, FDORDER 8,
// 82 of 96 rows of cells 0.74 and 1.15, 80 of 80 0.97 and 1.48; L=2, FDORDER 8, 50 of 64
// 0.90 and 1.13, 48 of 48 1.32 and 1.91; L=3, FDORDER 12, 40 of 48 0.88 and 0.98, 48 of
// 48 1.00 and 1.09.  With the 25 or 40 percent of every step's store the heights at
// which the two are equal lie within 5 of the table at DTINV 1, 2, 3, 4, 6 and 8; one
// and two rows are faster throughout.
constexpr int resident_fill16(int N, int L, int rows, int DTINV)
{
    constexpr unsigned char share[9][6] = {
        {46, 53, 58, 60, 60, 53}, {57, 65, 65, 60, 65, 67}, {51, 61, 62, 73, 75, 67}, {63, 78, 77, 84, 76, 84},  // L=0, 3-6
        {44, 44, 44, 52, 45, 49}, {53, 51, 55, 73, 60, 69},                                                      // L=1, 3-4
        {44, 44, 52, 63, 52, 68}, {66, 68, 76, 83, 83, 83},                                                      // L=2, 3-4
        {44, 56, 71, 84, 79, 84}};                                                                               // L=3, 3
    if (rows < 3) return 0;
    return share[(L == 0 ? 0 : 2 + 2 * L) + rows - 3][N - 1] + (L == 0 && rows >= 5 ? 40 : 25) / DTINV;
}

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

// Cell of the padded grid whose materials row r of a thread is given (c: the cell
// of its row 0): its own, or, where that lies past the grid's last row or column,
// cell (1, 1), which every grid has.  The last tile's rows can lie a tile's height
// past the padding.
__host__ __device__ inline unsigned material_cell(unsigned c, int r, int pitch, bool inside)
{
    return inside ? c + (unsigned)(r * pitch) : (unsigned)pitch + 1u;
}

// launch shape of a resident run, decided on the host (resident_plan)
struct ResidentPlan {
    int rows = 0;            // rows per thread, 0: not eligible
    int ty = 0, th = 0, tiles_y = 0, nwg = 0, words = 0;
    int cells = 0;           // rows of cells a tile has to hold (th: rounded up)
    size_t lds = 0;
};

// the plan for nslots shots of a grid on a device of ncu compute units with
// lds_max bytes of LDS per workgroup; snap_prec: that of the snapshots the run
// stores, 0 when it stores none; rows 0 when the run does not fit
ResidentPlan resident_plan(const StepGeom &g, int L, int nslots, int snap_prec, int ncu, size_t lds_max);
// one run of NT steps, fields zero at the start; r: a, inbox, stop and limit set
hipError_t launch_resident(const StepArgs &a, ResidentArgs r, const ResidentPlan &p, hipStream_t s);

}  // namespace ifos
