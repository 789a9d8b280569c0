// ifos_stepdev.h -- device code shared by the time-loop kernels: step flags,
// the work items of a launch, memory-variable indexing, 16-bit snapshots and
// the halo copies of periodic sides.
#pragma once
#include "ifos_cellmath.h"
#include "ifos_step.h"

namespace ifos {

__device__ __forceinline__ int step_number(const StepArgs &a, int k) { return a.base ? *gmem(a.base) + k + 1 : k; }

// Per-launch step flags, decided on the host: kSnapStep for a forward step
// that stores a snapshot, (nt-1) % DTINV == 0 (src/IFOS2D.c:1805); kCorrStep
// for an adjoint step that correlates, (NT-nt) % DTINV == 0
// (src/IFOS2D.c:2381).  Inside a graph unit (a.base set) step nt is
// base + k + 1 with base a multiple of the unit, and the unit a multiple of
// DTINV dividing NT, so both tests depend on k alone.
// The other flags restate fields of the argument block that every wave
// would otherwise load before it can branch: kForward (sw == 0), kAdjInt
// (adjoint with VELOCITY == 0: the integrated adjoint velocity,
// src/update_v_PML.c:140-143) and kEnergy (the preconditioner's energy sums).
constexpr int kSnapStep = 1, kCorrStep = 2, kForward = 4, kAdjInt = 8, kEnergy = 16;

// Workgroups are dealt round-robin to the 8 XCDs (workgroup h runs on XCD
// h % 8), and each XCD has its own L2.  With swizzle on, XCD x works through
// one contiguous run [xlo[x], xlo[x+1]) of the work items in row-major tile
// order, so the halos neighbouring tiles share, and the materials the slot
// groups of a tile share, are mostly fetched into one L2 once.  The runs have
// equal estimated cost rather than equal length (shaped_args).

// n / d for 0 <= n < 2^31 from (mul, sh) of make_div: t = mulhi(n, mul),
// q = (((n - t) >> 1) + t) >> sh; sh = 0 with mul = 0 marks d = 1
__device__ __forceinline__ uint32_t fdiv(uint32_t n, uint32_t mul, uint32_t sh)
{
    if (mul == 0) return n;
    const uint32_t t = __umulhi(n, mul);
    return (((n - t) >> 1) + t) >> sh;
}

// The work-item mapping of a launch, read from the argument block into
// locals once per workgroup, so that these loads issue together instead of
// one by one where they are first used.
struct ItemMap {
    int nbx, ntiles, nslots, ngroups, slot_major, swizzle;
    uint32_t nbx_mul, nbx_sh, ng_mul, ng_sh, nt_mul, nt_sh;
    int lo, hi;  // this workgroup's XCD run of items
};

__device__ __forceinline__ ItemMap item_map(const StepArgs &a)
{
    ItemMap m;
    m.nbx = a.nbx;
    m.ntiles = a.nbx * a.nby;
    m.nslots = a.nslots;
    m.ngroups = a.ngroups;
    m.slot_major = a.slot_major;
    m.swizzle = a.swizzle;
    m.nbx_mul = a.nbx_mul;
    m.nbx_sh = a.nbx_sh;
    m.ng_mul = a.ng_mul;
    m.ng_sh = a.ng_sh;
    m.nt_mul = a.nt_mul;
    m.nt_sh = a.nt_sh;
    const int x = blockIdx.x % 8;
    m.lo = a.xlo[x];
    m.hi = a.xlo[x + 1];
    return m;
}

// tile and first slot of work item it
__device__ __forceinline__ void item_of(const ItemMap &m, int it, int spb, int &blk, int &s0)
{
    if (m.slot_major) {
        const int grp = (int)fdiv(it, m.nt_mul, m.nt_sh);
        blk = it - grp * m.ntiles;
        s0 = grp * spb;
    } else {
        blk = (int)fdiv(it, m.ng_mul, m.ng_sh);
        s0 = (it - blk * m.ngroups) * spb;
    }
}

// items [first, end) with the given stride for this workgroup: one item per
// workgroup, or a persistent grid (gridDim.x a multiple of 8) looping over
// the items of its XCD's run
__device__ __forceinline__ void work_range(const ItemMap &m, int nitems, bool persistent, int &first, int &end,
                                           int &stride)
{
    const int h = blockIdx.x;
    int lo = 0, hi = nitems;
    if (m.swizzle) {
        lo = m.lo;
        hi = m.hi;
    }
    if (!persistent) {
        first = m.swizzle ? lo + h / 8 : h;
        end = m.swizzle ? (first < hi ? first + 1 : first) : first + 1;
        stride = 1;
    } else if (m.swizzle) {
        first = lo + h / 8;
        end = hi;
        stride = gridDim.x / 8;
    } else {
        first = h;
        end = nitems;
        stride = gridDim.x;
    }
}

// Memory variables r_l, p_l, q_l of a slot are interleaved per 64 cells of
// the padded grid: component k (r_l: l, p_l: L + l, q_l: 2L + l) of cell c
// sits at ((c - 1) / 64 * 3L + k) * 64 + (c - 1) % 64 from the slot's block
// of 3L fields.  The pitch is a multiple of 64 and a tile's cells start at
// column 1, so the 64 cells of a wavefront's row are one chunk and all 3L
// components of it one contiguous run: two streams (read, write) instead of
// 3L each, which DRAM serves faster (a copy with 32 separate arrays ran at
// 5.2 TB/s, the same bytes interleaved at 5.7 TB/s).  Cells are interior
// (c >= pitch + 1), so the index stays inside the block.
__device__ __forceinline__ long mv_index(long c, int k, int L3)
{
    const long cc = c - 1;
    return ((cc >> 6) * L3 + k) * 64 + (cc & 63);
}

// ---------------------------------------------------------------------------
// Points at a cell.  first_point: the first one of slot s at interior cell e,
// -1 when there is none; `any` (uniform): whether the cell's tile has points.
__device__ __forceinline__ bool tile_has(const PointMap &p, int s, int ntiles, int blk)
{
    const int so = __builtin_amdgcn_readfirstlane(s * (ntiles + 1) + blk);  // uniform
    return cmem(p.start)[so + 1] > cmem(p.start)[so];
}

__device__ __forceinline__ int first_point(const StepArgs &a, const PointMap &p, int s, long e, bool any)
{
    return any ? gmem(p.map)[(long)s * a.plane + e] : -1;
}

// point force (forward) or residual injection (adjoint) of point l at step
// nt, whose samples are s0, s1 (A: the argument block through a plain or a
// constant-space reference)
template <class A>
__device__ __forceinline__ void inject_values(A &a, int l, float s0, float s1, float rip, float rjp, float &vx,
                                              float &vy)
{
    const auto &g = a.g;
    if (a.sw == 0) {
        const int type = gmem(a.inj.type)[l];
        if (type == 2) vx += (g.DT * rip * s1) / (g.DH * g.DH);
        if (type == 3) vy += (g.DT * rjp * s1) / (g.DH * g.DH);
        if (type == 4) {
            vx += (g.DT * rip * gmem(a.inj.sin_azi)[l] * s0) / (g.DH * g.DH);
            vy += (g.DT * rjp * gmem(a.inj.cos_azi)[l] * s0) / (g.DH * g.DH);
        }
    } else {
        if (a.ADJOINT_TYPE == 1) { vx += s0; vy += s1; }
        if (a.ADJOINT_TYPE == 2) vy += s1;
        if (a.ADJOINT_TYPE == 3) vx += s0;
    }
}

template <class A>
__device__ __forceinline__ void inject(A &a, int l, int nt, float rip, float rjp, float &vx, float &vy)
{
    inject_values(a, l, gmem(a.inj.sig)[(long)l * a.NT + nt - 1], gmem(a.inj.sig1)[(long)l * a.NT + nt - 1], rip, rjp,
                  vx, vy);
}

// ---------------------------------------------------------------------------
// 16-bit snapshots.  A tile's values of one field are divided by 2^e, the
// smallest power of two above their largest magnitude (exact in binary
// floating point), and rounded to nearest-even BF16 or FP16.
template <class A>
__device__ __forceinline__ bool has_snap(A &a) { return a.snap[0] || a.snap16[0]; }

__device__ __forceinline__ int scale_exp(float m)
{
    if (!(m > 0.0f) || isinf(m)) return 0;
    return min(max(ilogbf(m) + 1, -120), 120);
}

__device__ __forceinline__ uint16_t enc16(float x, float inv_scale, int prec)
{
    const float y = x * inv_scale;
    if (prec == 1) {
        uint32_t u = __float_as_uint(y);
        u += 0x7FFFu + ((u >> 16) & 1u);
        return (uint16_t)(u >> 16);
    }
    return __builtin_bit_cast(uint16_t, (_Float16)y);
}

__device__ __forceinline__ float dec16(uint16_t h, float scale, int prec)
{
    if (prec == 1) return __uint_as_float((uint32_t)h << 16) * scale;
    return (float)__builtin_bit_cast(_Float16, h) * scale;
}

// largest |v| over the block of NW waves (blockDim.y == NW), for NF values at
// once; every thread of the block must call it (it holds two barriers)
template <int NF, int NW = kTileY>
__device__ __forceinline__ void block_absmax(float (&v)[NF], float (*lds)[kTileY])
{
#pragma unroll
    for (int f = 0; f < NF; f++) {
        float m = fabsf(v[f]);
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
        if (threadIdx.x == 0) lds[f][threadIdx.y] = m;
    }
    __syncthreads();
#pragma unroll
    for (int f = 0; f < NF; f++) {
        float m = lds[f][0];
#pragma unroll
        for (int w = 1; w < NW; w++) m = fmaxf(m, lds[f][w]);
        v[f] = m;
    }
    __syncthreads();
}

// store NF snapshot fields (first field index f0) of one cell of slot s for
// snapshot slot k; with 16-bit storage every thread of the block must call it
template <int NF>
__device__ __forceinline__ void snap_store(const StepArgs &a, int s, int f0, long k, long e, int blk, bool live,
                                           const float (&val)[NF], float (*lds)[kTileY])
{
    const long o = (long)s * a.sns + k * a.plane + e;
    if (a.snap_prec == 0) {
        if (live)
#pragma unroll
            for (int f = 0; f < NF; f++) gmem(a.snap[f0 + f])[o] = val[f];
        return;
    }
    float m[NF];
#pragma unroll
    for (int f = 0; f < NF; f++) m[f] = live ? val[f] : 0.0f;
    block_absmax<NF>(m, lds);
    const long ntile = (long)a.nbx * a.nby;
#pragma unroll
    for (int f = 0; f < NF; f++) {
        const int ex = scale_exp(m[f]);
        if (live) gmem(a.snap16[f0 + f])[o] = enc16(val[f], ldexpf(1.0f, -ex), a.snap_prec);
        if (threadIdx.x == 0 && threadIdx.y == 0) gmem(a.sscale[f0 + f])[(long)s * a.scs + k * ntile + blk] = ldexpf(1.0f, ex);
    }
}

// snap_store for the R cells (rows j .. j+R-1, interior indices e + r*NX) of
// a thread in a 64x(8/R) block of R-row threads; the 16-bit scale is the
// same 64x8 tile maximum as in snap_store
template <int NF, int R>
__device__ __forceinline__ void snap_store_rows(const StepArgs &a, int s, int f0, long k, long e, int blk,
                                                const bool (&live)[R], const float (&val)[R][NF],
                                                float (*lds)[kTileY])
{
    const long o = (long)s * a.sns + k * a.plane + e;
    const int NX = a.g.NX;
    if (a.snap_prec == 0) {
#pragma unroll
        for (int r = 0; r < R; r++)
            if (live[r])
#pragma unroll
                for (int f = 0; f < NF; f++) gmem(a.snap[f0 + f])[o + r * NX] = val[r][f];
        return;
    }
    float m[NF];
#pragma unroll
    for (int f = 0; f < NF; f++) {
        m[f] = live[0] ? fabsf(val[0][f]) : 0.0f;
#pragma unroll
        for (int r = 1; r < R; r++) m[f] = fmaxf(m[f], live[r] ? fabsf(val[r][f]) : 0.0f);
    }
    block_absmax<NF, kTileY / R>(m, lds);
    const long ntile = (long)a.nbx * a.nby;
#pragma unroll
    for (int f = 0; f < NF; f++) {
        const int ex = scale_exp(m[f]);
        const float inv = ldexpf(1.0f, -ex);
#pragma unroll
        for (int r = 0; r < R; r++)
            if (live[r]) gmem(a.snap16[f0 + f])[o + r * NX] = enc16(val[r][f], inv, a.snap_prec);
        if (threadIdx.x == 0 && threadIdx.y == 0) gmem(a.sscale[f0 + f])[(long)s * a.scs + k * ntile + blk] = ldexpf(1.0f, ex);
    }
}

__device__ __forceinline__ float snap_load(const StepArgs &a, int s, int f, long k, long e, int blk)
{
    const long o = (long)s * a.sns + k * a.plane + e;
    if (a.snap_prec == 0) return gmem(a.snap[f])[o];
    const float sc = gmem(a.sscale[f])[(long)s * a.scs + k * (long)a.nbx * a.nby + blk];
    return dec16(gmem(a.snap16[f])[o], sc, a.snap_prec);
}

// ---------------------------------------------------------------------------
// Periodic sides (BOUNDARY 1).  On one rank the reference's exchanges after
// each half step copy the opposite edge into the halo columns
// (src/exchange_v.c:143-228, src/exchange_s.c:145-229): after the velocity
// step vy to columns NX+1..NX+N and 2-N..0, vx to NX+1..NX+N-1 and 1-N..0;
// after the stress step (sources and free surface included) sxx to
// NX+1..NX+N and 2-N..0, sxy to NX+1..NX+N-1 and 1-N..0.  The cell that owns
// the final value also stores it into its halo copy.  No kernel of the same
// launch reads those halo columns: the velocity step reads stress halos, the
// stress step velocity halos.  The padded rows hold at least 16 columns left
// of column 1 and N+1 right of column NX, so the copies stay in their row.
template <int N, typename Ptr>
__device__ __forceinline__ void wrap_pair(const StepGeom &g, Ptr a, Ptr b, long c, int i, float av, float bv)
{
    // a: the field with N copies on the right and N-1 on the left (vy, sxx),
    // b: N-1 on the right and N on the left (vx, sxy)
    if (i <= N) {
        a[c + g.NX] = av;
        if (i <= N - 1) b[c + g.NX] = bv;
    }
    if (i >= g.NX - N + 1) {
        b[c - g.NX] = bv;
        if (i >= g.NX - N + 2) a[c - g.NX] = av;
    }
}

}  // namespace ifos
