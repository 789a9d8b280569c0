// ifos_resident_kernels.h -- the time loop as one launch (ifos_resident.h).
// The arithmetic is that of ifos_cellmath.h, operand for operand, so the
// results are the bits of the two-kernel step.
#pragma once
#include <type_traits>

#include "ifos_resident.h"
#include "ifos_stepdev.h"

namespace ifos {

// Offsets of the LDS arrays of a tile, in floats.  Row r, column x of the
// tile (0-based) sit at vx, vy, sxy: (r + N) * W + x + N; sxx (no rows above
// and below): r * W + x + N; syy (no columns to the sides): (r + N) * 64 + x.
template <int N>
struct ResLds {
    static constexpr int W = kTileX + 2 * N;
    __host__ __device__ static int vx(int) { return 0; }
    __host__ __device__ static int vy(int th) { return (th + 2 * N) * W; }
    __host__ __device__ static int sxy(int th) { return 2 * (th + 2 * N) * W; }
    __host__ __device__ static int sxx(int th) { return 3 * (th + 2 * N) * W; }
    __host__ __device__ static int syy(int th) { return 3 * (th + 2 * N) * W + th * W; }
    __host__ __device__ static int maxima(int th) { return syy(th) + (th + 2 * N) * kTileX; }
    __host__ __device__ static int total(int th) { return maxima(th) + 5 * th; }
};

// The argument block, read afresh: what a block of code needs of it is loaded
// there (scalar loads that hit the constant cache) instead of staying in
// registers for the whole run, and likewise the lane's cell offsets.
typedef const IFOS_CAS StepArgs *ArgPtr;
__device__ __forceinline__ ArgPtr afresh(ArgPtr p)
{
    asm volatile("" : "+s"(p));
    return p;
}
__device__ __forceinline__ unsigned afresh(unsigned v)
{
    asm volatile("" : "+v"(v));
    return v;
}

// element at a 32-bit byte offset from a uniform base: one scalar base and one
// offset register per access instead of a 64-bit address per lane
template <class P>
__device__ __forceinline__ auto &at(P base, unsigned byte)
{
    typedef typename std::remove_reference<decltype(*base)>::type T;
    if constexpr (std::is_const<T>::value) return *(P)((const IFOS_GAS char *)base + byte);
    else return *(P)((IFOS_GAS char *)base + byte);
}

// neighbour sides, as bits
constexpr int kBelow = 1, kAbove = 2, kRight = 4, kLeft = 8;

// Send one cell's pair of values to the neighbours that read them.  p is the
// field of which a tile reads N lines from below (or from the right) and
// N - 1 from above (left), q the one with N - 1 and N; y neighbours and x
// neighbours take different pairs.
struct XDest {
    int p, q;  // inbox word of row 0 for this lane's column, -1: not an edge column
};

__device__ __forceinline__ void send_word(unsigned long long *box, unsigned word, float v, int tag)
{
    const unsigned long long w = ((unsigned long long)(unsigned)tag << 32) | __float_as_uint(v);
    __hip_atomic_store(&at(gmem(box), word * 8u), w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <int N>
__device__ __forceinline__ void send_y(const ResidentArgs &ra, int sides, unsigned up, unsigned dn, int r, int tx, float p,
                                       float q, int tag)
{
    // up: word 0 of the "from below" lines of the tile above; dn: word 0 of
    // the "from above" lines of the tile below; r is uniform in a wavefront
    if ((sides & kAbove) && r < N) {
        send_word(ra.inbox, up + r * kTileX + tx, p, tag);
        if (r < N - 1) send_word(ra.inbox, up + (N + r) * kTileX + tx, q, tag);
    }
    const int b = r - (ra.th - N);
    if ((sides & kBelow) && b >= 0) {
        if (b >= 1) send_word(ra.inbox, dn + (b - 1) * kTileX + tx, p, tag);
        send_word(ra.inbox, dn + (N - 1 + b) * kTileX + tx, q, tag);
    }
}

template <int N>
__device__ __forceinline__ void send_x(const ResidentArgs &ra, const XDest &d, int r, float p, float q, int tag)
{
    if (d.p >= 0) send_word(ra.inbox, afresh(d.p) + r * (2 * N - 1), p, tag);
    if (d.q >= 0) send_word(ra.inbox, afresh(d.q) + r * (2 * N - 1), q, tag);
}

// Take this half step's halo out of the inbox `in` into LDS: py and qy are
// the fields read from below and above, px and qx those from the sides, each
// given by the LDS offset of its row 0, column 0.  Every thread polls its own
// words.  false: a neighbour did not answer within ra.limit, or another
// workgroup gave up.
template <int N>
__device__ __forceinline__ bool receive(const ResidentArgs &ra, const unsigned long long *in_, int sides, int tag,
                                        float *lds, int py, int spy, int qy, int sqy, int px, int spx, int qx, int sqx)
{
    constexpr int M = 2 * N - 1, U = 2;
    const auto in = gmem(in_);
    const int th = ra.th, nthr = kTileX * ra.ty, tid = (int)afresh(threadIdx.y * kTileX + threadIdx.x);
    const int total = ra.words;
    for (int q0 = tid; q0 < total; q0 += U * nthr) {
        unsigned wait = 0;
        int dst[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int q = q0 + u * nthr;
            dst[u] = 0;
            if (q < 2 * M * kTileX) {
                const bool above = q >= M * kTileX;
                const int k = above ? q - M * kTileX : q, l = k / kTileX, x = k % kTileX;
                if (!above) dst[u] = l < N ? py + (th + l) * spy + x : qy + (th + l - N) * sqy + x;
                else dst[u] = l < N - 1 ? py + (l - (N - 1)) * spy + x : qy + (l - (N - 1) - N) * sqy + x;
                if (sides & (above ? kAbove : kBelow)) wait |= 1u << u;
            } else if (q < total) {
                const int h = q - 2 * M * kTileX;
                const bool left = h >= M * th;
                const int k = left ? h - M * th : h, r = k / M, l = k % M;
                if (!left) dst[u] = l < N ? px + r * spx + kTileX + l : qx + r * sqx + kTileX + l - N;
                else dst[u] = l < N - 1 ? px + r * spx + l - (N - 1) : qx + r * sqx + l - (N - 1) - N;
                if (sides & (left ? kLeft : kRight)) wait |= 1u << u;
            }
        }
        unsigned long long since = 0;
        int tries = 0;
        while (wait) {
            unsigned long long w[U];
#pragma unroll
            for (int u = 0; u < U; u++)
                if (wait & (1u << u))
                    w[u] = __hip_atomic_load(&at(in, (unsigned)(q0 + u * nthr) * 8u), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
            for (int u = 0; u < U; u++)
                if ((wait & (1u << u)) && (int)(w[u] >> 32) == tag) {
                    lds[dst[u]] = __uint_as_float((unsigned)w[u]);
                    wait &= ~(1u << u);
                }
            if (wait && ((++tries & 63) == 0 || ra.limit == 0)) {
                const unsigned long long now = wall_clock64();
                if (since == 0) since = now;
                if (now - since >= ra.limit) {
                    __hip_atomic_store(gmem(ra.stop), 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    return false;
                }
                if (__hip_atomic_load(gmem(ra.stop), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return false;
            }
        }
    }
    return true;
}

// One cell's NF snapshot values (first field f0), cell offset e, row `row` of
// the tile.  FP32: stored.  16-bit: kept in the planes of `keep` (offset c in
// the padded grid; unused in a forward run) until the scale of their 64x8 tile
// is known, and the wavefront's maxima of the row go to LDS.
template <int NF, class A>
__device__ __forceinline__ void res_snap_put(A &a, int s, int f0, long k, unsigned e, unsigned c, bool live, int row,
                                             const float (&val)[NF], float *const (&keep)[NF], float *maxima)
{
    if (a.snap_prec == 0) {
        const long o = (long)s * a.sns + k * a.plane;
        if (live)
#pragma unroll
            for (int f = 0; f < NF; f++) at(gmem(a.snap[f0 + f]) + o, e * 4u) = val[f];
        return;
    }
#pragma unroll
    for (int f = 0; f < NF; f++) {
        if (live) at(gmem(keep[f]) + (long)s * a.ws, c * 4u) = val[f];
        float m = live ? fabsf(val[f]) : 0.0f;
#pragma unroll
        for (int w = 32; w > 0; w >>= 1) m = fmaxf(m, __shfl_xor(m, w));
        if (threadIdx.x == 0) maxima[row * NF + f] = m;
    }
}

// 16-bit storage: encode the kept values.  The 64x8 tiles of the scales lie
// whole inside the workgroup's tile (th is a multiple of 8 then).
template <int NF, int R, class A>
__device__ __forceinline__ void res_snap_encode(A &a, int s, int f0, long k, unsigned e, unsigned c, int i, int j,
                                                int row, int bx, float *const (&keep)[NF], const float *maxima)
{
    if (a.snap_prec == 0) return;
    __syncthreads();
    const long o = (long)s * a.sns + k * a.plane, ntile = (long)a.nbx * a.nby;
#pragma unroll 1
    for (int r = 0; r < R; r++, row++, j++, e += a.g.NX, c += a.g.pitch) {
        const int t0 = row / kTileY * kTileY;  // first row of the scale's tile
        const long blk = (long)((j - 1) / kTileY) * a.nbx + bx;
        if (i > a.g.NX || j > a.g.NY) continue;
#pragma unroll
        for (int f = 0; f < NF; f++) {
            float m = maxima[t0 * NF + f];
#pragma unroll
            for (int w = 1; w < kTileY; w++) m = fmaxf(m, maxima[(t0 + w) * NF + f]);
            const int ex = scale_exp(m);
            const float v = at(gmem(keep[f]) + (long)s * a.ws, c * 4u);
            at(gmem(a.snap16[f0 + f]) + o, e * 2u) = enc16(v, ldexpf(1.0f, -ex), a.snap_prec);
            if (threadIdx.x == 0 && row == t0) gmem(a.sscale[f0 + f])[(long)s * a.scs + k * ntile + blk] = ldexpf(1.0f, ex);
        }
    }
}

template <class A>
__device__ __forceinline__ float res_snap_load(A &a, int s, int f, long k, unsigned e, int blk)
{
    const long o = (long)s * a.sns + k * a.plane;
    if (a.snap_prec == 0) return at(gmem(a.snap[f]) + o, e * 4u);
    const float sc = gmem(a.sscale[f])[(long)s * a.scs + k * (long)a.nbx * a.nby + blk];
    return dec16(at(gmem(a.snap16[f]) + o, e * 2u), sc, a.snap_prec);
}

// One workgroup: the tile of 64 columns x th rows at (bx, by) of one slot,
// NT steps.  Thread (tx, ty) owns column tx, rows R*ty .. R*ty+R-1.
template <int N, int L, int R>
__global__ __launch_bounds__(kResidentThreads) void k_resident(const ResidentArgs ra)
{
    using D = ResLds<N>;
    constexpr int W = D::W, M = 2 * N - 1, L1 = L > 0 ? L : 1;
    const ArgPtr pa = cmem(ra.a);
    const auto &a = *pa;
    const auto &g = a.g;
    extern __shared__ float lds[];
    __shared__ int s_stop;  // half step in which a thread of this workgroup gave up, 0: none
    const int wg = (int)(blockIdx.x % 8) * ra.per + (int)blockIdx.x / 8;
    if ((int)blockIdx.x / 8 >= ra.per || wg >= ra.nwg) return;
    const int th = ra.th, tx = threadIdx.x, ty = __builtin_amdgcn_readfirstlane(threadIdx.y);
    const int s = wg / ra.ntile, t = wg - s * ra.ntile, by = t / a.nbx, bx = t - by * a.nbx;
    const int NX = g.NX, NY = g.NY, P = g.pitch;
    const int i = bx * kTileX + tx + 1, j0 = by * th, r0 = ty * R, j = j0 + r0 + 1;  // first row of this thread
    const unsigned c = (unsigned)(j * P + i), e = (unsigned)((j - 1) * NX + (i - 1));  // first cell of this thread
    const bool fwd = a.sw == 0;
    bool live[R];
#pragma unroll
    for (int r = 0; r < R; r++) live[r] = i <= NX && j + r <= NY;

    // ---- LDS, all zero (fields, and what lies outside the grid for good)
    for (int q = ty * kTileX + tx; q < D::total(th); q += kTileX * ra.ty) lds[q] = 0.0f;
    if (tx == 0 && ty == 0) s_stop = 0;
    // offsets of row 0, column 0
    const int oVX = D::vx(th) + N * W + N, oVY = D::vy(th) + N * W + N, oSXY = D::sxy(th) + N * W + N;
    const int oSXX = D::sxx(th) + N, oSYY = D::syy(th) + N * kTileX;
    float *const VX = lds + oVX, *const VY = lds + oVY, *const SXY = lds + oSXY, *const SXX = lds + oSXX;
    float *const SYY = lds + oSYY, *const maxima = lds + D::maxima(th);

    // ---- neighbours
    const int sides = (by + 1 < ra.tiles_y ? kBelow : 0) | (by > 0 ? kAbove : 0) | (bx + 1 < a.nbx ? kRight : 0) |
                      (bx > 0 ? kLeft : 0);
    const unsigned long long *in = ra.inbox + (long)wg * 2 * ra.words;
    const unsigned up = (unsigned)(wg - a.nbx) * 2 * ra.words;              // "from below" of the tile above
    const unsigned dn = (unsigned)(wg + a.nbx) * 2 * ra.words + M * kTileX;  // "from above" of the tile below
    XDest xd;
    xd.p = xd.q = -1;
    {
        const int lt = (wg - 1) * 2 * ra.words + 2 * M * kTileX + r0 * M;           // "from the right", tile on the left
        const int rt = (wg + 1) * 2 * ra.words + 2 * M * kTileX + (th + r0) * M;    // "from the left", tile on the right
        if (sides & kLeft) {
            if (tx < N) xd.p = lt + tx;
            if (tx < N - 1) xd.q = lt + N + tx;
        }
        if (sides & kRight) {
            if (tx >= kTileX - (N - 1)) xd.p = rt + tx - (kTileX - (N - 1));
            if (tx >= kTileX - N) xd.q = rt + N - 1 + tx - (kTileX - N);
        }
    }

    // ---- materials and memory variables
    float rip[R], rjp[R], m0[R], m1[R], m2[R], m3[R], m4[R], m5[R];
    float rr[R][L1], pp[R][L1], qq[R][L1];
#pragma unroll
    for (int r = 0; r < R; r++) {
        const unsigned ci = live[r] ? c + r * P : P + 1u;  // cell (1, 1): every grid has it
        rip[r] = at(gmem(a.rip), ci * 4u);
        rjp[r] = at(gmem(a.rjp), ci * 4u);
        if (L == 0) {
            m0[r] = at(gmem(a.f), ci * 4u);
            m1[r] = at(gmem(a.gl), ci * 4u);
            m2[r] = at(gmem(a.uipjp), ci * 4u);
        } else {
            m0[r] = at(gmem(a.mu), ci * 4u);
            m1[r] = at(gmem(a.pi), ci * 4u);
            m2[r] = at(gmem(a.muipjp), ci * 4u);
            m3[r] = at(gmem(a.taus), ci * 4u);
            m4[r] = at(gmem(a.taup), ci * 4u);
            m5[r] = at(gmem(a.tausipjp), ci * 4u);
        }
#pragma unroll
        for (int l = 0; l < L1; l++) rr[r][l] = pp[r][l] = qq[r][l] = 0.0f;
    }

    // ---- CPML: this column's strip position and profile values
    int hx = -1;
    if (i <= g.FW) hx = i - 1;
    else if (i >= NX - g.FW + 1 && i <= NX) hx = i - NX + 2 * g.FW - 1;
    float Kx = 1.0f, ax = 0.0f, bxp = 0.0f, Kxh = 1.0f, axh = 0.0f, bxh = 0.0f;
    if (hx >= 0) {
        Kx = gmem(g.pml.K_x)[hx]; ax = gmem(g.pml.a_x)[hx]; bxp = gmem(g.pml.b_x)[hx];
        Kxh = gmem(g.pml.K_xh)[hx]; axh = gmem(g.pml.a_xh)[hx]; bxh = gmem(g.pml.b_xh)[hx];
    }
    auto strip_y = [&](int jj) {
        if (!g.FREE_SURF && jj <= g.FW) return jj - 1;
        return jj >= NY - g.FW + 1 && jj <= NY ? jj - NY + 2 * g.FW - 1 : -1;
    };
    const unsigned hp = hx >= 0 ? (unsigned)((j - 1) * g.px + hx) : 0;  // its first cell in the x strips

    // ---- points at these cells
    int pi[R], pr[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        pi[r] = live[r] ? gmem(a.inj.map)[(long)s * a.plane + (e + r * NX)] : -1;
        pr[r] = live[r] && fwd ? gmem(a.rec.map)[(long)s * a.plane + (e + r * NX)] : -1;
    }
    const bool explosive = fwd && gmem(a.explosive)[s] != 0;
    const bool has_snaps = fwd && has_snap(a);
    const bool integ = !fwd && a.VELOCITY == 0, energy = a.wacc || a.wacc64;
    const float scale = L ? (float)(1.0 / (double)g.DH) : g.DT / g.DH;
    const int NT = a.NT, DTINV = a.DTINV, K_one = g.K_one, fw = g.FW, fs = g.FREE_SURF, vel = a.VELOCITY;
    const float DT = g.DT, DH = g.DH;
    float hc[N + 1], eta[L1 + 1], bip[L1 + 1], bjm[L1 + 1], cip[L1 + 1], cjm[L1 + 1];
#pragma unroll
    for (int m = 1; m <= N; m++) hc[m] = g.hc[m];
#pragma unroll
    for (int l = 1; l <= L1; l++) {
        eta[l] = a.eta[l];
        bip[l] = a.bip[l];
        bjm[l] = a.bjm[l];
        cip[l] = a.cip[l];
        cjm[l] = a.cjm[l];
    }
    __syncthreads();

    for (int nt = 1; nt <= NT; nt++) {
        const bool snap = has_snaps && (nt - 1) % DTINV == 0;
        const bool corr = !fwd && (NT - nt) % DTINV == 0;
        const long ks = fwd ? (nt - 1) / DTINV : (NT - nt) / DTINV;
        const bool rates = snap && vel == 1;

        // ================= velocities
        if (nt > 1 && !receive<N>(ra, in, sides, nt - 1, lds, oSYY, kTileX, oSXY, W, oSXX, W, oSXY, W)) s_stop = 2 * nt;
        __syncthreads();
        if (s_stop && s_stop <= 2 * nt) return;
        {
            float sxx_x[R], sxy_x[R], sxy_y[R], syy_y[R];
            {
                const float *S = SXY + r0 * W + tx, *Y = SYY + r0 * kTileX + tx, *X = SXX + r0 * W + tx;
                float cy[2 * N + R - 1], cs[2 * N + R - 1];
#pragma unroll
                for (int k = 0; k < 2 * N + R - 1; k++) {
                    cy[k] = S[(k - N) * W];
                    cs[k] = Y[(k - N + 1) * kTileX];
                }
#pragma unroll
                for (int r = 0; r < R; r++) {
                    __builtin_amdgcn_sched_barrier(0);
                    const float *sx = X + r * W, *sy = S + r * W;
                    sxx_x[r] = hc[1] * (sx[1] - sx[0]);
                    sxy_x[r] = hc[1] * (cy[N + r] - sy[-1]);
                    sxy_y[r] = hc[1] * (cy[N + r] - cy[N + r - 1]);
                    syy_y[r] = hc[1] * (cs[N + r] - cs[N + r - 1]);
#pragma unroll
                    for (int m = 2; m <= N; m++) {
                        sxx_x[r] = sxx_x[r] + hc[m] * (sx[m] - sx[1 - m]);
                        sxy_x[r] = sxy_x[r] + hc[m] * (sy[m - 1] - sy[-m]);
                        sxy_y[r] = sxy_y[r] + hc[m] * (cy[N + r + m - 1] - cy[N + r - m]);
                        syy_y[r] = syy_y[r] + hc[m] * (cs[N + r + m - 1] - cs[N + r - m]);
                    }
                }
            }
            // CPML: all memory values load before any is stored
            if (hx >= 0) {
                const auto &b = *afresh(pa);
                const auto p1 = gmem(b.psi_sxx_x) + (long)s * b.pss, p2 = gmem(b.psi_sxy_x) + (long)s * b.pss;
                const unsigned o = afresh(hp), px = b.g.px;
                float v1[R], v2[R];
#pragma unroll
                for (int r = 0; r < R; r++)
                    if (live[r]) v1[r] = at(p1, (o + r * px) * 4u), v2[r] = at(p2, (o + r * px) * 4u);
#pragma unroll
                for (int r = 0; r < R; r++)
                    if (live[r]) {
                        v1[r] = bxh * v1[r] + axh * sxx_x[r];
                        sxx_x[r] = (K_one ? sxx_x[r] : sxx_x[r] / Kxh) + v1[r];
                        v2[r] = bxp * v2[r] + ax * sxy_x[r];
                        sxy_x[r] = (K_one ? sxy_x[r] : sxy_x[r] / Kx) + v2[r];
                        at(p1, (o + r * px) * 4u) = v1[r];
                        at(p2, (o + r * px) * 4u) = v2[r];
                    }
            }
#pragma unroll
            for (int r = 0; r < R; r++) {
                const int h = strip_y(j + r);
                if (h >= 0 && i <= NX) {
                    const auto &b = *afresh(pa);
                    const auto &pm = b.g.pml;
                    const unsigned o = afresh((unsigned)(i - 1) * 4u);
                    const auto p1 = gmem(b.psi_syy_y) + (long)s * b.pss + (long)h * b.g.py;
                    const auto p2 = gmem(b.psi_sxy_y) + (long)s * b.pss + (long)h * b.g.py;
                    const float v1 = cmem(pm.b_yh)[h] * at(p1, o) + cmem(pm.a_yh)[h] * syy_y[r];
                    const float v2 = cmem(pm.b_y)[h] * at(p2, o) + cmem(pm.a_y)[h] * sxy_y[r];
                    syy_y[r] = divK(syy_y[r], pm.K_yh, h, K_one) + v1;
                    sxy_y[r] = divK(sxy_y[r], pm.K_y, h, K_one) + v2;
                    at(p1, o) = v1;
                    at(p2, o) = v2;
                }
            }
#pragma unroll
            for (int r = 0; r < R; r++) {
                __builtin_amdgcn_sched_barrier(0);
                const int o = (r0 + r) * W + tx;
                const float vx0 = VX[o], vy0 = VY[o];
                float vx = vel_new(vx0, DT, rip[r], sxx_x[r] + sxy_y[r], DH);
                float vy = vel_new(vy0, DT, rjp[r], sxy_x[r] + syy_y[r], DH);
                if (pi[r] >= 0) {
                    const auto &b = *afresh(pa);
                    for (int l = pi[r]; l >= 0; l = gmem(b.inj.next)[l]) inject(b, l, nt, rip[r], rjp[r], vx, vy);
                }
                if (!live[r]) vx = vy = 0.0f;
                VX[o] = vx;
                VY[o] = vy;
                send_y<N>(ra, sides, up + ra.words, dn + ra.words, r0 + r, (int)afresh(tx), vx, vy, nt);
                XDest xv = xd;  // the velocity half of the inboxes
                xv.p += xd.p >= 0 ? ra.words : 0;
                xv.q += xd.q >= 0 ? ra.words : 0;
                send_x<N>(ra, xv, r, vy, vx, nt);
                if (snap) {
                    const auto &b = *afresh(pa);
                    const float acc[2] = {vel_rate(rip[r], sxx_x[r] + sxy_y[r], DH),
                                          vel_rate(rjp[r], sxy_x[r] + syy_y[r], DH)};
                    float *const keep[2] = {b.vxp1, b.vyp1};
                    res_snap_put<2>(b, s, 0, ks, afresh(e) + r * NX, afresh(c) + r * P, live[r], r0 + r, acc, keep,
                                    maxima);
                }
                if (!live[r]) continue;
                if (integ || corr) {
                    const auto &b = *afresh(pa);
                    const auto qx = gmem(b.vxp1) + (long)s * b.ws, qy = gmem(b.vyp1) + (long)s * b.ws;
                    const unsigned cr = (afresh(c) + r * P) * 4u;
                    if (integ) {
                        at(qx, cr) += vx0 * DT;
                        at(qy, cr) += vy0 * DT;
                    } else {
                        at(qx, cr) = vx0;
                        at(qy, cr) = vy0;
                    }
                }
                if (energy) {
                    const auto &b = *afresh(pa);
                    const unsigned er = afresh(e) + r * NX;
                    if (b.wacc64) {
                        const auto Wd = gmem(b.wacc64) + (long)s * b.wacs;
                        at(Wd, er * 8u) += ((double)vx * (double)vx) + ((double)vy * (double)vy);
                    } else {
                        const auto Wf = gmem(b.wacc) + (long)s * b.wacs;
                        at(Wf, er * 4u) += ((vx * vx) + (vy * vy));
                    }
                }
            }
            if (snap) {
                const auto &b = *afresh(pa);
                float *const keep[2] = {b.vxp1, b.vyp1};
                res_snap_encode<2, R>(b, s, 0, ks, e, c, i, j, r0, bx, keep, maxima);
            }
        }

        // ================= stresses
        if (!receive<N>(ra, in + ra.words, sides, nt, lds, oVX, W, oVY, W, oVY, W, oVX, W)) s_stop = 2 * nt + 1;
        __syncthreads();
        if (s_stop && s_stop <= 2 * nt + 1) return;
        {
            float vxx[R], vyx[R], vxy[R], vyy[R];
            {
                const float *X = VX + r0 * W + tx, *Y = VY + r0 * W + tx;
                float cx[2 * N + R - 1], cy[2 * N + R - 1];  // cx[k]: vx row k-N+1; cy[k]: vy row k-N
#pragma unroll
                for (int k = 0; k < 2 * N + R - 1; k++) {
                    cx[k] = X[(k - N + 1) * W];
                    cy[k] = Y[(k - N) * W];
                }
#pragma unroll
                for (int r = 0; r < R; r++) {
                    __builtin_amdgcn_sched_barrier(0);
                    const float *vx = X + r * W, *vy = Y + r * W;
                    vxx[r] = hc[1] * (cx[N - 1 + r] - vx[-1]);
                    vyx[r] = hc[1] * (vy[1] - cy[N + r]);
                    vxy[r] = hc[1] * (cx[N + r] - cx[N - 1 + r]);
                    vyy[r] = hc[1] * (cy[N + r] - cy[N + r - 1]);
#pragma unroll
                    for (int m = 2; m <= N; m++) {
                        vxx[r] = vxx[r] + hc[m] * (vx[m - 1] - vx[-m]);
                        vyx[r] = vyx[r] + hc[m] * (vy[m] - vy[1 - m]);
                        vxy[r] = vxy[r] + hc[m] * (cx[N - 1 + r + m] - cx[N + r - m]);
                        vyy[r] = vyy[r] + hc[m] * (cy[N + r + m - 1] - cy[N + r - m]);
                    }
                    vxx[r] = vxx[r] * scale;
                    vyx[r] = vyx[r] * scale;
                    vxy[r] = vxy[r] * scale;
                    vyy[r] = vyy[r] * scale;
                }
            }
            if (hx >= 0) {
                const auto &b = *afresh(pa);
                const auto p1 = gmem(b.psi_vxx) + (long)s * b.pss, p2 = gmem(b.psi_vyx) + (long)s * b.pss;
                const unsigned o = afresh(hp), px = b.g.px;
                float v1[R], v2[R];
#pragma unroll
                for (int r = 0; r < R; r++)
                    if (live[r]) v1[r] = at(p1, (o + r * px) * 4u), v2[r] = at(p2, (o + r * px) * 4u);
#pragma unroll
                for (int r = 0; r < R; r++)
                    if (live[r]) {
                        v1[r] = bxp * v1[r] + ax * vxx[r];
                        vxx[r] = (K_one ? vxx[r] : vxx[r] / Kx) + v1[r];
                        v2[r] = bxh * v2[r] + axh * vyx[r];
                        vyx[r] = (K_one ? vyx[r] : vyx[r] / Kxh) + v2[r];
                        at(p1, (o + r * px) * 4u) = v1[r];
                        at(p2, (o + r * px) * 4u) = v2[r];
                    }
            }
#pragma unroll
            for (int r = 0; r < R; r++) {
                const int h = strip_y(j + r);
                if (h >= 0 && i <= NX) {
                    const auto &b = *afresh(pa);
                    const auto &pm = b.g.pml;
                    const unsigned o = afresh((unsigned)(i - 1) * 4u);
                    const auto p1 = gmem(b.psi_vyy) + (long)s * b.pss + (long)h * b.g.py;
                    const auto p2 = gmem(b.psi_vxy) + (long)s * b.pss + (long)h * b.g.py;
                    const float v1 = cmem(pm.b_y)[h] * at(p1, o) + cmem(pm.a_y)[h] * vyy[r];
                    const float v2 = cmem(pm.b_yh)[h] * at(p2, o) + cmem(pm.a_yh)[h] * vxy[r];
                    vyy[r] = divK(vyy[r], pm.K_y, h, K_one) + v1;
                    vxy[r] = divK(vxy[r], pm.K_yh, h, K_one) + v2;
                    at(p1, o) = v1;
                    at(p2, o) = v2;
                }
            }
#pragma unroll
            for (int r = 0; r < R; r++) {
                __builtin_amdgcn_sched_barrier(0);
                const int o = (r0 + r) * W + tx, oy = (r0 + r) * kTileX + tx;
                float sxx = SXX[o], syy = SYY[oy], sxy = SXY[o];
                float ux = 0.0f, uy = 0.0f, uxy = 0.0f;
                ViscCell vc;
                if (L == 0) {
                    if (rates) rates_elastic(m0[r], m1[r], m2[r], DT, vxx[r], vyx[r], vxy[r], vyy[r], ux, uy, uxy);
                    stress_elastic(m0[r], m1[r], m2[r], vxx[r], vyx[r], vxy[r], vyy[r], sxx, syy, sxy);
                } else {
                    // opaque, so that the products formed from them stay out of
                    // the registers between steps
                    asm volatile("" : "+v"(m0[r]), "+v"(m1[r]), "+v"(m2[r]), "+v"(m3[r]), "+v"(m4[r]), "+v"(m5[r]));
                    visc_coeffs(L, DT, m0[r], m1[r], m2[r], m3[r], m4[r], m5[r], vc);
                    stress_visc<L1>(vc, eta, bip, bjm, cip, cjm, DT, vxx[r], vyx[r], vxy[r], vyy[r], sxx,
                                    syy, sxy, rr[r], pp[r], qq[r], rates, ux, uy, uxy);
                }
                if (explosive && pi[r] >= 0) {
                    const auto &b = *afresh(pa);
                    for (int l = pi[r]; l >= 0; l = gmem(b.exp.next)[l]) {
                        const float amp = explosive_amp(b.exp.sig + (long)l * NT - 1, nt, NT, DH);
                        sxx = add_half(sxx, amp);
                        syy = add_half(syy, amp);
                    }
                }
                const int jr = j + r;  // row of the grid
                if (fs && by == 0 && jr <= N + 1) {
                    // free surface: the mirrored rows above, and row 1 itself
                    if (jr >= 2) SYY[(2 - jr - 1) * kTileX + tx] = live[r] ? -syy : 0.0f;
                    if (jr <= N) SXY[(1 - jr - 1) * W + tx] = live[r] ? -sxy : 0.0f;
                    if (jr == 1) {
                        syy = 0.0f;
                        if (rates) uy = 0.0f;
                        if (L) {
#pragma unroll
                            for (int l = 0; l < L1; l++) qq[r][l] = 0.0f;
                        }
                        float dx = 0.0f, dy = 0.0f;
                        const float *vx = VX + o, *vy = VY + o;
#pragma unroll
                        for (int m = 1; m <= N; m++) {
                            dx += hc[m] * (vx[m - 1] - vx[-m]);
                            dy += hc[m] * (vy[(m - 1) * W] - vy[-m * W]);
                        }
                        const float dh24 = 1.0 / (double)DH;
                        dx *= dh24;
                        dy *= dh24;
                        if (hx >= 0) {
                            const auto &b = *afresh(pa);
                            const auto ps = gmem(b.psi_vxxs) + (long)s * b.pss + (unsigned)hx;
                            const float v = bxp * *ps + ax * dx;
                            dx = (K_one ? dx : dx / Kx) + v;
                            *ps = v;
                        }
                        if (L == 0)
                            surface_elastic_update((float)((double)m0[r] * 2.0), m1[r], DT, dx, dy, sxx, rates, ux);
                        else
                            surface_visc_update<L1>(vc.mu, vc.pi, vc.taus, vc.taup, eta, DT, dx, dy, sxx, pp[r],
                                                    rates, ux);
                    }
                }
                if (!live[r]) sxx = syy = sxy = 0.0f;
                SXX[o] = sxx;
                SYY[oy] = syy;
                SXY[o] = sxy;
                send_y<N>(ra, sides, up, dn, r0 + r, (int)afresh(tx), syy, sxy, nt);
                send_x<N>(ra, xd, r, sxx, sxy, nt);
                if (snap) {
                    const auto &b = *afresh(pa);
                    const float u[3] = {vel ? ux : sxx, vel ? uy : syy, vel ? uxy : sxy};
                    float *const keep[3] = {b.ux, b.uy, b.uxy};
                    res_snap_put<3>(b, s, 2, ks, afresh(e) + r * NX, afresh(c) + r * P, live[r], r0 + r, u, keep,
                                    maxima + 2 * th);
                }
                if (pr[r] >= 0) {
                    const auto &b = *afresh(pa);
                    for (int l = pr[r]; l >= 0; l = gmem(b.rec.next)[l]) {
                        gmem(b.seis_vx)[(long)l * NT + nt - 1] = VX[o];
                        gmem(b.seis_vy)[(long)l * NT + nt - 1] = VY[o];
                    }
                }
                if (jr == NY / 2 && i == NX / 2) {
                    const auto nf = gmem(afresh(pa)->nan_flag);
                    if (nf && isnan(VY[o]) && *nf == 0) *nf = nt;
                }
            }
            if (snap) {
                const auto &b = *afresh(pa);
                float *const keep[3] = {b.ux, b.uy, b.uxy};
                res_snap_encode<3, R>(b, s, 2, ks, e, c, i, j, r0, bx, keep, maxima + 2 * th);
            }
            if (corr) {
#pragma unroll 1
                for (int r = 0; r < R; r++) {
                    if (i > NX || j + r > NY) break;
                    const auto &b = *afresh(pa);
                    const int o = (r0 + r) * W + tx, oy = (r0 + r) * kTileX + tx;
                    const unsigned cr = (afresh(c) + r * P) * 4u, ei = afresh(e) + r * NX, er = ei * 4u;
                    const int blk = (j + r - 1) / kTileY * b.nbx + bx;
                    const long wco = (long)s * b.wcs, wo = (long)s * b.ws;
                    const auto Wr = gmem(b.wc_rho) + wco, Wl = gmem(b.wc) + wco, Wu = gmem(b.wc_u) + wco;
                    float wr = at(Wr, er), w = at(Wl, er), wu = at(Wu, er);
                    correlate_cell(at(gmem(b.vxp1) + wo, cr), at(gmem(b.vyp1) + wo, cr), SXX[o], SYY[oy], SXY[o],
                                   res_snap_load(b, s, 0, ks, ei, blk), res_snap_load(b, s, 1, ks, ei, blk),
                                   res_snap_load(b, s, 2, ks, ei, blk), res_snap_load(b, s, 3, ks, ei, blk),
                                   res_snap_load(b, s, 4, ks, ei, blk), at(gmem(b.muss), er), at(gmem(b.lamss), er),
                                   at(gmem(b.vs_i), er) > 0.0f, wr, w, wu);
                    at(Wr, er) = wr;
                    at(Wl, er) = w;
                    at(Wu, er) = wu;
                }
            }
        }
    }

    // ---- the final wavefields, where the two-kernel step keeps them
#pragma unroll
    for (int r = 0; r < R; r++)
        if (live[r]) {
            const int o = (r0 + r) * W + tx;
            const long wo = (long)s * a.ws;
            const unsigned cr = c + r * P;
            at(gmem(a.vx) + wo, cr * 4u) = VX[o];
            at(gmem(a.vy) + wo, cr * 4u) = VY[o];
            at(gmem(a.sxx) + wo, cr * 4u) = SXX[o];
            at(gmem(a.syy) + wo, cr * 4u) = SYY[(r0 + r) * kTileX + tx];
            at(gmem(a.sxy) + wo, cr * 4u) = SXY[o];
        }
}

// LDS bytes of a tile (host)
template <int N>
size_t resident_lds(int th)
{
    return sizeof(float) * (size_t)ResLds<N>::total(th);
}

template <int N, int L, int R>
static hipError_t resident_launch(const ResidentArgs &r, const ResidentPlan &p, hipStream_t s)
{
    const hipError_t e = hipFuncSetAttribute((const void *)&k_resident<N, L, R>,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)p.lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((k_resident<N, L, R>), dim3(8 * r.per), dim3(kTileX, p.ty), p.lds, s, r);
    return hipGetLastError();
}

template <int N, int L, int R = 1>
static hipError_t resident_rows(const ResidentArgs &r, const ResidentPlan &p, hipStream_t s)
{
    if (p.rows == R) return resident_launch<N, L, R>(r, p, s);
    if constexpr (R < resident_max_rows(L)) return resident_rows<N, L, R + 1>(r, p, s);
    return hipErrorInvalidValue;
}

template <int N>
hipError_t resident_n(int L, const ResidentArgs &r, const ResidentPlan &p, hipStream_t s)
{
    switch (L) {
    case 0: return resident_rows<N, 0>(r, p, s);
    case 1: return resident_rows<N, 1>(r, p, s);
    case 2: return resident_rows<N, 2>(r, p, s);
    case 3: return resident_rows<N, 3>(r, p, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace ifos
