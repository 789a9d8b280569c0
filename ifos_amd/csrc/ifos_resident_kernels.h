// ifos_resident_kernels.h -- the time loop as one launch (ifos_resident.h).
// The arithmetic is that of ifos_cellmath.h, operand for operand, so the
// results are the bits of the two-kernel step.
#pragma once
#include <type_traits>

#include "ifos_resident.h"
#include "ifos_stepdev.h"

namespace ifos {

// Offsets of the LDS arrays of a tile, in floats, for the highest tile of R rows
// per thread (compile-time, so that one address register serves several arrays
// through the instructions' offsets).  Row r, column x of the tile (0-based) sit
// at vx, vy, sxy: (r + N) * W + x + N; sxx (no rows above and below): r * W + x +
// N; syy (no columns to the sides): (r + N) * 64 + x.
template <int N, int R>
struct ResLds {
    static constexpr int W = kTileX + 2 * N, TH = kResidentThreads / kTileX * R, H = TH + 2 * N;
    static constexpr int vx = 0, vy = H * W, sxy = 2 * H * W, sxx = 3 * H * W, syy = 3 * H * W + TH * W;
    static constexpr int maxima = syy + H * kTileX;  // of 16-bit snapshots, 5 per row
    // CPML profiles of the columns (6 floats, then 2 doubles, [.][64]) and of
    // the rows ([row] of 6 floats and 2 doubles), moduli of the surface row
    static constexpr int xprof = (maxima + 5 * TH + 1) / 2 * 2, yprof = xprof + 10 * kTileX;
    static constexpr int surface = yprof + 10 * TH;
    static constexpr int planes = surface + 4 * kTileX;  // per-cell coefficients outside registers, [plane][row][64]
    static constexpr int plane = TH * kTileX;
    // the FP64 reciprocals of the profiles are read as whole doubles
    static_assert(xprof % 2 == 0 && yprof % 2 == 0, "FP64 profile values at odd floats");
};

// Coefficients of a cell: 2 d, e, dip per mechanism, 2 f, g, fipjp (the latter
// three alone when elastic), DT times the two buoyancies.
constexpr int coefficients(int L) { return 3 * L + 5; }

// How many of them, the first in that order, sit in LDS instead of registers.
// With several rows per thread as many as fit beside the largest tile (with all
// of them in registers 36 values of every thread spilled to scratch on 1024x512,
// L=2, FDORDER 8, and a step took 13.0 us instead of 10.6, 9.7 since the array is
// aligned).  With one row only where the registers would spill: L=2, FDORDER 12,
// 1024x256 7.9 / 7.0 us a step, FDORDER 8, 1024x128 5.0 / 4.8, L=3, FDORDER 8, 1024x256
// 5.8 / 5.5, FDORDER 4 5.3 / 5.1; L=2, FDORDER 4 does not spill and a gradient's pair
// of steps of 301x151 went from 8.7 to 8.8.
template <int N, int L, int R>
constexpr int lds_coefficients()
{
    if (R == 1) return N >= 4 && L >= 2 ? 3 * L + 3 : L >= 3 ? 3 * L : 0;
    const int n = ((163840 - 256) / 4 - ResLds<N, R>::planes) / ResLds<N, R>::plane;
    return n < 0 ? 0 : n < coefficients(L) ? n : coefficients(L);
}

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
__device__ __forceinline__ int afresh_uniform(int v)
{
    asm volatile("" : "+s"(v));
    return v;
}
__device__ __forceinline__ float afresh(float v)
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
__device__ __forceinline__ void send_y(const ResidentArgs &ra, int sides, unsigned up, unsigned dn, int r, int tx,
                                       float p, float q, int tag)
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
__device__ __forceinline__ void send_x(const ResidentArgs &ra, const XDest &d, unsigned half, int r, float p, float q,
                                       int tag)
{
    if (d.p >= 0) send_word(ra.inbox, afresh((unsigned)d.p) + half + r * (2 * N - 1), p, tag);
    if (d.q >= 0) send_word(ra.inbox, afresh((unsigned)d.q) + half + r * (2 * N - 1), q, tag);
}

// Where inbox word q of a tile goes, as the LDS offset of its cell for the
// half step whose fields are given by their offsets of row 0, column 0 and
// row strides (py, qy from below and above, px, qx from the sides); side: the
// neighbour it comes from.
template <int N>
__device__ __forceinline__ int word_cell(int q, int th, int py, int spy, int qy, int sqy, int px, int spx, int qx,
                                         int sqx, int &side)
{
    constexpr int M = 2 * N - 1;
    if (q < 2 * M * kTileX) {
        const bool above = q >= M * kTileX;
        const int k = above ? q - M * kTileX : q, l = k / kTileX, x = k % kTileX;
        side = above ? kAbove : kBelow;
        if (!above) return l < N ? py + (th + l) * spy + x : qy + (th + l - N) * sqy + x;
        return l < N - 1 ? py + (l - (N - 1)) * spy + x : qy + (l - (N - 1) - N) * sqy + x;
    }
    const int h = q - 2 * M * kTileX;
    const bool left = h >= M * th;
    const int k = left ? h - M * th : h, r = k / M, l = k % M;
    side = left ? kLeft : kRight;
    if (!left) return l < N ? px + r * spx + kTileX + l : qx + r * sqx + kTileX + l - N;
    return l < N - 1 ? px + r * spx + l - (N - 1) : qx + r * sqx + l - (N - 1) - N;
}

// inbox words per thread: resident_plan keeps one-row tiles high enough for
// three; of the others the lowest have the most (16 rows of R - 1 cells did not
// hold them)
template <int N, int R>
constexpr int words_per_thread()
{
    const int ty = 16 * (R - 1) / R + 1;
    return R == 1 ? kWordsPerThread : ((2 * N - 1) * 2 * (kTileX + R * ty) + kTileX * ty - 1) / (kTileX * ty);
}

// CPML profile values of a column or row, with the reciprocals for div_by
struct Profile {
    float K, a, b, Kh, ah, bh;
    double rK, rKh;
};

// two derivatives through an absorbing strip: new memory values m and n, then
// d / K + m.  (Where every K is 1 the division returns d.)
__device__ __forceinline__ void absorb(float &d, float &m, float Kd, double rd, float ad, float bd, float &f, float &n,
                                       float Kf, double rf, float af, float bf)
{
    m = bd * m + ad * d;
    n = bf * n + af * f;
    div_by2(d, f, Kd, Kf, rd, rf);
    d = d + m;
    f = f + n;
}

// Take a half step's halo out of the inbox into LDS.  Thread t polls words t,
// t + threads, ...; cell[u] holds the LDS offset of its u-th word in the low
// (SHIFT 0) or high (SHIFT 16) half, on its set of words that come.  A word
// whose tag matches carries its value.  false: a neighbour did not answer
// within ra.limit, or another workgroup gave up.
template <int U, int SHIFT>
__device__ __forceinline__ bool receive(const ResidentArgs &ra, const unsigned long long *in_, int tag, float *lds,
                                        unsigned first, unsigned step, const unsigned (&cell)[U])
{
    const auto in = gmem(in_);
    unsigned long long since = 0;
    int tries = 0;
    unsigned long long w[U];
    for (;;) {
        bool ready = true;
#pragma unroll
        for (int u = 0; u < U; u++)
            if (cell[u]) w[u] = __hip_atomic_load(&at(in, afresh(first) + u * step), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int u = 0; u < U; u++)
            if (cell[u]) ready &= (int)(w[u] >> 32) == tag;
        if (ready) break;
        if ((++tries & 63) == 0 || ra.limit == 0) {
            const unsigned long long now = wall_clock64();
            if (since == 0) since = now;
            if (now - since >= ra.limit) {
                __hip_atomic_store(gmem(ra.stop), 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                return false;
            }
            if (__hip_atomic_load(gmem(ra.stop), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return false;
        }
    }
#pragma unroll
    for (int u = 0; u < U; u++)
        if (cell[u]) lds[(cell[u] >> SHIFT) & 0xFFFFu] = __uint_as_float((unsigned)w[u]);
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
    using D = ResLds<N, R>;
    constexpr int W = D::W, M = 2 * N - 1, L1 = L > 0 ? L : 1;
    const ArgPtr pa = cmem(ra.a);
    const auto &a = *pa;
    const auto &g = a.g;
    // aligned for the profiles' doubles: the array begins behind s_stop (at byte 4 a
    // shot gradient of 1700x350, L=2 took 62.6 ms instead of 58.1)
    extern __shared__ __attribute__((aligned(16))) float lds[];
    __shared__ int s_stop;  // half step in which a thread of this workgroup gave up, 0: none
    const int wg = (int)(blockIdx.x % 8) * ra.per + (int)blockIdx.x / 8;
    if ((int)blockIdx.x / 8 >= ra.per || wg >= ra.nwg) return;
    const int th = ra.th, tx = threadIdx.x, ty = __builtin_amdgcn_readfirstlane(threadIdx.y);
    const int s = wg / ra.ntile, t = wg - s * ra.ntile, by = t / a.nbx, bx = t - by * a.nbx;
    const int NX = g.NX, NY = g.NY, P = g.pitch;
    const int i = bx * kTileX + tx + 1, j0 = by * th, r0 = ty * R, j = j0 + r0 + 1;  // first row of this thread
    const unsigned c = (unsigned)(j * P + i), e = (unsigned)((j - 1) * NX + (i - 1));  // first cell of this thread
    bool live[R];
#pragma unroll
    for (int r = 0; r < R; r++) live[r] = i <= NX && j + r <= NY;

    // ---- the fields in LDS, all zero (what lies outside the grid stays so)
    for (int q = ty * kTileX + tx; q < D::maxima; q += kTileX * ra.ty) lds[q] = 0.0f;
    if (tx == 0 && ty == 0) s_stop = 0;
    // offsets of row 0, column 0
    constexpr int oVX = D::vx + N * W + N, oVY = D::vy + N * W + N, oSXY = D::sxy + N * W + N;
    constexpr int oSXX = D::sxx + N, oSYY = D::syy + N * kTileX;
    float *const VX = lds + oVX, *const VY = lds + oVY, *const SXY = lds + oSXY, *const SXX = lds + oSXX;
    float *const SYY = lds + oSYY, *const maxima = lds + D::maxima;

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

    // ---- this thread's words of the inbox: LDS offsets for the stresses (low
    // half) and the velocities (high half), 0: none
    constexpr int U = words_per_thread<N, R>();
    unsigned cell[U];
    const unsigned word0 = (unsigned)(ty * kTileX + tx), wstep = (unsigned)(kTileX * ra.ty);
#pragma unroll
    for (int u = 0; u < U; u++) {
        const int q = (int)(word0 + u * wstep);
        cell[u] = 0;
        if (q < ra.words) {
            int side;
            const unsigned cs = word_cell<N>(q, th, oSYY, kTileX, oSXY, W, oSXX, W, oSXY, W, side);
            const unsigned cv = word_cell<N>(q, th, oVX, W, oVY, W, oVY, W, oVX, W, side);
            if (sides & side) cell[u] = cs | cv << 16;
        }
    }

    // ---- materials and memory variables.  Up to one row per thread the
    // buoyancies stay beside their products with DT; else they are read again
    // where they are needed (snapshots, point forces).
    constexpr bool kOne = R == 1;
    float ripk = 0.0f, rjpk = 0.0f;
    constexpr int NC = coefficients(L), NP = lds_coefficients<N, L, R>(), NR = NC > NP ? NC - NP : 1;
    constexpr int cF2 = 3 * L, cG = 3 * L + 1, cFip = 3 * L + 2, cDtx = 3 * L + 3, cDty = 3 * L + 4;
    float creg[R][NR];
    float *const clds = lds + D::planes + r0 * kTileX + tx;
    auto coef = [&](int r, int k) -> float {
        if (k < NP) return clds[k * D::plane + r * kTileX];
        return creg[r][k - NP];
    };
    auto set_coef = [&](int r, int k, float v) {
        if (k < NP) clds[k * D::plane + r * kTileX] = v;
        else creg[r][k - NP] = v;
    };
    float rr[R][L1], pp[R][L1], qq[R][L1];
    float eta[L1 + 1], bip[L1 + 1], bjm[L1 + 1], cip[L1 + 1], cjm[L1 + 1], hc[N + 1];
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
#pragma unroll
    for (int r = 0; r < R; r++) {
        const unsigned ci = material_cell(c, r, P, live[r]) * 4u;
        const float bx_ = at(gmem(a.rip), ci), by_ = at(gmem(a.rjp), ci);
        if (r == 0) ripk = bx_, rjpk = by_;
        set_coef(r, cDtx, g.DT * bx_);
        set_coef(r, cDty, g.DT * by_);
        if (L == 0) {
            set_coef(r, cF2, 2.0f * at(gmem(a.f), ci));
            set_coef(r, cG, at(gmem(a.gl), ci));
            set_coef(r, cFip, at(gmem(a.uipjp), ci));
        } else {
            ViscCell vc;
            visc_coeffs(L, g.DT, at(gmem(a.mu), ci), at(gmem(a.pi), ci), at(gmem(a.muipjp), ci),
                        at(gmem(a.taus), ci), at(gmem(a.taup), ci), at(gmem(a.tausipjp), ci), vc);
            ViscUpdate<L1> v;
            visc_update(vc, eta, v);
#pragma unroll
            for (int l = 0; l < L; l++) {
                set_coef(r, 3 * l, v.d2[l]);
                set_coef(r, 3 * l + 1, v.e[l]);
                set_coef(r, 3 * l + 2, v.dip[l]);
            }
            set_coef(r, cF2, v.f2);
            set_coef(r, cG, v.g);
            set_coef(r, cFip, v.fipjp);
            if (r == 0 && ty == 0) {
                float *const sf = lds + D::surface + tx;
                sf[0] = vc.mu;
                sf[kTileX] = vc.pi;
                sf[2 * kTileX] = vc.taus;
                sf[3 * kTileX] = vc.taup;
            }
        }
#pragma unroll
        for (int l = 0; l < L1; l++) rr[r][l] = pp[r][l] = qq[r][l] = 0.0f;
    }
    auto buoyancies = [&](int r, float &x, float &y) {
        if constexpr (kOne) {
            x = ripk;
            y = rjpk;
        } else {
            const auto &b = *afresh(pa);
            const unsigned ci = material_cell(afresh(c), r, b.g.pitch, live[r]) * 4u;
            x = at(gmem(b.rip), ci);
            y = at(gmem(b.rjp), ci);
        }
    };

    // ---- CPML: strip positions of this column and of the rows, and their
    // profiles, in registers with one row per thread, else in LDS
    const int fw = g.FW, fs = g.FREE_SURF;
    auto strip = [&](int k, int n, bool low) {
        if (low && k <= fw) return k - 1;
        return k >= n - fw + 1 && k <= n ? k - n + 2 * fw - 1 : -1;
    };
    const int hx = strip(i, NX, true);
    unsigned yrows = 0;  // rows of this thread in a y strip (uniform in a wavefront)
#pragma unroll
    for (int r = 0; r < R; r++) yrows |= strip(j + r, NY, !fs) >= 0 ? 1u << r : 0u;
    const int ylow = fs ? 0 : fw, yshift = 2 * fw - NY;
    auto strip_row = [&](int jj) { return jj - 1 + (jj > ylow ? yshift : 0); };
    const bool inx = hx >= 0;
    Profile xp = {1.0f, 0.0f, 0.0f, 1.0f, 0.0f, 0.0f, 1.0, 1.0}, yp = xp;
    auto profile = [](int h, const float *K, const float *a_, const float *b, const float *Kh, const float *ah,
                      const float *bh) {
        Profile p = {gmem(K)[h], gmem(a_)[h], gmem(b)[h], gmem(Kh)[h], gmem(ah)[h], gmem(bh)[h], 0.0, 0.0};
        p.rK = 1.0 / (double)p.K;
        p.rKh = 1.0 / (double)p.Kh;
        return p;
    };
    if (inx) xp = profile(hx, g.pml.K_x, g.pml.a_x, g.pml.b_x, g.pml.K_xh, g.pml.a_xh, g.pml.b_xh);
    if (kOne && strip(j, NY, !fs) >= 0)
        yp = profile(strip(j, NY, !fs), g.pml.K_y, g.pml.a_y, g.pml.b_y, g.pml.K_yh, g.pml.a_yh, g.pml.b_yh);
    float *const xl = lds + D::xprof + tx, *const yl = lds + D::yprof;
    if (!kOne) {
        if (ty == 0) {
            xl[0] = xp.K; xl[kTileX] = xp.a; xl[2 * kTileX] = xp.b;
            xl[3 * kTileX] = xp.Kh; xl[4 * kTileX] = xp.ah; xl[5 * kTileX] = xp.bh;
            double *const xd2 = (double *)(lds + D::xprof + 6 * kTileX) + tx;
            xd2[0] = xp.rK;
            xd2[kTileX] = xp.rKh;
        }
        for (int r = ty * kTileX + tx; r < th; r += kTileX * ra.ty) {
            const int h = strip(j0 + r + 1, NY, !fs);
            Profile q = {1.0f, 0.0f, 0.0f, 1.0f, 0.0f, 0.0f, 1.0, 1.0};
            if (h >= 0) q = profile(h, g.pml.K_y, g.pml.a_y, g.pml.b_y, g.pml.K_yh, g.pml.a_yh, g.pml.b_yh);
            float *const y = yl + 10 * r;
            y[0] = q.K; y[1] = q.a; y[2] = q.b; y[3] = q.Kh; y[4] = q.ah; y[5] = q.bh;
            *(double *)(y + 6) = q.rK;
            *(double *)(y + 8) = q.rKh;
        }
    }
    auto column = [&]() {
        if constexpr (kOne) return xp;
        const double *const xd2 = (const double *)(lds + D::xprof + 6 * kTileX) + tx;
        return Profile{xl[0], xl[kTileX], xl[2 * kTileX], xl[3 * kTileX], xl[4 * kTileX], xl[5 * kTileX], xd2[0],
                       xd2[kTileX]};
    };
    auto row = [&](int r) {
        if constexpr (kOne) return yp;
        const float *const y = yl + 10 * (r0 + r);
        return Profile{y[0], y[1], y[2], y[3], y[4], y[5], *(const double *)(y + 6), *(const double *)(y + 8)};
    };
    // byte offsets of the first row's CPML memory
    const unsigned px4 = (unsigned)g.px * 4u, py4 = (unsigned)g.py * 4u;
    const unsigned ox = inx ? (unsigned)((j - 1) * g.px + hx) * 4u : 0u, oy = (unsigned)(min(i, NX) - 1) * 4u;
    const long po = (long)s * a.pss;

    // ---- points at these cells: rows with a source (adjoint: a receiver to
    // inject at) and rows with a receiver to record, as bits, and the first
    // point of the first such row; the others are looked up again
    unsigned inj_rows = 0, rec_rows = 0;
    int inj_first = -1, rec_first = -1;
#pragma unroll
    for (int r = R - 1; r >= 0; r--)
        if (live[r]) {
            const int l = gmem(a.inj.map)[(long)s * a.plane + (e + r * NX)];
            if (l >= 0) inj_rows |= 1u << r, inj_first = l;
            const int q = a.sw == 0 ? gmem(a.rec.map)[(long)s * a.plane + (e + r * NX)] : -1;
            if (q >= 0) rec_rows |= 1u << r, rec_first = q;
        }
    auto first_of = [&](unsigned rows, int first, const int *map, int r) {
        if ((rows & ((1u << r) - 1)) == 0) return (int)afresh((unsigned)first);
        return (int)gmem(map)[(long)s * pa->plane + (afresh(e) + r * NX)];
    };
    const bool fwd = a.sw == 0;
    const bool explosive = fwd && gmem(a.explosive)[s] != 0;
    const bool has_snaps = fwd && has_snap(a);
    const bool integ = !fwd && a.VELOCITY == 0, energy = a.wacc != nullptr, energy64 = a.wacc64 != nullptr;
    const int NT = a.NT, DTINV = a.DTINV, vel = a.VELOCITY;
    const float DT = g.DT, DH = g.DH, scale = L ? (float)(1.0 / (double)g.DH) : g.DT / g.DH;
    const double rDH = 1.0 / (double)DH;
    const float dthalbe = DT / 2.0;
    // adjoint: vxp1, vyp1 of the correlation; energies of the preconditioner
    float hvx[R], hvy[R], en[R];
#pragma unroll
    for (int r = 0; r < R; r++) hvx[r] = hvy[r] = en[r] = 0.0f;
    // steps until the next snapshot or correlation, and its slot
    int until = fwd ? 0 : DTINV - 1;
    long ks = fwd ? 0 : (long)NT / DTINV - 1;
    __syncthreads();

    for (int nt = 1; nt <= NT; nt++) {
        const bool mark = until == 0;
        const bool snap = mark && has_snaps, corr = mark && !fwd;
        const bool rates = snap && vel == 1;
        float q1 = 0.0f, q2 = 0.0f, q3 = 0.0f, q4 = 0.0f, n1 = 0.0f, n2 = 0.0f, n3 = 0.0f, n4 = 0.0f;

        // ================= velocities
        // loads that need no neighbour go ahead of the wait: the samples of a
        // point, with one row per thread the CPML memory
        const auto &bv = *afresh(pa);
        auto load_v = [&](int r) {
            const auto &b = bv;
            const unsigned kx = afresh(ox) + r * px4;
            if (inx && live[r]) n1 = at(gmem(b.psi_sxx_x) + po, kx), n2 = at(gmem(b.psi_sxy_x) + po, kx);
            if (!(yrows >> r & 1u)) return;
            const unsigned ky = afresh(oy) + strip_row(j + r) * py4;
            n3 = at(gmem(b.psi_syy_y) + po, ky), n4 = at(gmem(b.psi_sxy_y) + po, ky);
        };
        load_v(0);
        float s0 = 0.0f, s1 = 0.0f;
        if (inj_rows) {
            const long k = (long)(int)afresh((unsigned)inj_first) * NT + nt - 1;
            s0 = gmem(a.inj.sig)[k];
            s1 = gmem(a.inj.sig1)[k];
        }
        if (nt > 1 && !receive<U, 0>(ra, in, nt - 1, lds, word0 * 8u, wstep * 8u, cell)) s_stop = 2 * nt;
        __syncthreads();
        int stop = s_stop;
        {
            const float *S = SXY + r0 * W + tx, *Y = SYY + r0 * kTileX + tx, *X = SXX + r0 * W + tx;
            float cy[2 * N + R - 1], cs[2 * N + R - 1];  // cy[k]: sxy row k-N; cs[k]: syy row k-N+1
#pragma unroll
            for (int k = 0; k < 2 * N - 1; k++) {
                cy[k] = S[(k - N) * W];
                cs[k] = Y[(k - N + 1) * kTileX];
            }
#pragma unroll
            for (int r = 0; r < R; r++) {
                if (!kOne) __builtin_amdgcn_sched_barrier(0);
                q1 = n1, q2 = n2, q3 = n3, q4 = n4;
                if (r + 1 < R) load_v(r + 1);
                cy[2 * N - 1 + r] = S[(N - 1 + r) * W];
                cs[2 * N - 1 + r] = Y[(N + r) * kTileX];
                // one row per thread: every LDS value is on its way before the first is
                // used (more rows have no registers to spare for it)
                const int o = (r0 + r) * W + tx;
                float sx[2 * N], sy[2 * N];  // columns i-N+1 .. i+N and i-N .. i+N-1
#pragma unroll
                for (int k = 0; k < 2 * N; k++) {
                    sx[k] = X[r * W + k - N + 1];
                    sy[k] = k == N ? 0.0f : S[r * W + k - N];
                }
                const float vx0 = VX[o], vy0 = VY[o];
                if (kOne) __builtin_amdgcn_sched_barrier(0);
                if (r == 0 && stop && stop <= 2 * nt) return;
                sy[N] = cy[N + r];
                float sxx_x = hc[1] * (sx[N] - sx[N - 1]);
                float sxy_x = hc[1] * (sy[N] - sy[N - 1]);
                float sxy_y = hc[1] * (cy[N + r] - cy[N + r - 1]);
                float syy_y = hc[1] * (cs[N + r] - cs[N + r - 1]);
#pragma unroll
                for (int m = 2; m <= N; m++) {
                    sxx_x = sxx_x + hc[m] * (sx[N + m - 1] - sx[N - m]);
                    sxy_x = sxy_x + hc[m] * (sy[N + m - 1] - sy[N - m]);
                    sxy_y = sxy_y + hc[m] * (cy[N + r + m - 1] - cy[N + r - m]);
                    syy_y = syy_y + hc[m] * (cs[N + r + m - 1] - cs[N + r - m]);
                }
                if (inx && live[r]) {
                    const Profile x = column();
                    const unsigned kx = afresh(ox) + r * px4;
                    absorb(sxx_x, q1, x.Kh, x.rKh, x.ah, x.bh, sxy_x, q2, x.K, x.rK, x.a, x.b);
                    at(gmem(bv.psi_sxx_x) + po, kx) = q1;
                    at(gmem(bv.psi_sxy_x) + po, kx) = q2;
                }
                if ((yrows >> r & 1u) && i <= NX) {
                    const Profile y = row(r);
                    const unsigned ky = afresh(oy) + strip_row(j + r) * py4;
                    absorb(syy_y, q3, y.Kh, y.rKh, y.ah, y.bh, sxy_y, q4, y.K, y.rK, y.a, y.b);
                    at(gmem(bv.psi_syy_y) + po, ky) = q3;
                    at(gmem(bv.psi_sxy_y) + po, ky) = q4;
                }
                const float sumx = sxx_x + sxy_y, sumy = sxy_x + syy_y;
                float vx = coef(r, cDtx) * sumx, vy = coef(r, cDty) * sumy;  // vel_new
                div_by2(vx, vy, DH, DH, rDH, rDH);
                vx = vx0 + vx;
                vy = vy0 + vy;
                if (inj_rows >> r & 1u) {
                    const auto &b = *afresh(pa);
                    float rip, rjp;
                    buoyancies(r, rip, rjp);
                    int l = first_of(inj_rows, inj_first, b.inj.map, r);
                    if ((inj_rows & ((1u << r) - 1)) == 0) {
                        inject_values(b, l, s0, s1, rip, rjp, vx, vy);
                        l = gmem(b.inj.next)[l];
                    }
                    for (; l >= 0; l = gmem(b.inj.next)[l]) inject(b, l, nt, rip, rjp, vx, vy);
                }
                if (i > NX || (kOne ? j : afresh_uniform(j)) + r > NY) vx = vy = 0.0f;
                VX[o] = vx;
                VY[o] = vy;
                send_y<N>(ra, sides, up + ra.words, dn + ra.words, (kOne ? r0 : afresh_uniform(r0)) + r, (int)afresh((unsigned)tx), vx, vy, nt);
                send_x<N>(ra, xd, ra.words, r, vy, vx, nt);
                if (!fwd) {
                    if (integ) {
                        hvx[r] += vx0 * DT;
                        hvy[r] += vy0 * DT;
                    } else if (corr) {
                        hvx[r] = vx0;
                        hvy[r] = vy0;
                    }
                }
                if (energy) en[r] += ((vx * vx) + (vy * vy));
                if (snap) {
                    const auto &b = *afresh(pa);
                    float rip, rjp;
                    buoyancies(r, rip, rjp);
                    const float acc[2] = {vel_rate(rip, sumx, afresh(DH)), vel_rate(rjp, sumy, afresh(DH))};
                    float *const keep[2] = {b.vxp1, b.vyp1};
                    res_snap_put<2>(b, s, 0, ks, afresh(e) + r * NX, afresh(c) + r * P, live[r], r0 + r, acc, keep,
                                    maxima);
                }
                if (energy64 && live[r]) {
                    const auto &b = *afresh(pa);
                    const auto Wd = gmem(b.wacc64) + (long)s * b.wacs;
                    at(Wd, (afresh(e) + r * NX) * 8u) += ((double)vx * (double)vx) + ((double)vy * (double)vy);
                }
            }
            if (snap) {
                const auto &b = *afresh(pa);
                float *const keep[2] = {b.vxp1, b.vyp1};
                res_snap_encode<2, R>(b, s, 0, ks, afresh(e), afresh(c), i, j, r0, bx, keep, maxima);
            }
        }

        // ================= stresses
        const auto &bs = *afresh(pa);
        auto load_s = [&](int r) {
            const auto &b = bs;
            const unsigned kx = afresh(ox) + r * px4;
            if (inx && live[r]) n1 = at(gmem(b.psi_vxx) + po, kx), n2 = at(gmem(b.psi_vyx) + po, kx);
            if (!(yrows >> r & 1u)) return;
            const unsigned ky = afresh(oy) + strip_row(j + r) * py4;
            n3 = at(gmem(b.psi_vyy) + po, ky), n4 = at(gmem(b.psi_vxy) + po, ky);
        };
        load_s(0);
        float amp = 0.0f;
        if (explosive && inj_rows)
            amp = explosive_amp(a.exp.sig + (long)(int)afresh((unsigned)inj_first) * NT - 1, nt, NT, afresh(DH));
        if (!receive<U, 16>(ra, in + ra.words, nt, lds, word0 * 8u, wstep * 8u, cell)) s_stop = 2 * nt + 1;
        __syncthreads();
        stop = s_stop;
        {
            const float *X = VX + r0 * W + tx, *Y = VY + r0 * W + tx;
            float cx[2 * N + R - 1], cy[2 * N + R - 1];  // cx[k]: vx row k-N+1; cy[k]: vy row k-N
#pragma unroll
            for (int k = 0; k < 2 * N - 1; k++) {
                cx[k] = X[(k - N + 1) * W];
                cy[k] = Y[(k - N) * W];
            }
#pragma unroll
            for (int r = 0; r < R; r++) {
                if (!kOne) __builtin_amdgcn_sched_barrier(0);
                q1 = n1, q2 = n2, q3 = n3, q4 = n4;
                if (r + 1 < R) load_s(r + 1);
                cx[2 * N - 1 + r] = X[(N + r) * W];
                cy[2 * N - 1 + r] = Y[(N - 1 + r) * W];
                const int o = (r0 + r) * W + tx, oyy = (r0 + r) * kTileX + tx;
                float xv[2 * N], yv[2 * N];  // vx at columns i-N .. i+N-1, vy at i-N+1 .. i+N
#pragma unroll
                for (int k = 0; k < 2 * N; k++) {
                    xv[k] = k == N ? 0.0f : X[r * W + k - N];
                    yv[k] = k == N - 1 ? 0.0f : Y[r * W + k - N + 1];
                }
                float sxx = SXX[o], syy = SYY[oyy], sxy = SXY[o];
                if (kOne) __builtin_amdgcn_sched_barrier(0);
                if (r == 0 && stop && stop <= 2 * nt + 1) return;
                xv[N] = cx[N - 1 + r];
                yv[N - 1] = cy[N + r];
                float vxx = hc[1] * (xv[N] - xv[N - 1]);
                float vyx = hc[1] * (yv[N] - yv[N - 1]);
                float vxy = hc[1] * (cx[N + r] - cx[N - 1 + r]);
                float vyy = hc[1] * (cy[N + r] - cy[N + r - 1]);
#pragma unroll
                for (int m = 2; m <= N; m++) {
                    vxx = vxx + hc[m] * (xv[N + m - 1] - xv[N - m]);
                    vyx = vyx + hc[m] * (yv[N + m - 1] - yv[N - m]);
                    vxy = vxy + hc[m] * (cx[N - 1 + r + m] - cx[N + r - m]);
                    vyy = vyy + hc[m] * (cy[N + r + m - 1] - cy[N + r - m]);
                }
                vxx = vxx * scale;
                vyx = vyx * scale;
                vxy = vxy * scale;
                vyy = vyy * scale;
                if (inx && live[r]) {
                    const Profile x = column();
                    const unsigned kx = afresh(ox) + r * px4;
                    absorb(vxx, q1, x.K, x.rK, x.a, x.b, vyx, q2, x.Kh, x.rKh, x.ah, x.bh);
                    at(gmem(bs.psi_vxx) + po, kx) = q1;
                    at(gmem(bs.psi_vyx) + po, kx) = q2;
                }
                if ((yrows >> r & 1u) && i <= NX) {
                    const Profile y = row(r);
                    const unsigned ky = afresh(oy) + strip_row(j + r) * py4;
                    absorb(vyy, q3, y.K, y.rK, y.a, y.b, vxy, q4, y.Kh, y.rKh, y.ah, y.bh);
                    at(gmem(bs.psi_vyy) + po, ky) = q3;
                    at(gmem(bs.psi_vxy) + po, ky) = q4;
                }
                float ux = 0.0f, uy = 0.0f, uxy = 0.0f;
                if (L == 0) {
                    const float f2 = coef(r, cF2), gl = coef(r, cG), fip = coef(r, cFip);
                    if (rates)
                        rates_elastic(0.5f * afresh(f2), afresh(gl), afresh(fip), afresh(DT), vxx, vyx, vxy, vyy, ux,
                                      uy, uxy);
                    stress_elastic(f2, gl, fip, vxx, vyx, vxy, vyy, sxx, syy, sxy);
                } else {
                    ViscUpdate<L1> v;
                    v.f2 = coef(r, cF2);
                    v.g = coef(r, cG);
                    v.fipjp = coef(r, cFip);
                    if (!kOne) v.f2 = afresh(v.f2);  // its FP64 value need not stay in registers
#pragma unroll
                    for (int l = 0; l < L; l++) {
                        v.d2[l] = coef(r, 3 * l);
                        v.e[l] = coef(r, 3 * l + 1);
                        v.dip[l] = coef(r, 3 * l + 2);
                    }
                    stress_visc(v, bip, bjm, cip, cjm, dthalbe, afresh(DT), vxx, vyx, vxy, vyy, sxx, syy, sxy, rr[r],
                                pp[r], qq[r], rates, ux, uy, uxy);
                }
                if (explosive && (inj_rows >> r & 1u)) {
                    const auto &b = *afresh(pa);
                    int l = first_of(inj_rows, inj_first, b.inj.map, r);
                    float x = amp;
                    if (inj_rows & ((1u << r) - 1)) x = explosive_amp(b.exp.sig + (long)l * NT - 1, nt, NT, afresh(DH));
                    for (;;) {
                        sxx = add_half(sxx, x);
                        syy = add_half(syy, x);
                        l = gmem(b.exp.next)[l];
                        if (l < 0) break;
                        x = explosive_amp(b.exp.sig + (long)l * NT - 1, nt, NT, afresh(DH));
                    }
                }
                const int jr = (kOne ? j : afresh_uniform(j)) + r;  // row of the grid
                if (fs && by == 0 && jr <= N + 1) {
                    // free surface: the mirrored rows above, and row 1 itself
                    if (jr >= 2) SYY[(2 - jr - 1) * kTileX + tx] = live[r] ? -syy : 0.0f;
                    if (jr <= N) SXY[(1 - jr - 1) * W + tx] = live[r] ? -sxy : 0.0f;
                    if (r == 0 && jr == 1) {
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
                        const float dh24 = 1.0 / (double)afresh(DH);
                        dx *= dh24;
                        dy *= dh24;
                        if (inx) {
                            const auto &b = *afresh(pa);
                            const auto ps = gmem(b.psi_vxxs) + (long)s * b.pss + (unsigned)hx;
                            const Profile x = column();
                            float v = *ps;
                            v = x.b * v + x.a * dx;
                            dx = div_by(dx, x.K, x.rK) + v;
                            *ps = v;
                        }
                        if (L == 0) {
                            surface_elastic_update(afresh(coef(r, cF2)), afresh(coef(r, cG)), DT, dx, dy, sxx, rates, ux);
                        } else {
                            const float *const sf = lds + D::surface + tx;
                            surface_visc_update<L1>(sf[0], sf[kTileX], sf[2 * kTileX], sf[3 * kTileX], eta, DT, dx,
                                                    dy, sxx, pp[r], rates, ux);
                        }
                    }
                }
                if (i > NX || jr > NY) sxx = syy = sxy = 0.0f;
                SXX[o] = sxx;
                SYY[oyy] = syy;
                SXY[o] = sxy;
                send_y<N>(ra, sides, up, dn, (kOne ? r0 : afresh_uniform(r0)) + r, (int)afresh((unsigned)tx), syy, sxy, nt);
                send_x<N>(ra, xd, 0, r, sxx, sxy, nt);
                if (snap) {
                    const auto &b = *afresh(pa);
                    const float u[3] = {vel ? ux : sxx, vel ? uy : syy, vel ? uxy : sxy};
                    float *const keep[3] = {b.ux, b.uy, b.uxy};
                    res_snap_put<3>(b, s, 2, ks, afresh(e) + r * NX, afresh(c) + r * P, live[r], r0 + r, u, keep,
                                    maxima + 2 * th);
                }
                if (rec_rows >> r & 1u) {
                    const auto &b = *afresh(pa);
                    for (int l = first_of(rec_rows, rec_first, b.rec.map, r); l >= 0; l = gmem(b.rec.next)[l]) {
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
                res_snap_encode<3, R>(b, s, 2, ks, afresh(e), afresh(c), i, j, r0, bx, keep, maxima + 2 * th);
            }
            if (corr) {
#pragma unroll
                for (int r = 0; r < R; r++) {
                    if (!live[r]) break;
                    if (!kOne) __builtin_amdgcn_sched_barrier(0);
                    const auto &b = *afresh(pa);
                    const int o = (r0 + r) * W + tx, oyy = (r0 + r) * kTileX + tx;
                    const unsigned ei = afresh(e) + r * NX, er = ei * 4u;
                    const int blk = (j + r - 1) / kTileY * b.nbx + bx;
                    const long wco = (long)s * b.wcs;
                    const auto Wr = gmem(b.wc_rho) + wco, Wl = gmem(b.wc) + wco, Wu = gmem(b.wc_u) + wco;
                    float wr = at(Wr, er), w = at(Wl, er), wu = at(Wu, er);
                    correlate_cell(hvx[r], hvy[r], SXX[o], SYY[oyy], SXY[o], res_snap_load(b, s, 0, ks, ei, blk),
                                   res_snap_load(b, s, 1, ks, ei, blk), res_snap_load(b, s, 2, ks, ei, blk),
                                   res_snap_load(b, s, 3, ks, ei, blk), res_snap_load(b, s, 4, ks, ei, blk),
                                   at(gmem(b.muss), er), at(gmem(b.lamss), er), at(gmem(b.vs_i), er) > 0.0f, wr, w,
                                   wu);
                    at(Wr, er) = wr;
                    at(Wl, er) = w;
                    at(Wu, er) = wu;
                }
            }
        }
        if (mark) {
            until = DTINV;
            ks += fwd ? 1 : -1;
        }
        until--;
    }

    // ---- the final wavefields, where the two-kernel step keeps them, and the energies
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
            if (energy) at(gmem(a.wacc) + (long)s * a.wacs, (e + r * NX) * 4u) = en[r];
        }
}

// LDS bytes of a workgroup (host)
template <int N, int L, int R>
static size_t resident_lds_rows(int rows)
{
    typedef ResLds<N, R> D;
    static_assert(4 * D::planes + 256 <= 163840, "fields of the tallest tile exceed the LDS");
    if (rows == R) return sizeof(float) * (size_t)(D::planes + lds_coefficients<N, L, R>() * D::plane);
    if constexpr (R < resident_max_rows(N, L)) return resident_lds_rows<N, L, R + 1>(rows);
    return (size_t)-1;
}

template <int N>
size_t resident_lds(int L, int rows)
{
    switch (L) {
    case 0: return resident_lds_rows<N, 0, 1>(rows);
    case 1: return resident_lds_rows<N, 1, 1>(rows);
    case 2: return resident_lds_rows<N, 2, 1>(rows);
    case 3: return resident_lds_rows<N, 3, 1>(rows);
    default: return (size_t)-1;
    }
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
    if constexpr (R < resident_max_rows(N, L)) return resident_rows<N, L, R + 1>(r, p, s);
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
