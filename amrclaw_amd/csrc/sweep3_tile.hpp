// sweep3_tile.hpp -- the 3-D step fused over a block of cells, with every
// face on chip (FP32 storage and arithmetic).
//
// The phase kernels of sweep3.hpp reproduce step3.f's accumulation into the
// six flux arrays, which live in HBM.  Here one workgroup owns a tile of at
// most TILE3_MAX cells per direction of one grid and runs the x-, y- and
// z-sweeps and the update for it alone:
//   * the tile and two cells on every side (the cells the tile's lines read,
//     ghost cells of the grid where the tile reaches its edge) are staged in
//     LDS once;
//   * each sweep solves the lines through the tile and one line on every
//     side of it across the sweep (their transverse increments reach the
//     tile's cells), tr + 1 lanes per line, one lane per interface:
//     interfaces 0 .. tr of a tile with tr cells along the line (lanes 0
//     and tr also solve interfaces -1 and tr+1, whose waves the limiter
//     needs);
//   * instead of accumulating faces and differencing them afterwards, every
//     face contribution goes at once to the two cells it separates, in an
//     LDS array dq of the tile's cells: a face value F between cells a < b
//     enters the update as q(a) -= (dt/h) F, q(b) += (dt/h) F (stepgrid.f
//     (3-D):150-173 with fm = fp = F for the transverse increments of
//     step3.f:221-250, 279-310), the normal fluxes as
//     q(c) -= dt/h (faddm(c+1) - faddp(c));
//   * four waves solve at once, any lines, and those that add at the same time
//     touch no cell of each other (all four, or in small tiles two after the
//     other two), the lanes of a wave in ordered steps (tile3_rounds,
//     tile3_sweep): no atomics on dq, the sums are formed in a fixed order and
//     the result is deterministic.
// The per-interface arithmetic (rpn3, limiter, cqxx, the rpt3 / rptt3
// splits and their 1/2, 1/6 weights, flux3.f:220-628) is that of the phase
// kernel; only the order in which each cell's increments are summed differs
// from the reference, so the result agrees with it to FP32 rounding.  The
// step reads q from one buffer and writes the updated interiors into another,
// whose ghost cells a batch keeps equal to the first's and a level's step copies.
//
// Bound by vector issue (the SIMDs issue vector instructions in about 80 % of
// their cycles at 4 cycles each), so what counts is instructions per
// interface: the splits by wave strengths with the face weights in the speeds
// (Euler3::split_scaled), the method's switches at compile time, a cell's
// values together in LDS and scalar row bookkeeping took the Euler sweeps from
// 2300 to 1830 vector instructions an interface and 256 uneven grids
// (2,023,768 cells) from 984 to 700 us a step.  Full chunks from any rows, added
// in two phases, instead of waves of one row each in three classes of rows: 700
// -> 680 us, 6 grids 141 -> 134, the levels of a 64^3 run (tiles of 8 .. 11
// cells) 11.7 -> 10.2 ms.  One phase instead of two in the sweeps whose waves lie
// far enough apart: 512 grids of 16 .. 32 cells 1.31 -> 1.18 ms, 8 grids of 40^3
// 260 -> 234 us.
#pragma once
#include <cstdint>
#include "lanes.hpp"
#include "sweep3.hpp"
#include "tile3_rounds.hpp"

namespace amrgpu {

constexpr int TILE3_MAX = 15;        // cells per direction of a tile (15: lines of 16 lanes fill a wave)
constexpr int TILE3_LANES = 256;     // four waves
constexpr int TILE3_XCDS = 8;        // workgroups go to the XCDs in turn
constexpr int TILE3_WG_PER_CU = 2;   // workgroups a CU holds (LDS and registers sized for it)

// a tile: grid `patch`, 0-based first interior cell (i0, j0, k0), extents, and
// its marked faces marks[mark0 ..+ nmark)
struct Tile3 {
    int32_t patch;
    int16_t i0, j0, k0, tx, ty, tz, pad;
    int32_t mark0, nmark;
};

// A face of a tile whose flux the coarse-fine registers read (fluxsv.f,
// fluxad.f), in the tile's cells: the lower face, normal to dir (0 x, 1 y, 2
// z), of cell (x, y, z); along dir the cell may be one past the tile.
struct Mark3 {
    int16_t x, y, z, dir;
};

struct Tile3Args {
    const void* qin;                // solutions at time t (grid layout of Patch3)
    void* qout;                     // interiors at t + dt (ghost cells: see marks)
    const Patch3* patches;
    const Tile3* tiles;
    int32_t ntiles;
    int32_t nv;
    // the tiles of XCD x are tiles[xcd_start[x] ..+ xcd_count[x]]: workgroup
    // b runs on XCD b % 8 and takes its (b / 8)-th tile
    int32_t xcd_start[TILE3_XCDS], xcd_count[TILE3_XCDS];
    double dtd[3];                  // dt/dx, dt/dy, dt/dz
    Method3 meth;
    unsigned long long* cfl_patch;  // per-patch max Courant number (double bits)
    // a level's step (face null for a batch): the marked faces and the level's
    // flux blocks, of which only those faces are written (merged form, as the
    // phase kernels leave them); the ghost cells of qout receive qin's (a batch's
    // stay as they are)
    const Mark3* marks;
    float* face;
};

// Marked faces in LDS: for every face of the tile its mark's number + 1 (0:
// none), the x-faces first; per mark the transverse increments and faddm
// times dt/h, a sum for the waves of either phase, then faddp - faddm.
struct Mark3Lds {
    uint16_t* map;
    float* acc;
};
__host__ __device__ constexpr int mark3_faces(int tx, int ty, int tz) {
    return (tx + 1) * ty * tz + tx * (ty + 1) * tz + tx * ty * (tz + 1);
}
template <int NV>
__host__ __device__ constexpr size_t mark3_lds_bytes(int tx, int ty, int tz, int nmark) {
    return ((size_t)mark3_faces(tx, ty, tz) * 2 + 3) / 4 * 4 + (size_t)nmark * 3 * NV * sizeof(float);
}

// LDS of a tile workgroup: the staged box and the increments
template <int NV>
__host__ __device__ constexpr size_t tile3_lds_bytes(int bx, int by, int bz, int cells) {
    return ((size_t)NV * bx * by * bz + (size_t)NV * cells) * sizeof(float);
}

// Wave-synchronous ordering: the LDS accesses of one wave before this point
// are complete and visible to its other lanes after it (as __syncwarp).
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// idx = tid + TILE3_LANES i written as digits (x, y, z, m) of the radices
// (nx, ny, nz): stepped by TILE3_LANES with one carry per digit instead of
// three integer divisions per element (a digit plus its step plus a carry
// stays below twice its radix, so one subtraction brings it back)
struct Digits3 {
    int x, y, z, m, sx, sy, sz, sm, nx, ny, nz;
    __device__ __forceinline__ Digits3(int idx, int nx_, int ny_, int nz_) : nx(nx_), ny(ny_), nz(nz_) {
        int r = idx;
        x = r % nx; r /= nx; y = r % ny; r /= ny; z = r % nz; m = r / nz;
        r = TILE3_LANES;
        sx = r % nx; r /= nx; sy = r % ny; r /= ny; sz = r % nz; sm = r / nz;
    }
    __device__ __forceinline__ void step() {
        x += sx;
        int c = x >= nx;
        x -= c ? nx : 0;
        y += sy + c;
        c = y >= ny;
        y -= c ? ny : 0;
        z += sz + c;
        c = z >= nz;
        z -= c ? nz : 0;
        m += sm + c;
    }
};

__device__ __forceinline__ void lds_add(float* p, float v) {
    __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// one sweep of a tile (D: 1 x, 2 y, 3 z, a template parameter so that every
// component index of the solver is a compile-time constant).
//
// Schedule (tile3_rounds): the lines Q = -1 .. tq, P = -1 .. tp in one order, in
// which a wave takes chunks of up to lpw = 64 / (tr + 1) consecutive lines, from
// any rows, tr + 1 lanes per line.  The waves that add at the same time hold
// lines at least 2 n + 3 apart, so the cells these touch are disjoint: all waves
// of a round where the tile has lines enough, else those of a phase.  Within a
// wave the lines of a chunk touch common cells; each lane adds its increments to
// the nine cells (dQ, dP) around its own in ordered steps, in each of which the
// wave's lanes touch distinct cells.
//
// STD: the method is known to be the standard one (std_method3: second order,
// all transverse and double-transverse terms, MC limiter on every wave, no
// f-waves), so its switches are compile-time constants.
//
// MARK: increments to marked faces are also added to the faces' own sums, one
// for either phase, while the waves solve.  A wave's LDS additions happen in
// program order, each touching distinct faces; the waves of a phase touch
// distinct faces as they touch distinct cells, so these sums have a fixed order
// too.
template <class Sol, int D, bool STD, bool MARK>
__device__ __forceinline__ void tile3_sweep(const Tile3Args& a, float* qs, float* dq,
                                            int tx, int ty, int tz, int bx, int by, int wave,
                                            int wl, float& cfl, const Mark3Lds& mk) {
    using T = float;
    constexpr int NV = Sol::NV, NW = Sol::NW;
    constexpr int d = D;
    const Method3& M = a.meth;
    const bool trans = STD || M.m3 > 0, cq = STD || M.m3 >= 2, tt = STD || M.m4 > 0;
    const bool tt2 = STD || M.m4 == 2, second = STD || M.order != 1;
    bool limit = STD;
    for (int w = 0; w < NW; w++) limit = limit || M.mthlim[w] > 0;
    // axes (r, Q, P): x (x, y, z), y (y, x, z), z (z, x, y); LDS strides (a
    // cell's components lie together: NV is odd, so 64 cells in a row touch
    // 64 banks, and a cell's values are one base and constant offsets)
    const int sx = NV, sy = bx * NV, sz = bx * by * NV;
    const int tr = d == 1 ? tx : (d == 2 ? ty : tz);
    const int tq = d == 1 ? ty : tx;
    const int tp = d == 3 ? ty : tz;
    const int rs = d == 1 ? sx : (d == 2 ? sy : sz);
    const int qsd = d == 1 ? sy : sx;
    const int psd = d == 3 ? sy : sz;
    // dq strides (tile cells, x fastest)
    const int drs = NV * (d == 1 ? 1 : (d == 2 ? tx : tx * ty));
    const int dqs = NV * (d == 1 ? tx : 1);
    const int dps = NV * (d == 3 ? tx : tx * ty);
    const T dtdx = T(a.dtd[d - 1]);
    const T dtdy_p = T(a.dtd[d % 3]);
    const T dtdz_p = T(a.dtd[(d + 1) % 3]);
    const T dtQ = T(a.dtd[d == 1 ? 1 : 0]);     // across Q (type A faces)
    const T dtP = T(a.dtd[d == 3 ? 1 : 2]);     // across P (type B faces)
    const bool g_to_a = d != 2;
    // map indices of the faces across r, Q and P: base and strides of a cell's
    // lower face in each of the three face arrays
    const int nfx = (tx + 1) * ty * tz, nfy = tx * (ty + 1) * tz;
    auto fbase = [&](int ax) { return ax == 0 ? 0 : (ax == 1 ? nfx : nfx + nfy); };
    auto fstr = [&](int ax, int along) {
        const int w = tx + (ax == 0), h = ty + (ax == 1);
        return along == 0 ? 1 : (along == 1 ? w : w * h);
    };
    constexpr int AR = D - 1, AQ = D == 1 ? 1 : 0, AP = D == 3 ? 1 : 2;
    const T half_t = T(0.5) * dtdx;
    const T sixth = T(1) / T(6);
    const T g6 = sixth * dtdx * dtdz_p;   // weights of the double-transverse terms
    const T h6 = sixth * dtdx * dtdy_p;

    // a line's lanes take its interfaces 0 .. tr; the limiter's outer
    // neighbours (interfaces -1 and tr+1, waves only) are solved by lanes 0
    // and tr themselves
    const int L = tr + 1;                      // lanes of a line
    const int lpw = 64 / L;                    // lines of a chunk
    const int li = wl / L;                     // this lane's line in the chunk
    const int e = wl - li * L;                 // interface e: between cells e-1, e
    // the lines in order, the shorter of the two axes across them running
    // fastest; wave w takes chunks w R .. w R + R - 1, one a round
    const Tile3Rounds sch = tile3_rounds(tr, tq, tp);
    const bool qfast = tq <= tp;
    const int nfast = (qfast ? tq : tp) + 2, nlines = (tq + 2) * (tp + 2);
    const int inv = 65536 / nfast + 1;         // line / nfast = line * inv >> 16 (line < 300)
    const int phase = wave & 1;
#pragma unroll 1
    for (int rd = 0; rd < sch.rounds; rd++) {
        const int chunk = wave * sch.rounds + rd;
        const bool wlive = wave < sch.waves && chunk * lpw < nlines;   // (the whole wave)
        const int line0 = chunk * lpw + li;
        const bool live = wlive && li < lpw && line0 < nlines;
        const int line = live ? line0 : 0;
        const int slow = __mul24(line, inv) >> 16, fast = line - __mul24(slow, nfast);
        const int Q = (qfast ? fast : slow) - 1, P = (qfast ? slow : fast) - 1;
        const int ec = live ? e : 0;
        const bool own = live && e >= 1;   // completes a cell of the tile's length
        // lane e completes cell c = e-1 of the line (tile cells 0 .. t-1):
        // acc[(dQ+1) + 3 (dP+1)] collects its increments to cell
        // (c, Q+dQ, P+dP)
        T acc[9][NV];
        if (wlive) {
            // cells e-1 and e of the line (local -2 .. t+1)
            const int b0 = 2 * (sx + sy + sz) + __mul24(P, psd) + __mul24(Q, qsd) + __mul24(ec - 1, rs);
            T ql[NV], qrr[NV];
#pragma unroll
            for (int m = 0; m < NV; m++) {
                ql[m] = qs[b0 + m];
                qrr[m] = qs[b0 + rs + m];
            }
            const typename Sol::Cache cache = Sol::prep(M.ph, ql, qrr);
            T wave_[NW][NV], s[NW], amdq[NV], apdq[NV];
            Sol::rpn3(M.ph, d, ql, qrr, cache, wave_, s, amdq, apdq);
            // Courant number of interfaces 1 .. n+1 of every line
            // (ghost lines included), each counted by some tile
            if (live && e >= 0 && e <= tr) {
#pragma unroll
                for (int w = 0; w < NW; w++) cfl = dmax1(dmax1(cfl, dtdx * s[w]), -dtdx * s[w]);
            }
            T fadm[NV], fadp[NV], cqxx[NV];
#pragma unroll
            for (int m = 0; m < NV; m++) {
                fadm[m] = T(0) + amdq[m];
                fadp[m] = T(0) - apdq[m];
                cqxx[m] = T(0);
            }
            if (second) {
                if (limit) {   // inlinelimiter.f on unlimited neighbour waves
                    // w(e) . w(e+1) at lane e; the product with the wave
                    // before is the one of lane e-1
                    T dotr[NW], dotl[NW];
#pragma unroll
                    for (int w = 0; w < NW; w++) {
                        T x = T(0);
#pragma unroll
                        for (int m = 0; m < NV; m++) x = x + lane_down(wave_[w][m], L) * wave_[w][m];
                        dotr[w] = x;
                        dotl[w] = lane_up(x, L);
                    }
                    if (live && (e == 0 || e == tr)) {
                        // the outer neighbour of the line's end: interface -1
                        // (cells -2, -1) for lane 0, tr+1 (cells tr, tr+1) for
                        // lane tr (both when tr = 0 cannot happen: tr >= 1)
                        const int bx0 = e == 0 ? b0 - rs : b0 + rs;
                        T xl[NV], xr[NV];
#pragma unroll
                        for (int m = 0; m < NV; m++) {
                            xl[m] = qs[bx0 + m];
                            xr[m] = qs[bx0 + rs + m];
                        }
                        const typename Sol::Cache cx = Sol::prep(M.ph, xl, xr);
                        T wx[NW][NV], sx_[NW], amx[NV], apx[NV];
                        Sol::rpn3(M.ph, d, xl, xr, cx, wx, sx_, amx, apx);
#pragma unroll
                        for (int w = 0; w < NW; w++) {
                            T x = T(0);
#pragma unroll
                            for (int m = 0; m < NV; m++) x = x + wx[w][m] * wave_[w][m];
                            if (e == 0) dotl[w] = x;
                            else dotr[w] = x;
                        }
                    }
                    if (live && e >= 0 && e <= tr) {
#pragma unroll
                        for (int w = 0; w < NW; w++) {
                            const int mth = STD ? 4 : M.mthlim[w];
                            if (mth == 0) continue;
                            T wn2 = T(0);
#pragma unroll
                            for (int m = 0; m < NV; m++) wn2 = wn2 + wave_[w][m] * wave_[w][m];
                            if (wn2 == T(0)) continue;
                            using Mth = typename Sol::Math;
                            T rr = Mth::ratio(s[w] > T(0) ? dotl[w] : dotr[w], wn2);
                            T wlim = phi_limiter3<Mth>(mth, rr);
#pragma unroll
                            for (int m = 0; m < NV; m++) wave_[w][m] = wlim * wave_[w][m];
                        }
                    }
                }
                const T dtdxave = T(0.5) * (dtdx + dtdx);
#pragma unroll
                for (int m = 0; m < NV; m++) {
                    T c = T(0);
#pragma unroll
                    for (int w = 0; w < NW; w++) {
                        const T fac = !STD && M.use_fwaves ? (s[w] >= T(0) ? T(1) : T(-1)) : fabs(s[w]);
                        c = c + T(0.5) * fac * (T(1) - fabs(s[w]) * dtdxave) * wave_[w][m];
                    }
                    cqxx[m] = c;
                    fadm[m] = fadm[m] + c;
                    fadp[m] = fadp[m] + c;
                }
            }
#pragma unroll
            for (int k = 0; k < 9; k++)
#pragma unroll
                for (int m = 0; m < NV; m++) acc[k][m] = T(0);
            {
                // normal fluxes: q(c) -= dt/dx (faddm(c+1) - faddp(c))
#pragma unroll
                for (int m = 0; m < NV; m++) {
                    const T fpl = lane_up(fadp[m], L);
                    acc[4][m] = T(0) - dtdx * (fadm[m] - fpl);
                }
            }
            // adds v to the mark, if any, of the face at place i of the map
            auto mark_add = [&](int i, bool ok, const T* v) {
                const int id = ok ? mk.map[i] : 0;
                if (id) {
#pragma unroll
                    for (int m = 0; m < NV; m++) lds_add(&mk.acc[((id - 1) * 3 + phase) * NV + m], v[m]);
                }
                return id;
            };
            if constexpr (MARK) {
                T sc[NV];
#pragma unroll
                for (int m = 0; m < NV; m++) sc[m] = dtdx * fadm[m];
                const int at = fbase(AR) + __mul24(P, fstr(AR, AP)) + __mul24(Q, fstr(AR, AQ)) + __mul24(e, fstr(AR, AR));
                const int id = mark_add(at, live && Q >= 0 && Q < tq && P >= 0 && P < tp, sc);
                if (id) {
#pragma unroll
                    for (int m = 0; m < NV; m++)
                        mk.acc[((id - 1) * 3 + 2) * NV + m] = fadp[m] - fadm[m];
                }
            }
            // the lower faces across Q and across P of this lane's cell
            int atQ = 0, atP = 0;
            if constexpr (MARK) {
                atQ = fbase(AQ) + __mul24(P, fstr(AQ, AP)) + __mul24(Q, fstr(AQ, AQ)) + __mul24(e - 1, fstr(AQ, AR));
                atP = fbase(AP) + __mul24(P, fstr(AP, AP)) + __mul24(Q, fstr(AP, AQ)) + __mul24(e - 1, fstr(AP, AR));
            }
            if (trans) {
                // the splits both families use, once: of cqxx, A+dq and A-dq
                // along icoor 2 and 3 (index 0: 2, 1: 3; [0] down-, [1] up-going)
                T Cs[2][2][NV], As[2][2][NV], Ms[2][2][NV];
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    if (cq) Sol::split(M.ph, d, 2 + i, ql, qrr, cache, cqxx, Cs[i][0], Cs[i][1]);
                    Sol::split(M.ph, d, 2 + i, ql, qrr, cache, apdq, As[i][0], As[i][1]);
                    Sol::split(M.ph, d, 2 + i, ql, qrr, cache, amdq, Ms[i][0], Ms[i][1]);
                }
#pragma unroll
                for (int fam = 0; fam < 2; fam++) {
                    // fam 0 = gadd: primary split along icoor 2; fam 1 = hadd
                    const int ip = fam, is = 1 - fam;   // primary, secondary
                    const int icp = 2 + ip;
                    // slot (s, o) is the face Q+s-1 of cell row P+o (type
                    // A, across Q) or the face P+s-1 of cell row Q+o (type
                    // B, across P); a face enters the cells on its two sides
                    // with weight h, which all its terms carry from here on
                    const bool to_a = (fam == 0) == g_to_a;
                    const T h = to_a ? dtQ : dtP;
                    const T hw6 = h * (fam == 0 ? g6 : h6);
                    const T hh = h * half_t, hc = h * dtdx;
                    // The increments of cell e-1: right-cell partials of
                    // interface e-1 (they move one lane up) and left-cell
                    // increments of interface e, flux3.f:450-505.  Slot
                    // k = (s-1)*3 + (o+1).  r: cell e (A+dq side), v: cell
                    // e-1 (A-dq side); the correction enters them with
                    // opposite signs.
                    T v[6][NV], r[6][NV];
                    auto half = [&](T (&x)[6][NV], const T (&S)[2][2][NV], const T sg) {
#pragma unroll
                        for (int m = 0; m < NV; m++) {
                            x[1][m] = -hh * S[ip][0][m];
                            x[4][m] = -hh * S[ip][1][m];
                            if (cq) {
                                x[1][m] = x[1][m] + sg * hc * Cs[ip][0][m];
                                x[4][m] = x[4][m] + sg * hc * Cs[ip][1][m];
                            }
                        }
                        if (tt) {
                            // x[5], x[2] (o = +1) enter with a minus sign below
                            T tmp[NV];
#pragma unroll
                            for (int m = 0; m < NV; m++)
                                tmp[m] = tt2 ? S[is][1][m] - sg * T(3) * Cs[is][1][m] : S[is][1][m];
                            Sol::split_times(M.ph, d, icp, cache, hw6, tmp, x[2], x[5]);
#pragma unroll
                            for (int m = 0; m < NV; m++)
                                tmp[m] = tt2 ? S[is][0][m] - sg * T(3) * Cs[is][0][m] : S[is][0][m];
                            Sol::split_times(M.ph, d, icp, cache, hw6, tmp, x[0], x[3]);
#pragma unroll
                            for (int m = 0; m < NV; m++) {
                                x[4][m] = x[4][m] + (x[5][m] - x[3][m]);
                                x[1][m] = x[1][m] + (x[2][m] - x[0][m]);
                            }
                        }
                    };
                    half(r, As, T(1));
                    half(v, Ms, T(-1));
#pragma unroll
                    for (int o = -1; o <= 1; o++) {
                        if (o != 0 && !tt) continue;
#pragma unroll
                        for (int s2 = 1; s2 <= 2; s2++) {
                            const int k = (s2 - 1) * 3 + o + 1;
                            // lower cell (dQ, dP) and upper cell of the face
                            const int kl = to_a ? (s2 - 1) + 3 * (o + 1) : (o + 1) + 3 * (s2 - 1);
                            const int ku = to_a ? s2 + 3 * (o + 1) : (o + 1) + 3 * s2;
                            T ys[NV];
#pragma unroll
                            for (int m = 0; m < NV; m++) {
                                const T y = lane_up_add(r[k][m], v[k][m]);
                                acc[kl][m] = o == 1 ? acc[kl][m] + y : acc[kl][m] - y;
                                acc[ku][m] = o == 1 ? acc[ku][m] - y : acc[ku][m] + y;
                                ys[m] = o == 1 ? -y : y;
                            }
                            if constexpr (MARK) {
                                const int fQ = to_a ? Q + s2 - 1 : Q + o, fP = to_a ? P + o : P + s2 - 1;
                                const bool ok = own && fQ >= 0 && fQ < tq + (to_a ? 1 : 0) && fP >= 0 &&
                                                fP < tp + (to_a ? 0 : 1);
                                mark_add(to_a ? atQ + (s2 - 1) * fstr(AQ, AQ) + o * fstr(AQ, AP)
                                              : atP + (s2 - 1) * fstr(AP, AP) + o * fstr(AP, AQ),
                                         ok, ys);
                            }
                        }
                    }
                }
            }
        }
        // ordered steps: in each, the wave's lanes add to distinct cells (its lines
        // differ).  All waves add at once where they touch no cell of each other
        // (tile3_rounds), else first those of phase 0, then those of phase 1.
        auto add = [&] {
            const int c = e - 1;
            const int dbase = __mul24(P, dps) + __mul24(Q, dqs) + __mul24(c, drs);
            auto step = [&](const int k) {
                const int dQ = k % 3 - 1, dP = k / 3 - 1;
                const bool in = own && Q + dQ >= 0 && Q + dQ < tq && P + dP >= 0 && P + dP < tp;
                if (in) {
                    const int di = dbase + dQ * dqs + dP * dps;
#pragma unroll
                    for (int m = 0; m < NV; m++) {
                        T* x = &dq[di + m];
                        *x = *x + acc[k][m];
                    }
                }
                wave_sync();
            };
            if (!trans) {
                step(4);   // nothing goes past the line's own cells
                return;
            }
#pragma unroll
            for (int k = 0; k < 9; k++) step(k);
        };
        __syncthreads();   // the waves of the round before have added
        if (wlive && (phase == 0 || sch.phases == 1)) add();
        if (sch.phases == 2) {
            __syncthreads();
            if (wlive && phase == 1) add();
        }
    }
}

template <class Sol, bool STD, bool MARK>
__global__ __launch_bounds__(TILE3_LANES, TILE3_WG_PER_CU) void sweep3_tile_kernel(Tile3Args a) {
    using T = float;
    constexpr int NV = Sol::NV;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int xcd = blockIdx.x % TILE3_XCDS, k = blockIdx.x / TILE3_XCDS;
    if (k >= a.xcd_count[xcd]) return;   // (the whole workgroup: no barrier reached)
    const Tile3 td = a.tiles[a.xcd_start[xcd] + k];
    const Patch3 pt = a.patches[td.patch];
    const int tx = td.tx, ty = td.ty, tz = td.tz;
    const int bx = tx + 4, by = ty + 4, bz = tz + 4;
    const int nbox = bx * by * bz, ncell = tx * ty * tz;
    T* qs = reinterpret_cast<T*>(smem_raw);   // [bz][by][bx][NV], local -2 .. t+1
    T* dq = qs + NV * nbox;                   // [tz][ty][tx][NV]
    const int tid = threadIdx.x;

    const int64_t mit = pt.mx + 4, mij = mit * (pt.my + 4);
    const int64_t plane = mij * (pt.mz + 4);
    const T* qin = static_cast<const T*>(a.qin) + pt.qoff;
    // array index of local cell (-2, -2, -2): 1-based cell i0 + 1 - 2 sits
    // at index i0 + 1 - 2 + 1 = i0 (two ghost cells)
    const int64_t g0 = (int64_t)td.k0 * mij + (int64_t)td.j0 * mit + td.i0;
    {
        Digits3 u(tid, bx, by, bz);
        for (int idx = tid; idx < NV * nbox; idx += TILE3_LANES, u.step())
            qs[((u.z * by + u.y) * bx + u.x) * NV + u.m] = qin[u.m * plane + g0 + (int64_t)u.z * mij + (int64_t)u.y * mit + u.x];
    }
    for (int idx = tid; idx < NV * ncell; idx += TILE3_LANES) dq[idx] = T(0);
    Mark3Lds mk{};
    // a mark's place in the map: its face array, row by row
    auto mark_at = [&](const Mark3& f) {
        const int nfx = (tx + 1) * ty * tz, nfy = tx * (ty + 1) * tz;
        const int w = tx + (f.dir == 0), h = ty + (f.dir == 1);
        return (f.dir == 0 ? 0 : (f.dir == 1 ? nfx : nfx + nfy)) + (f.z * h + f.y) * w + f.x;
    };
    if constexpr (MARK) {
        mk.map = reinterpret_cast<uint16_t*>(dq + NV * ncell);
        const int words = (mark3_faces(tx, ty, tz) + 1) / 2;
        mk.acc = dq + NV * ncell + words;
        uint32_t* w = reinterpret_cast<uint32_t*>(mk.map);
        for (int idx = tid; idx < words; idx += TILE3_LANES) w[idx] = 0;
        for (int idx = tid; idx < td.nmark * 3 * NV; idx += TILE3_LANES) mk.acc[idx] = T(0);
        __syncthreads();
        for (int idx = tid; idx < td.nmark; idx += TILE3_LANES)
            mk.map[mark_at(a.marks[td.mark0 + idx])] = (uint16_t)(idx + 1);
    }
    __syncthreads();

    // the wave's number in a scalar register, so that its rows and chunks are
    // scalar work
    const int wave = __builtin_amdgcn_readfirstlane(tid / 64), wl = tid - wave * 64;
    T cfl = T(0);

    tile3_sweep<Sol, 1, STD, MARK>(a, qs, dq, tx, ty, tz, bx, by, wave, wl, cfl, mk);
    tile3_sweep<Sol, 2, STD, MARK>(a, qs, dq, tx, ty, tz, bx, by, wave, wl, cfl, mk);
    tile3_sweep<Sol, 3, STD, MARK>(a, qs, dq, tx, ty, tz, bx, by, wave, wl, cfl, mk);
    __syncthreads();

    // q(t + dt) = q(t) + dq on the tile's cells
    T* qout = static_cast<T*>(a.qout) + pt.qoff;
    {
        Digits3 u(tid, tx, ty, tz);
        for (int idx = tid; idx < NV * ncell; idx += TILE3_LANES, u.step()) {
            const T v = qs[((u.z + 2) * bx * by + (u.y + 2) * bx + (u.x + 2)) * NV + u.m] +
                        dq[((u.z * ty + u.y) * tx + u.x) * NV + u.m];
            qout[u.m * plane + g0 + (int64_t)(u.z + 2) * mij + (int64_t)(u.y + 2) * mit + (u.x + 2)] = v;
        }
    }
    if constexpr (MARK) {
        // the grid's ghost cells keep their time-t values: of the staged box,
        // what lies outside the grid, each cell written by the tile beside it
        // (the tile's range extended by two cells at the grid's own sides)
        const int xl = td.i0 == 0 ? 0 : 2, xh = td.i0 + tx == pt.mx ? bx : bx - 2;
        const int yl = td.j0 == 0 ? 0 : 2, yh = td.j0 + ty == pt.my ? by : by - 2;
        const int zl = td.k0 == 0 ? 0 : 2, zh = td.k0 + tz == pt.mz ? bz : bz - 2;
        if (xl == 0 || xh == bx || yl == 0 || yh == by || zl == 0 || zh == bz) {
            Digits3 u(tid, bx, by, bz);
            for (int idx = tid; idx < NV * nbox; idx += TILE3_LANES, u.step()) {
                const bool mine = u.x >= xl && u.x < xh && u.y >= yl && u.y < yh && u.z >= zl && u.z < zh;
                const bool cell = u.x >= 2 && u.x < bx - 2 && u.y >= 2 && u.y < by - 2 && u.z >= 2 &&
                                  u.z < bz - 2;
                if (mine && !cell)
                    qout[u.m * plane + g0 + (int64_t)u.z * mij + (int64_t)u.y * mit + u.x] =
                        qs[((u.z * by + u.y) * bx + u.x) * NV + u.m];
            }
        }
        // the marked faces into the grid's flux block: fm and fp - fm (gm, gp
        // likewise), hm and hp
        const Faces3 F = faces3(pt, NV);
        for (int idx = tid; idx < td.nmark * NV; idx += TILE3_LANES) {
            const int id = idx / NV, m = idx - id * NV;
            const Mark3 f = a.marks[td.mark0 + id];
            const T lo = T(double(mk.acc[id * 3 * NV + m] + mk.acc[(id * 3 + 1) * NV + m]) / a.dtd[f.dir]);
            const T df = mk.acc[(id * 3 + 2) * NV + m];
            const int x = td.i0 + f.x, y = td.j0 + f.y, z = td.k0 + f.z;
            const int w = pt.mx + (f.dir == 0), h = pt.my + (f.dir == 1);
            const int64_t at = m * (f.dir == 0 ? F.sx : (f.dir == 1 ? F.sy : F.sz)) +
                               ((int64_t)z * h + y) * w + x;
            a.face[(f.dir == 0 ? F.fm : (f.dir == 1 ? F.gm : F.hm)) + at] = lo;
            a.face[(f.dir == 0 ? F.fp : (f.dir == 1 ? F.gp : F.hp)) + at] = f.dir == 2 ? lo + df : df;
        }
    }
    double cd = double(cfl);
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        double o2 = __shfl_xor(cd, off, 64);
        cd = cd > o2 ? cd : o2;
    }
    if ((tid & 63) == 0) atomic_max_nonneg3(&a.cfl_patch[td.patch], cd);
}

}  // namespace amrgpu
