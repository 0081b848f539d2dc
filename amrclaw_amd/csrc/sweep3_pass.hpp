// sweep3_pass.hpp -- the 3-D step in two passes over a work space in HBM: every
// line of the three sweeps solved at once, then every face summed.
//
// step3.f adds each line's increments to the faces in the order of its loops,
// and an FP64 step has to keep that order bit for bit.  The phase kernels
// (sweep3.hpp) keep it by marching a workgroup through a grid's planes; a batch
// of few grids then leaves most of the chip idle (32 grids of 8 .. 32 cells a
// side: 713 waves for 1024 SIMDs, vector issue 12 %), and each block of planes
// solves its two neighbours again.  Here
//   pass3_solve_kernel<D>  takes the lines of sweep D in any order, one lane
//     per interface, and stores what flux3.f returns for the line: gadd and
//     hadd of each cell and faddm / faddp of each interface (flux3.f:220-628),
//     each interface solved once (lines of more than 61 cells are cut into
//     pieces that solve their ends twice);
//   pass3_face_kernel      sums, one face component per thread, the increments
//     step3.f:140-321 adds to that face, in its order: the x-, y-, z-sweep, in
//     each the lines in ascending (plane, line) order.
// The work space takes 14 * nv values per interface and sweep (560 bytes for
// Euler); the host cuts a batch into runs of grids that share it.
//
// Bound by that traffic: 32 grids (324 k cells) write 0.66 GB of work space at
// 1.75 TB/s (a large copy on this card writes 2.4 TB/s) and read it back at 2.8
// TB/s.  Measured against the phase kernels, FP64 Euler, method(3) = 22, a step:
// one grid of 21x18x13 1,140 -> 88 us, 32 grids 2,147 -> 649 us, 128 3,443 ->
// 2,084 us, 512 12.35 -> 7.65 ms; with one Courant atomic a workgroup and grid
// instead of one a wave, 512 6.9 ms, 8 grids of 40^3 1,050 -> 900 us.
#pragma once
#include "lanes.hpp"
#include "sweep3.hpp"

namespace amrgpu {

constexpr int PASS3_CELLS = 61;        // cells of a line one wave can take (64 lanes)
constexpr int PASS3_SLOTS = 14;        // gadd 0..5, hadd 6..11, faddm, faddp

// the work-space offsets of a grid's three sweeps
struct Pass3Ws {
    int64_t off[3];
};
// one wave's share of a sweep: pieces [unit0, ..) of lines of a grid
struct Pass3Wave {
    int32_t patch, unit0;
};

// geometry of sweep d of a grid: cells n along the lines, NQ x NP lines inside
// (one more on each side is solved), pieces per line, cells and lanes of a piece
struct Pass3Geom {
    int n, NQ, NP, nseg, w, L, lpw;
};
__host__ __device__ inline Pass3Geom pass3_geom(const Patch3& p, int d) {
    Pass3Geom g;
    g.n = d == 1 ? p.mx : (d == 2 ? p.my : p.mz);
    g.NQ = d == 1 ? p.my : p.mx;
    g.NP = d == 3 ? p.my : p.mz;
    g.nseg = (g.n + PASS3_CELLS - 1) / PASS3_CELLS;
    g.w = (g.n + g.nseg - 1) / g.nseg;
    g.L = g.w + 3;
    g.lpw = 64 / g.L;
    return g;
}
__host__ __device__ inline int64_t pass3_elems(const Patch3& p, int d, int nv) {
    const Pass3Geom g = pass3_geom(p, d);
    return (int64_t)PASS3_SLOTS * nv * (g.NQ + 2) * (g.NP + 2) * (g.n + 1);
}

struct Pass3Args {
    const void* q;
    void* ws;
    void* face;
    const Patch3* patches;
    const Pass3Ws* off;             // of every grid, from the run's work space
    const Pass3Wave* waves;
    const Block3* blocks;           // face kernel: 256 face components each
    int32_t nwaves, nblocks;
    double dtd[3];
    Method3 meth;
    unsigned long long* cfl_patch;
};

template <class Sol, typename T, int D>
__global__ __launch_bounds__(256, 2) void pass3_solve_kernel(Pass3Args a) {
    constexpr int NV = Sol::NV, NW = Sol::NW;
    __shared__ T park[2][2][2][NV][256];
    const int wv = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (wv >= a.nwaves) return;   // the whole wave leaves
    const Method3& M = a.meth;
    const Pass3Wave W = a.waves[wv];
    const Patch3 pt = a.patches[W.patch];
    const Pass3Geom G = pass3_geom(pt, D);
    const int lane = threadIdx.x & 63;
    const int li = lane / G.L, e = lane - li * G.L;
    const int unit = W.unit0 + li, nunits = (G.NQ + 2) * (G.NP + 2) * G.nseg;
    const bool live = li < G.lpw && unit < nunits;
    const int uc = live ? unit : W.unit0;
    const int line = uc / G.nseg, c0 = (uc - line * G.nseg) * G.w;
    const int wc = min(G.w, G.n - c0);                 // cells of this piece
    const int P = line / (G.NQ + 2), Q = line - P * (G.NQ + 2);
    const int r = c0 + min(e, wc + 2);                 // interface between cells r-1 and r
    const bool inner = live && e >= 1 && e <= wc + 1;  // interfaces 1 .. n+1
    const int64_t mit = pt.mx + 4, mij = mit * (pt.my + 4), plane = mij * (pt.mz + 4);
    const int64_t qr_s = D == 1 ? 1 : (D == 2 ? mit : mij);
    const int64_t qq_s = D == 1 ? mit : 1, qp_s = D == 3 ? mit : mij;
    const T* q = static_cast<const T*>(a.q) + pt.qoff + r * qr_s + (Q + 1) * qq_s + (P + 1) * qp_s;
    T ql[NV], qrr[NV];   // cell r - 1 at index r (two ghost cells), cell r after it
#pragma unroll
    for (int m = 0; m < NV; m++) {
        ql[m] = q[m * plane];
        qrr[m] = q[m * plane + qr_s];
    }
    const T dtdx = T(a.dtd[D - 1]);
    const T dtdy_p = T(a.dtd[D % 3]), dtdz_p = T(a.dtd[(D + 1) % 3]);
    const T half_t = T(0.5) * dtdx;
    const T sixth = T(1) / T(6);
    const T g6 = sixth * dtdx * dtdz_p, h6 = sixth * dtdx * dtdy_p;
    const bool trans = M.m3 > 0, cq = M.m3 >= 2, tt = M.m4 > 0;
    bool limit = false;
    for (int w = 0; w < NW; w++) limit = limit || M.mthlim[w] > 0;

    const typename Sol::Cache cache = Sol::prep(M.ph, ql, qrr);
    T wave[NW][NV], s[NW], amdq[NV], apdq[NV];
    Sol::rpn3(M.ph, D, ql, qrr, cache, wave, s, amdq, apdq);
    T cfl = T(0);
    if (inner) {
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
    if (M.order != 1) {
        if (limit) {   // inlinelimiter.f on unlimited neighbour waves
#pragma unroll
            for (int w = 0; w < NW; w++) {
                T wn2 = T(0), dotr = T(0);
#pragma unroll
                for (int m = 0; m < NV; m++) {
                    wn2 = wn2 + wave[w][m] * wave[w][m];
                    dotr = dotr + wave[w][m] * lane_down(wave[w][m], 0);
                }
                const T dotl = lane_up(dotr, 0);   // the product of the interface before
                const int mth = M.mthlim[w];
                if (mth != 0 && inner && wn2 != T(0)) {
                    using Mth = typename Sol::Math;
                    const T wl = phi_limiter3<Mth>(mth, Mth::ratio(s[w] > T(0) ? dotl : dotr, wn2));
#pragma unroll
                    for (int m = 0; m < NV; m++) wave[w][m] = wl * wave[w][m];
                }
            }
        }
        const T dtdxave = T(0.5) * (dtdx + dtdx);
#pragma unroll
        for (int m = 0; m < NV; m++) {
            T c = T(0);
#pragma unroll
            for (int w = 0; w < NW; w++) {
                const T fac = M.use_fwaves ? (s[w] >= T(0) ? T(1) : T(-1)) : fabs(s[w]);
                c = c + T(0.5) * fac * (T(1) - fabs(s[w]) * dtdxave) * wave[w][m];
            }
            cqxx[m] = c;
            fadm[m] = fadm[m] + c;
            fadp[m] = fadp[m] + c;
        }
    }
    // this line's row of the work space: interface r at r - 1, cell c at c - 1
    const int64_t rl = G.n + 1, cs = (int64_t)(G.NQ + 2) * (G.NP + 2) * rl;
    T* out = static_cast<T*>(a.ws) + a.off[W.patch].off[D - 1] + (int64_t)line * rl;
    // an interface two pieces share is stored by the one it begins
    if (inner && (e <= wc || r == G.n + 1) && Q >= 1 && Q <= G.NQ && P >= 1 && P <= G.NP) {
#pragma unroll
        for (int m = 0; m < NV; m++) {
            out[(12 * NV + m) * cs + r - 1] = fadm[m];
            out[(13 * NV + m) * cs + r - 1] = fadp[m];
        }
    }
    if (trans) {
        const bool cell = live && e >= 2 && e <= wc + 1;   // completes cell r - 1
        // the splits both families use, once: of cqxx, A+dq and A-dq along
        // icoor 2 and 3 (index 0: 2, 1: 3; [0] down-, [1] up-going).  Those of
        // cqxx and A-dq wait in LDS, each lane its own (no barrier): held in
        // registers they allow one wave per SIMD only (322 registers)
        T As[2][2][NV];
        const int tid = threadIdx.x;
        auto Cs = [&](int i, int s, int m) -> T& { return park[0][i][s][m][tid]; };
        auto Ms = [&](int i, int s, int m) -> T& { return park[1][i][s][m][tid]; };
#pragma unroll
        for (int i = 0; i < 2; i++) {
            T x[NV], y[NV];
            if (cq) {
                Sol::split(M.ph, D, 2 + i, ql, qrr, cache, cqxx, x, y);
#pragma unroll
                for (int m = 0; m < NV; m++) Cs(i, 0, m) = x[m], Cs(i, 1, m) = y[m];
            }
            Sol::split(M.ph, D, 2 + i, ql, qrr, cache, amdq, x, y);
#pragma unroll
            for (int m = 0; m < NV; m++) Ms(i, 0, m) = x[m], Ms(i, 1, m) = y[m];
            Sol::split(M.ph, D, 2 + i, ql, qrr, cache, apdq, As[i][0], As[i][1]);
        }
#pragma unroll
        for (int fam = 0; fam < 2; fam++) {
            // fam 0 = gadd: primary split along icoor 2; fam 1 = hadd
            const int ip = fam, is = 1 - fam, icp = 2 + ip;
            const T w6 = fam == 0 ? g6 : h6;
            T tmp[NV], rm[NV], rp[NV], sm[NV], sp[NV];
            // right-cell partials of this interface, slot k = (s-1)*3 + (o+1),
            // statement order of flux3.f:450-505 (A+dq side)
            T v[6][NV];
#pragma unroll
            for (int m = 0; m < NV; m++) {
                v[0][m] = v[2][m] = v[3][m] = v[5][m] = T(0);
                v[1][m] = T(0) - half_t * As[ip][0][m];
                v[4][m] = T(0) - half_t * As[ip][1][m];
            }
            if (tt) {
#pragma unroll
                for (int m = 0; m < NV; m++)
                    tmp[m] = M.m4 == 2 ? As[is][1][m] - T(3) * Cs(is, 1, m) : As[is][1][m];
                Sol::split(M.ph, D, icp, ql, qrr, cache, tmp, rm, rp);      // "p" part
#pragma unroll
                for (int m = 0; m < NV; m++)
                    tmp[m] = M.m4 == 2 ? As[is][0][m] - T(3) * Cs(is, 0, m) : As[is][0][m];
                Sol::split(M.ph, D, icp, ql, qrr, cache, tmp, sm, sp);      // "m" part
#pragma unroll
                for (int m = 0; m < NV; m++) {
                    v[4][m] = v[4][m] + w6 * (rp[m] - sp[m]);
                    v[1][m] = v[1][m] + w6 * (rm[m] - sm[m]);
                    v[5][m] = T(0) - w6 * rp[m];
                    v[2][m] = T(0) - w6 * rm[m];
                    v[3][m] = T(0) + w6 * sp[m];
                    v[0][m] = T(0) + w6 * sm[m];
                }
            }
            if (cq) {
#pragma unroll
                for (int m = 0; m < NV; m++) {
                    v[4][m] = v[4][m] + dtdx * Cs(ip, 1, m);
                    v[1][m] = v[1][m] + dtdx * Cs(ip, 0, m);
                }
            }
            // cell r-1: the left neighbour's partials, then this interface's
            // left-cell increments (A-dq side)
#pragma unroll
            for (int k = 0; k < 6; k++)
#pragma unroll
                for (int m = 0; m < NV; m++) v[k][m] = lane_up(v[k][m], 0);
#pragma unroll
            for (int m = 0; m < NV; m++) {
                v[1][m] = v[1][m] - half_t * Ms(ip, 0, m);
                v[4][m] = v[4][m] - half_t * Ms(ip, 1, m);
            }
            if (tt) {
#pragma unroll
                for (int m = 0; m < NV; m++)
                    tmp[m] = M.m4 == 2 ? Ms(is, 1, m) + T(3) * Cs(is, 1, m) : Ms(is, 1, m);
                Sol::split(M.ph, D, icp, ql, qrr, cache, tmp, rm, rp);
#pragma unroll
                for (int m = 0; m < NV; m++)
                    tmp[m] = M.m4 == 2 ? Ms(is, 0, m) + T(3) * Cs(is, 0, m) : Ms(is, 0, m);
                Sol::split(M.ph, D, icp, ql, qrr, cache, tmp, sm, sp);
#pragma unroll
                for (int m = 0; m < NV; m++) {
                    v[4][m] = v[4][m] + w6 * (rp[m] - sp[m]);
                    v[1][m] = v[1][m] + w6 * (rm[m] - sm[m]);
                    v[5][m] = v[5][m] - w6 * rp[m];
                    v[2][m] = v[2][m] - w6 * rm[m];
                    v[3][m] = v[3][m] + w6 * sp[m];
                    v[0][m] = v[0][m] + w6 * sm[m];
                }
            }
            if (cq) {
#pragma unroll
                for (int m = 0; m < NV; m++) {
                    v[4][m] = v[4][m] - dtdx * Cs(ip, 1, m);
                    v[1][m] = v[1][m] - dtdx * Cs(ip, 0, m);
                }
            }
            if (cell) {
#pragma unroll
                for (int k = 0; k < 6; k++) {
                    if (!tt && k != 1 && k != 4) continue;   // exact zeros, never read
#pragma unroll
                    for (int m = 0; m < NV; m++) out[((fam * 6 + k) * NV + m) * cs + r - 2] = v[k][m];
                }
            }
        }
    }
    double cd = double(cfl);
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        const double o2 = __shfl_xor(cd, off, 64);
        cd = cd > o2 ? cd : o2;
    }
    // one atomic for the neighbouring waves of a grid in the workgroup: tens of
    // thousands of waves share a few grids' words, all in one cache line or a few
    // (8 grids of 40^3, advection, 14,112 waves a sweep: 165 us a launch with an
    // atomic from every wave, 47 with this).  Looking at the word first, at the
    // wave's start or end, queues on the same line.  Each wave's lane 0 leaves its
    // value and its grid in places of its own wave in LDS.
    T* mine = &park[0][0][0][0][threadIdx.x & 192];
    if (lane == 0) {
        mine[0] = T(cd);
        mine[1] = T(W.patch);   // lane 1's place, of the same wave
    }
    __syncthreads();
    const int w0 = threadIdx.x >> 6, n = min(4, a.nwaves - (int)blockIdx.x * 4);
    if (lane == 0 && (w0 == 0 || mine[1 - 64] != mine[1])) {
        for (int w = w0 + 1; w < n && mine[(w - w0) * 64 + 1] == mine[1]; w++)
            cd = fmax(cd, double(mine[(w - w0) * 64]));
        atomic_max_nonneg3(&a.cfl_patch[W.patch], cd);
    }
}

// faces of a grid in the face kernel's numbering: x, y, z arrays, component
// slowest within each
__host__ __device__ inline int64_t pass3_face_count(const Patch3& p, int nv) {
    const Faces3 F = faces3(p, nv);
    return nv * (F.sx + F.sy + F.sz);
}

// The idx-th element of an X x Y x Z box in bricks: strips of bx along x, in
// each strips of by along y, in each z, then y, then x.
__device__ __forceinline__ void pass3_brick(int idx, int X, int Y, int Z, int bx, int by, int& x,
                                            int& y, int& z) {
    const int sx = idx / (bx * Y * Z);
    idx -= sx * bx * Y * Z;
    const int wx = min(bx, X - sx * bx);
    const int sy = idx / (wx * by * Z);
    idx -= sy * wx * by * Z;
    const int wy = min(by, Y - sy * by);
    z = idx / (wx * wy);
    idx -= z * wx * wy;
    y = idx / wx;
    x = idx - y * wx + sx * bx;
    y += sy * by;
}

// The sums read two sweeps whose lines run along different axes: a wave takes
// a brick of faces (4 x 4 x 4, or 8 x 8 in the plane of the two lines), so that
// either sweep's values come in runs, and consecutive workgroups go to one XCD,
// whose L2 then serves what its neighbours fetched (workgroups are dealt to the
// eight XCDs in turn).
template <int NV, typename T>
__global__ __launch_bounds__(256) void pass3_face_kernel(Pass3Args a) {
    const int per = gridDim.x / 8, b = (blockIdx.x % 8) * per + blockIdx.x / 8;
    if (b >= a.nblocks) return;
    const Block3 blk = a.blocks[b];
    const int64_t id = (int64_t)blk.pb * 256 + threadIdx.x;   // pb: block number within the grid
    const Patch3 pt = a.patches[blk.patch];
    const Faces3 F = faces3(pt, NV);
    if (id >= NV * (F.sx + F.sy + F.sz)) return;
    const bool trans = a.meth.m3 > 0, tt = a.meth.m4 > 0;
    const T* ws = static_cast<const T*>(a.ws);
    const Pass3Ws off = a.off[blk.patch];
    T* face = static_cast<T*>(a.face);
    const int mx = pt.mx, my = pt.my, mz = pt.mz;
    // value `slot` of line (Q, P), cell or interface c (1-based), of sweep d
    auto at = [&](int d, int slot, int m, int P, int Q, int c) -> T {
        const int n = d == 1 ? mx : (d == 2 ? my : mz), NQ = d == 1 ? my : mx, NP = d == 3 ? my : mz;
        const int64_t rl = n + 1, lines = (int64_t)(NQ + 2) * (NP + 2);
        return ws[off.off[d - 1] + ((slot * NV + m) * lines + (int64_t)P * (NQ + 2) + Q) * rl + c - 1];
    };
    // the increments of one family (f: 0 gadd, 6 hadd) of sweep d to the face
    // whose upper cell is line Qf across Q (across P in `acrossP`)
    auto across_q = [&](T& x1, T& x2, int d, int f, int m, int Pf, int Qf, int c) {
#pragma unroll
        for (int o = 1; o >= -1; o--) {            // planes Pf-1, Pf, Pf+1
            if (o != 0 && !tt) continue;
            const T lo = at(d, f + 3 + o + 1, m, Pf - o, Qf - 1, c), hi = at(d, f + o + 1, m, Pf - o, Qf, c);
            x1 = (x1 + lo) + hi;
            x2 = (x2 + lo) + hi;
        }
    };
    auto across_p = [&](T& x1, T& x2, int d, int f, int m, int Pf, int Qf, int c) {
#pragma unroll
        for (int s = 2; s >= 1; s--) {             // plane Pf-1 (its upper face), then Pf
#pragma unroll
            for (int o = 1; o >= -1; o--) {        // lines Qf-1, Qf, Qf+1
                if (o != 0 && !tt) continue;
                const T v = at(d, f + (s - 1) * 3 + o + 1, m, Pf - (s - 1), Qf - o, c);
                x1 = x1 + v;
                x2 = x2 + v;
            }
        }
    };
    if (id < NV * F.sx) {
        const int m = (int)(id / F.sx);
        int i, j, k;
        pass3_brick((int)(id - m * F.sx), mx + 1, my, mz, 4, 4, i, j, k);
        const int64_t to = m * F.sx + ((int64_t)k * my + j) * (mx + 1) + i;
        i++, j++, k++;
        T fm = at(1, 12, m, k, j, i), fp = at(1, 13, m, k, j, i);
        if (trans) {
            across_q(fm, fp, 2, 6, m, k, i, j);    // y-sweep hadd: P = k, Q = i, cell j
            across_q(fm, fp, 3, 0, m, j, i, k);    // z-sweep gadd: P = j, Q = i, cell k
        }
        face[F.fm + to] = fm;
        face[F.fp + to] = fp;
    } else if (id < NV * (F.sx + F.sy)) {
        const int64_t l = id - NV * F.sx;
        const int m = (int)(l / F.sy);
        int i, j, k;
        pass3_brick((int)(l - m * F.sy), mx, mz, my + 1, 8, 8, i, k, j);
        const int64_t to = m * F.sy + ((int64_t)k * (my + 1) + j) * mx + i;
        i++, j++, k++;
        T gm = T(0), gp = T(0);
        if (trans) across_q(gm, gp, 1, 0, m, k, j, i);   // x-sweep gadd: P = k, Q = j, cell i
        gm = gm + at(2, 12, m, k, i, j);
        gp = gp + at(2, 13, m, k, i, j);
        if (trans) across_p(gm, gp, 3, 6, m, j, i, k);   // z-sweep hadd: face across P = j
        face[F.gm + to] = gm;
        face[F.gp + to] = gp;
    } else {
        const int64_t l = id - NV * (F.sx + F.sy);
        const int m = (int)(l / F.sz);
        int i, j, k;
        pass3_brick((int)(l - m * F.sz), mx, my, mz + 1, 8, 8, i, j, k);
        const int64_t to = m * F.sz + ((int64_t)k * my + j) * mx + i;
        i++, j++, k++;
        T hm = T(0), hp = T(0);
        if (trans) {
            across_p(hm, hp, 1, 6, m, k, j, i);    // x-sweep hadd: face across P = k, Q = j
            across_p(hm, hp, 2, 0, m, k, i, j);    // y-sweep gadd: face across P = k, Q = i
        }
        hm = hm + at(3, 12, m, j, i, k);
        hp = hp + at(3, 13, m, j, i, k);
        face[F.hm + to] = hm;
        face[F.hp + to] = hp;
    }
}

}  // namespace amrgpu
