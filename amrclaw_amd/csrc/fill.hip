// fill.hip -- executes ghost-cell fill programs.
// Built with -ffp-contract=off: the time blend and the coarse-fine
// interpolation are evaluated exactly as the reference's FP64 code.
#include <hip/hip_runtime.h>
#include "fill.hpp"
#include "sweep.hpp"

namespace amrgpu {

// the values of a buffer: a level's storage, or FP64 scratch or arena
template <typename E>
struct Cells {
    E* p;
    int32_t nrow, plane;
    __device__ double load(int m, int i, int j) const { return at((int64_t)m * plane + (int64_t)j * nrow + i); }
    __device__ double at(int64_t k) const { return (double)p[k]; }
    __device__ void store(int m, int i, int j, double v) const { put((int64_t)m * plane + (int64_t)j * nrow + i, v); }
    __device__ void put(int64_t k, double v) const { p[k] = (E)v; }
};

// what an operation other than FOP_COPY reads: always scratch or arena
__device__ __forceinline__ Cells<const double> src_cells(const FillArgs& a, const FillProg& pr, const FillItem& op) {
    return {(op.src_space == FSP_SCRATCH ? pr.scratch : a.arena) + op.src_off, op.src_nrow, op.src_plane};
}

// f(the operation's destination).  The kind is told apart here, once: asked for
// at every element, it doubled the loads, stores and addresses in flight of the
// FP32 kernels (151 registers, now 117 and 127; a ghost fill of a 1024^2 level 43.7
// -> 31.4 us, of 64 grids of 32^2 22.3 -> 20.7, of 1,600 of 24^2 75.6 -> 70.6).
template <typename S, class F>
__device__ __forceinline__ void with_dst(const FillArgs& a, const FillProg& pr, const FillItem& op, const F& f) {
    double* w = (op.dst_space == FSP_SCRATCH ? pr.scratch : a.arena) + op.dst_off;
    if constexpr (sizeof(S) == sizeof(double)) {
        if (op.dst_space >= 0) w = static_cast<double*>(a.lvl_new[op.dst_space]) + op.dst_off;
        f(Cells<double>{w, op.dst_nrow, op.dst_plane});
    } else if (op.dst_space >= 0) {
        f(Cells<S>{static_cast<S*>(a.lvl_new[op.dst_space]) + op.dst_off, op.dst_nrow, op.dst_plane});
    } else {
        f(Cells<double>{w, op.dst_nrow, op.dst_plane});
    }
}

// cell idx of the ring cstore.f walks: sides 1 (left column), 2 (top row), 3
// (right column), 4 (bottom row) of the coarsened patch, corners excluded
__device__ __forceinline__ int64_t ring_cell(int idx, int nrow, int ncol) {
    const int n1 = ncol - 2, n2 = nrow - 2;
    int i, j;
    if (idx < n1) { i = 0; j = 1 + idx; }
    else if (idx < n1 + n2) { i = 1 + idx - n1; j = ncol - 1; }
    else if (idx < 2 * n1 + n2) { i = nrow - 1; j = 1 + idx - n1 - n2; }
    else { i = 1 + idx - 2 * n1 - n2; j = 0; }
    return (int64_t)j * nrow + i;
}

// the aux-mode copy of a saveqc program: aux values of the coarse grids
// into the coarse patch (icall.f's aux part) and the patch's ring into
// auxc1d (cstore.f); NEEDS_TO_BE_SET stays where no coarse grid reached
template <int NT>
__device__ void fill_aux_op(const FillArgs& a, const FillProg& pr, const FillItem& op, int tid) {
    const int na = a.naux;
    if (op.type == FOP_COPY) {
        const double* sa = a.lvl_aux[op.src_space] + op.src_off * a.auxk + op.src_shift;
        double* da = pr.scratch + op.dst_off * a.auxk + op.dst_shift;
        const int ncell = op.ni * op.nj;
        for (int t = tid; t < ncell * na; t += NT) {
            const int c = t / ncell, r = t - c * ncell;
            const int dj = r / op.ni, di = r - dj * op.ni;
            da[(int64_t)c * op.dst_plane + (int64_t)dj * op.dst_nrow + di] =
                sa[(int64_t)c * op.src_plane + (int64_t)dj * op.src_nrow + di];
        }
    } else if (op.type == FOP_RING) {
        const double* sa = pr.scratch + op.src_off * a.auxk;
        double* ac1d = a.lvl_reg[op.level] + op.aux_off;
        const int len = 2 * (op.ni - 2 + op.nj - 2);
        for (int t = tid; t < len * na; t += NT) {
            const int idx = t / na, c = t - idx * na;
            ac1d[(int64_t)idx * na + c] = sa[(int64_t)c * op.src_plane + ring_cell(idx, op.ni, op.nj)];
        }
    }
}

// t = tid + NT k written as digits (i, j, m) of the radices (ni, nj):
// stepped by NT with one carry per digit instead of two integer divisions
// per element (a digit plus its step plus a carry stays below twice its
// radix, so one subtraction brings it back)
template <int NT>
struct Digits2 {
    int i, j, m, si, sj, sm, ni, nj;
    __device__ __forceinline__ Digits2(int t, int ni_, int nj_)
        : ni(ni_ > 0 ? ni_ : 1), nj(nj_ > 0 ? nj_ : 1) {   // (an empty op runs no element)
        i = t % ni; t /= ni; j = t % nj; m = t / nj;
        int r = NT;
        si = r % ni; r /= ni; sj = r % nj; sm = r / nj;
    }
    __device__ __forceinline__ void step() {
        i += si;
        int c = i >= ni;
        i -= c ? ni : 0;
        j += sj + c;
        c = j >= nj;
        j -= c ? nj : 0;
        m += sm + c;
    }
};

// every element (cell x component) of a rectangle from `load` into `dst`,
// four elements a thread in flight
template <int NT, typename E, class Load>
__device__ __forceinline__ void copy_rect(const FillItem& op, const Cells<E>& dst, int tid, int nv,
                                          const Load& load) {
    const int n = op.ni * op.nj * nv;
    Digits2<NT> u(tid, op.ni, op.nj);
    for (int t = tid; t < n; t += 4 * NT) {
        double v[4];
        int64_t d[4];
#pragma unroll
        for (int k = 0; k < 4; k++, u.step()) {
            d[k] = t + NT * k < n ? (int64_t)u.m * dst.plane + (int64_t)u.j * dst.nrow + u.i : -1;
            if (d[k] >= 0) v[k] = load((int64_t)u.m * op.src_plane + (int64_t)u.j * op.src_nrow + u.i);
        }
#pragma unroll
        for (int k = 0; k < 4; k++)
            if (d[k] >= 0) dst.put(op.dst_shift + d[k], v[k]);
    }
}

// components n .. n + C - 1 of the interpolation at one fine cell: all the
// coarse values are loaded before the first store (to an array the compiler
// cannot tell apart from theirs)
template <int C, typename E>
__device__ __forceinline__ void interp_cell(const Cells<const double>& crs, const Cells<E>& dst, int n,
                                            int64_t s, int64_t d, double eta1, double eta2) {
    double p10[C], m10[C], c0[C], p01[C], m01[C];
#pragma unroll
    for (int k = 0; k < C; k++) {
        const int64_t b = s + (int64_t)(n + k) * crs.plane;
        p10[k] = crs.at(b + 1);
        m10[k] = crs.at(b - 1);
        c0[k] = crs.at(b);
        p01[k] = crs.at(b + crs.nrow);
        m01[k] = crs.at(b - crs.nrow);
    }
#pragma unroll
    for (int k = 0; k < C; k++) {
        const double dupc = p10[k] - c0[k], dumc = c0[k] - m10[k], ducc = p10[k] - m10[k];
        double du = fmin(fabs(dupc), fabs(dumc));
        du = fmin(2.0 * du, 0.5 * fabs(ducc));
        const double fu = fmax(0.0, copysign(1.0, dupc * dumc));
        const double uslope = du * copysign(1.0, ducc) * fu;
        const double dvpc = p01[k] - c0[k], dvmc = c0[k] - m01[k], dvcc = p01[k] - m01[k];
        double dv = fmin(fabs(dvpc), fabs(dvmc));
        dv = fmin(2.0 * dv, 0.5 * fabs(dvcc));
        const double fv = fmax(0.0, copysign(1.0, dvpc * dvmc));
        const double vslope = dv * copysign(1.0, dvcc) * fv;
        dst.put(d + (int64_t)(n + k) * dst.plane, c0[k] + eta1 * uslope + eta2 * vslope);
    }
}

// One side of bc2amr: the cells [i0, i0 + ni) x [j0, j0 + nj), none of which is
// read, from the cells (ai i + bi, aj j + bj), component `flip` negated.
struct BcSide { int ni, nj, i0, j0, ai, bi, aj, bj, flip; };

// Components m0 .. m0 + C - 1 of B cells a thread in flight.  By cells, so that
// the digits are stepped once a cell: the four sides of a 1024^2 grid of four
// components take a ghost fill of 32 us, element by element 52.
template <int NT, int C, int B, typename E>
__device__ __forceinline__ void bc_cells(const Cells<E>& b, const BcSide& sd, int tid, int m0) {
    const int n = sd.ni * sd.nj;
    Digits2<NT> u(tid, sd.ni, 1 << 30);   // (i, j) of a cell; j does not wrap
    for (int t = tid; t < n; t += B * NT) {
        double v[B][C];
        int64_t d[B];
#pragma unroll
        for (int k = 0; k < B; k++, u.step()) {
            const int i = sd.i0 + u.i, j = sd.j0 + u.j;
            d[k] = t + NT * k < n ? (int64_t)m0 * b.plane + (int64_t)j * b.nrow + i : -1;
            if (d[k] >= 0) {
                const int64_t s = (int64_t)m0 * b.plane + (int64_t)(sd.aj * j + sd.bj) * b.nrow +
                                  (sd.ai * i + sd.bi);
#pragma unroll
                for (int m = 0; m < C; m++) {
                    v[k][m] = b.at(s + (int64_t)m * b.plane);
                    if (m0 + m == sd.flip) v[k][m] = -v[k][m];
                }
            }
        }
#pragma unroll
        for (int k = 0; k < B; k++)
            if (d[k] >= 0) {
#pragma unroll
                for (int m = 0; m < C; m++) b.put(d[k] + (int64_t)m * b.plane, v[k][m]);
            }
    }
}
template <int NT, typename E>
__device__ __forceinline__ void bc_side(const Cells<E>& b, const BcSide& sd, int tid, int nv) {
    int m = 0;
    for (; m + 4 <= nv; m += 4) bc_cells<NT, 4, 2>(b, sd, tid, m);
    if (nv - m == 3) bc_cells<NT, 3, 3>(b, sd, tid, m);
    else if (nv - m == 2) bc_cells<NT, 2, 4>(b, sd, tid, m);
    else if (nv - m == 1) bc_cells<NT, 1, 8>(b, sd, tid, m);
}

constexpr int FILL_CHUNK = 8;   // items read at a time
constexpr int FILL_WORDS = sizeof(FillItem) / 4;

// an item out of LDS into scalar registers
__device__ __forceinline__ FillItem uniform_item(const int32_t* sh) {
    union { FillItem it; int32_t w[FILL_WORDS]; } u;
#pragma unroll
    for (int k = 0; k < FILL_WORDS; k++) u.w[k] = __builtin_amdgcn_readfirstlane(sh[k]);
    return u.it;
}

// one operation, over the threads of the workgroup
template <typename S, int NT>
__device__ __forceinline__ void fill_op(const FillArgs& a, const FillProg& pr, const FillItem& op, int tid) {
    const int nv = a.nv;
    const int ncell = op.ni * op.nj;

    if (op.type == FOP_COPY) {
        const S* qn = static_cast<const S*>(a.lvl_new[op.src_space]) + op.src_off + op.src_shift;
        const S* qo = static_cast<const S*>(a.lvl_old[op.src_space]) + op.src_off + op.src_shift;
        int mode = a.tmode[op.src_space];
        if (op.flags & FOPF_FORCE_NEW) mode = TIME_NEW;
        else if (op.flags & FOPF_FORCE_OLD) mode = TIME_OLD;
        else if (op.flags & FOPF_BIG) mode = a.big_old ? TIME_OLD : TIME_NEW;
        const double ai = a.alphai[op.src_space], ac = a.alphac[op.src_space];
        const S* q1 = mode == TIME_OLD ? qo : qn;
        with_dst<S>(a, pr, op, [&](const auto& dst) {
            if (mode != TIME_BLEND)
                copy_rect<NT>(op, dst, tid, nv, [&](int64_t k) { return (double)q1[k]; });
            else
                copy_rect<NT>(op, dst, tid, nv, [&](int64_t k) { return (double)qn[k] * ai + (double)qo[k] * ac; });
        });
    } else if (op.type == FOP_INTERP) {
        const Cells<const double> crs = src_cells(a, pr, op);
        const double dxf = a.hx[op.level], dyf = a.hy[op.level];
        const double dxc = a.hx[op.level - 1], dyc = a.hy[op.level - 1];
        const double xlow_coarse = a.xlower + op.iplo * dxc;
        const double ylow_coarse = a.ylower + op.jplo * dyc;
        const double ratiox = (double)op.ratx, ratioy = (double)op.raty;
        const unsigned char* mask = pr.masks + op.mask_off;
        with_dst<S>(a, pr, op, [&](const auto& dst) {
            Digits2<NT> u(tid, op.ni, 1 << 30);   // (i, j) of cell c; j does not wrap
            for (int c = tid; c < ncell; c += NT, u.step()) {
                if (mask[c]) continue;
                const int jf = u.j + 1, if_ = u.i + 1;   // 1-based
                const int j_coarse = (int)floor((double)(jf + op.jlo - 1) / ratioy) - op.jplo + 1;
                const double ycent_coarse = ylow_coarse + ((double)j_coarse - .5) * dyc;
                const double ycent_fine = a.ylower + ((double)(jf - 1 + op.jlo) + .5) * dyf;
                const double eta2 = (ycent_fine - ycent_coarse) / dyc;
                const int i_coarse = (int)floor((double)(if_ + op.ilo - 1) / ratiox) - op.iplo + 1;
                const double xcent_coarse = xlow_coarse + ((double)i_coarse - .5) * dxc;
                const double xcent_fine = a.xlower + ((double)(if_ - 1 + op.ilo) + .5) * dxf;
                const double eta1 = (xcent_fine - xcent_coarse) / dxc;
                const int64_t s = (int64_t)(j_coarse - 1) * crs.nrow + i_coarse - 1;
                const int64_t d = op.dst_shift + (int64_t)u.j * dst.nrow + u.i;
                int n = 0;
                for (; n + 4 <= nv; n += 4) interp_cell<4>(crs, dst, n, s, d, eta1, eta2);
                if (nv - n == 3) interp_cell<3>(crs, dst, n, s, d, eta1, eta2);
                else if (nv - n == 2) interp_cell<2>(crs, dst, n, s, d, eta1, eta2);
                else if (nv - n == 1) interp_cell<1>(crs, dst, n, s, d, eta1, eta2);
            }
        });
    } else if (op.type == FOP_FILVAL) {
        // src: the coarse patch grown by one coarse cell (ni x nj); dst: the
        // new grid; mask: its interior cells, row by row, 1 where an old
        // grid supplied the value (the reference's setflags test)
        const Cells<const double> crs = src_cells(a, pr, op);
        const int rx = op.ratx, ry = op.raty, mic = op.ni, mjc = op.nj;
        const int ncx = mic - 2, ncc = ncx * (mjc - 2), nx = ncx * rx;
        const unsigned char* mask = pr.masks + op.mask_off;
        with_dst<S>(a, pr, op, [&](const auto& dst) {
            for (int t = tid; t < ncc * nv; t += NT) {
                const int m = t / ncc, c = t - m * ncc;
                const int jc = c / ncx + 1, ic = c - (jc - 1) * ncx + 1;   // 0-based, 1..mic-2
                const double vc = crs.load(m, ic, jc);
                const double vxp = crs.load(m, ic + 1, jc), vxm = crs.load(m, ic - 1, jc);
                const double vyp = crs.load(m, ic, jc + 1), vym = crs.load(m, ic, jc - 1);
                double s1p = vxp - vc, s1m = vc - vxm;
                double slopex = fmin(fabs(s1p), fabs(s1m)) * copysign(1.0, vxp - vxm);
                if (s1m * s1p <= 0.0) slopex = 0.0;
                s1p = vyp - vc;
                s1m = vc - vym;
                double slopey = fmin(fabs(s1p), fabs(s1m)) * copysign(1.0, vyp - vym);
                if (s1m * s1p <= 0.0) slopey = 0.0;
                for (int jco = 1; jco <= ry; jco++) {
                    const double yoff = ((double)jco - 0.5) / (double)ry - 0.5;
                    const int jf = (jc - 1) * ry + jco - 1;                    // interior, 0-based
                    for (int ico = 1; ico <= rx; ico++) {
                        const double xoff = ((double)ico - 0.5) / (double)rx - 0.5;
                        const int if_ = (ic - 1) * rx + ico - 1;
                        if (!mask[(int64_t)jf * nx + if_])
                            dst.store(m, NGHOST + if_, NGHOST + jf, vc + xoff * slopex + yoff * slopey);
                    }
                }
            }
        });
    } else if (op.type == FOP_COPYBACK) {
        const Cells<const double> src = src_cells(a, pr, op);
        with_dst<S>(a, pr, op, [&](const auto& dst) {
            copy_rect<NT>(op, dst, tid, nv, [&](int64_t k) { return src.at(k); });
        });
    } else if (op.type == FOP_RING) {
        const Cells<const double> src = src_cells(a, pr, op);
        double* qc1d = a.lvl_reg[op.level] + op.dst_off;
        const int len = 2 * (op.ni - 2 + op.nj - 2);
        for (int t = tid; t < len * nv; t += NT) {
            const int idx = t / nv, m = t - idx * nv;
            qc1d[(int64_t)idx * nv + m] = src.at((int64_t)m * src.plane + ring_cell(idx, op.ni, op.nj));
        }
    } else if (op.type == FOP_COARSEN) {
        // coarsen.f:15-30: dst(i, j) = mean of src(2i..2i+1, 2j..2j+1)
        const Cells<const double> src = src_cells(a, pr, op);
        const Cells<double> dst{a.arena + op.dst_off, op.dst_nrow, op.dst_plane};
        for (int t = tid; t < ncell * nv; t += NT) {
            const int m = t / ncell, c = t - m * ncell;
            const int j = c / op.ni, i = c - j * op.ni;
            const double v = (src.load(m, 2 * i, 2 * j) + src.load(m, 2 * i + 1, 2 * j) +
                              src.load(m, 2 * i, 2 * j + 1) + src.load(m, 2 * i + 1, 2 * j + 1)) / 4.0;
            dst.store(m, i, j, v);
        }
    } else if (op.type == FOP_BC) {
        // sides in the reference's order, each complete before the next:
        // extrapolation (1) or mirrored (wall, 3).  One loop over the sides, not
        // four copies of its body: the FP32 kernel would keep its arguments in
        // scratch (1.2 KB a lane, six times the time).
        with_dst<S>(a, pr, op, [&](const auto& dst) {
            const int nrow = op.ni, ncol = op.nj;
#pragma unroll 1
            for (int side = 0; side < 4; side++) {
                if (side > 0) __syncthreads();
                // cells on a low side, the 1-based first column / row of a high one
                const int w = side == 0 ? op.bc[0] : (side == 1 ? op.bc[1] : (side == 2 ? op.bc[2] : op.bc[3]));
                const int kind = a.mthbc[side];
                if (w <= 0 || (kind != 1 && kind != 3)) continue;
                const bool high = side & 1, y = side >= 2, wall = kind == 3;
                const int n = high ? (y ? ncol : nrow) - w + 1 : w, from = high ? w - 1 : 0;
                const int mul = wall ? -1 : 0;
                const int add = wall ? (high ? 2 * w - 3 : 2 * w - 1) : (high ? w - 2 : w);
                BcSide sd{n, ncol, from, 0, mul, add, 1, 0, wall ? 1 : -1};
                if (y) sd = BcSide{nrow, n, 0, from, 1, 0, mul, add, wall ? 2 : -1};
                bc_side<NT>(dst, sd, tid, nv);
            }
        });
    }
}

// One workgroup per unit.  The unit's items are read into LDS FILL_CHUNK at a
// time.  Items of one stage do not wait for each other: each starts with the
// wave after the one that the item before it ended with, so that several small
// ones (a coarse patch out of four grids) run on different waves.
//
// Bound by latency, a unit's chain of dependent loads.  A level step of 28
// periodic advection grids took 4 launches of 3.6 us and now one of 7.9 us for
// the ghost fill and the finer level's saveqc together, a Euler one of 39 grids
// 17.6 -> 10.8 us, the three of a coarse step of 2,048 grids 271 -> 215 us.
template <typename S, int NT>
__global__ __launch_bounds__(NT) void fill_kernel(FillArgs a) {
    __shared__ int32_t sh[FILL_CHUNK * FILL_WORDS];
    const int tid = threadIdx.x;
    if (a.clear && blockIdx.x == 0)
        for (int64_t t = tid; t < a.nclear; t += NT) a.clear[t] = 0ull;
    const int first = a.prog[0].nunits;
    const bool second = (int)blockIdx.x >= first;
    const FillProg& pr = a.prog[second ? 1 : 0];
    const FillUnit un = pr.units[blockIdx.x - (second ? first : 0)];
    int rot = 0;
    for (int k0 = 0; k0 < un.n; k0 += FILL_CHUNK) {
        const int nk = un.n - k0 < FILL_CHUNK ? un.n - k0 : FILL_CHUNK;
        const int32_t* src = reinterpret_cast<const int32_t*>(pr.items + un.item0 + k0);
        if (k0 > 0) __syncthreads();
        for (int w = tid; w < nk * FILL_WORDS; w += NT) sh[w] = src[w];
        __syncthreads();
        for (int k = 0; k < nk; k++) {
            const FillItem op = uniform_item(sh + k * FILL_WORDS);
            if (op.sync) __syncthreads();
            const int t = (tid - rot) & (NT - 1);
            if (a.aux_mode) fill_aux_op<NT>(a, pr, op, t);
            else fill_op<S, NT>(a, pr, op, t);
            const int n = op.type == FOP_COPY ? op.ni * op.nj * a.nv : op.ni * op.nj;
            rot = (rot + ((n + 63) & ~63)) & (NT - 1);
        }
    }
}

hipError_t launch_fill(int esize, const FillArgs& a, hipStream_t st) {
    const int n = a.prog[0].nunits + a.prog[1].nunits;
    if (n <= 0) return hipSuccess;
    // many units: two waves each, so that more of them are resident (level 2 of
    // 2,048 grids, 11,845 units: 92 us at four waves, 82 at two, 108 at one);
    // few: the longest one decides (24 grids, 111 units: 21.6, 28.6, 39.8 us)
    const bool narrow = n >= 4096;
    if (esize == 8 && narrow)
        hipLaunchKernelGGL((fill_kernel<double, 128>), dim3(n), dim3(128), 0, st, a);
    else if (esize == 8)
        hipLaunchKernelGGL((fill_kernel<double, 256>), dim3(n), dim3(256), 0, st, a);
    else if (narrow)
        hipLaunchKernelGGL((fill_kernel<float, 128>), dim3(n), dim3(128), 0, st, a);
    else
        hipLaunchKernelGGL((fill_kernel<float, 256>), dim3(n), dim3(256), 0, st, a);
    return hipGetLastError();
}

}  // namespace amrgpu
