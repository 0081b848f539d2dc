// regs.hip -- coarse-fine register kernels: qad + fluxad (the fine side of
// the registers), upbnd (reflux into coarse cells), the averaging of fine
// cells onto the coarse cells they cover and the conservation total.  FP64 arithmetic in the
// reference's order; built with -ffp-contract=off.
#include <hip/hip_runtime.h>
#include "qad.hpp"
#include "regs.hpp"
#include "sweep.hpp"

namespace amrgpu {

// components m0 .. m0 + C - 1 of upbnd.f:62-124 for one coarse cell, its
// register slots in list order
template <int C, typename S>
__device__ __forceinline__ void upbnd_cell(const UpdateArgs& a, const UpbndCell& c, S* q, int plane,
                                           double capa, int m0) {
    double v[C];
#pragma unroll
    for (int k = 0; k < C; k++) v[k] = (double)q[(int64_t)(m0 + k) * plane];
    for (int e = c.e0; e < c.e1; e++) {
        const UpbndEntry en = a.entries[e];
        const double* svd = a.reg + a.fine_patches[en.kid].reg_off + (int64_t)a.nv * (en.lkid - 1) + m0;
        const double sgnm = a.mcapa > 0 ? en.sgnm / capa : en.sgnm;
#pragma unroll
        for (int k = 0; k < C; k++) v[k] = v[k] + sgnm * svd[k] / a.area;
    }
#pragma unroll
    for (int k = 0; k < C; k++) q[(int64_t)(m0 + k) * plane] = (S)v[k];
}

// components m0 .. m0 + C - 1 of update.f:95-177 for one coarse cell, the mean
// of its fine cells, which start at qf (R > 0: R x R of them); all loads of
// the components go out before the first store.  capf: the fine cells'
// capacities, which weigh them (update.f:147-161), or null.
template <int C, int R, typename S>
__device__ __forceinline__ void average_cell(const UpdateArgs& a, S* q, int planec, const S* qf, int planef,
                                             int mitotf, const double* capf, double div, int m0) {
    const int rx = R > 0 ? R : a.ratx, ry = R > 0 ? R : a.raty;
    double v[C];
#pragma unroll
    for (int k = 0; k < C; k++) v[k] = 0.0;
#pragma unroll
    for (int jco = 0; jco < ry; jco++)
#pragma unroll
        for (int ico = 0; ico < rx; ico++) {
            const int64_t lf = (int64_t)jco * mitotf + ico;
#pragma unroll
            for (int k = 0; k < C; k++) {
                const double f = (double)qf[(int64_t)(m0 + k) * planef + lf];
                v[k] = v[k] + (capf ? f * capf[lf] : f);
            }
        }
#pragma unroll
    for (int k = 0; k < C; k++) q[(int64_t)(m0 + k) * planec] = (S)(v[k] / div);
}

// update.f:61-177: workgroups of upbnd (one coarse cell a thread; cells a finer
// grid covers are not in the list) and of averaging (one tile of coarse cells
// each) in one launch, as they write different cells.
//
// Averaging is bound by memory: neighbouring threads take neighbouring coarse
// cells of a row.  2,048 grids of 5,583 FP64 cells (457 MB read and written),
// 270,000 refluxed cells: 89 us, 5.1 TB/s (255 with columns of cells to
// neighbouring threads and a search for the block in each).
template <typename S>
__global__ __launch_bounds__(256) void update_kernel(UpdateArgs a, int upbnd_groups) {
    const int nv = a.nv;
    int m = 0;
    if ((int)blockIdx.x < upbnd_groups) {
        const int t = blockIdx.x * 256 + threadIdx.x;
        if (t >= a.ncells) return;
        const UpbndCell c = a.cells[t];
        const PatchDesc pd = a.patches[c.grid];
        const int64_t li = (int64_t)c.j * pd.mitot + c.i;
        S* q = static_cast<S*>(a.q) + pd.off + li;
        // capacity: the sign divided by the coarse cell's capacity (upbnd.f:104-108)
        const double capa =
            a.mcapa > 0 ? a.aux_c[pd.off * a.auxk + (int64_t)(a.mcapa - 1) * pd.plane + li] : 1.0;
        for (; m + 4 <= nv; m += 4) upbnd_cell<4, S>(a, c, q, pd.plane, capa, m);
        if (nv - m == 3) upbnd_cell<3, S>(a, c, q, pd.plane, capa, m), m += 3;
        for (; m < nv; m++) upbnd_cell<1, S>(a, c, q, pd.plane, capa, m);
        return;
    }
    const AvgTile tile = a.tiles[blockIdx.x - upbnd_groups];
    const AvgBlock b = a.blocks[tile.block];
    const int c = tile.c0 + (int)threadIdx.x;
    if (c >= b.ni * b.nj) return;
    const int cj = c / b.ni, ci = c - cj * b.ni;
    const PatchDesc pc = a.patches[b.grid];
    const PatchDesc pf = a.fine_patches[b.kid];
    const int64_t lic = (int64_t)(b.cj0 + cj) * pc.mitot + (b.ci0 + ci);
    const int64_t lif = (int64_t)(b.fj0 + cj * a.raty) * pf.mitot + (b.fi0 + ci * a.ratx);
    S* q = static_cast<S*>(a.q) + pc.off + lic;
    const S* qf = static_cast<const S*>(a.qf) + pf.off + lif;
    const double totrat = (double)(a.ratx * a.raty);
    if (a.mcapa > 0) {
        const double* capf = a.aux_f + pf.off * a.auxk + (int64_t)(a.mcapa - 1) * pf.plane + lif;
        const double capc = a.aux_c[pc.off * a.auxk + (int64_t)(a.mcapa - 1) * pc.plane + lic];
        for (; m < nv; m++)
            average_cell<1, 0, S>(a, q, pc.plane, qf, pf.plane, pf.mitot, capf, totrat * capc, m);
        return;
    }
    const bool two = a.ratx == 2 && a.raty == 2;
    for (; m + 4 <= nv; m += 4) {
        if (two) average_cell<4, 2, S>(a, q, pc.plane, qf, pf.plane, pf.mitot, nullptr, totrat, m);
        else average_cell<4, 0, S>(a, q, pc.plane, qf, pf.plane, pf.mitot, nullptr, totrat, m);
    }
    if (two && nv - m == 3) {
        average_cell<3, 2, S>(a, q, pc.plane, qf, pf.plane, pf.mitot, nullptr, totrat, m);
        m += 3;
    }
    for (; m < nv; m++) {
        if (two) average_cell<1, 2, S>(a, q, pc.plane, qf, pf.plane, pf.mitot, nullptr, totrat, m);
        else average_cell<1, 0, S>(a, q, pc.plane, qf, pf.plane, pf.mitot, nullptr, totrat, m);
    }
}

// a lane's double, read by the whole wave (lane index uniform)
__device__ __forceinline__ double lane_value(double v, int k) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffll), k);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), k);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// conck.f:36-63 in the reference's order: one wave walks the grids in level
// order, rows j, then columns i; each lane loads one cell of a 64-cell chunk
// of the row (coalesced) and the chunk is added lane by lane in ascending i
// by a loop uniform over the wave, so the total is the reference's
// sequential FP64 sum bit for bit.  A diagnostic: one wave, latency-bound.
template <typename S>
__global__ __launch_bounds__(64) void conck_kernel(const PatchDesc* patches, int npatch,
                                                   const void* qv, double* out, const double* aux,
                                                   int mcapa, int auxk) {
    const int lane = threadIdx.x;
    double tot = 0.0;
    for (int p = 0; p < npatch; p++) {
        const PatchDesc pd = patches[p];
        const S* q = static_cast<const S*>(qv) + pd.off;
        // capacity: q(1) * capa (conck.f:56-60)
        const double* ca = mcapa > 0 ? aux + pd.off * auxk + (int64_t)(mcapa - 1) * pd.plane : nullptr;
        for (int j = 0; j < pd.my; j++) {
            const S* row = q + (int64_t)(j + NGHOST) * pd.mitot + NGHOST;
            const double* crow = ca ? ca + (int64_t)(j + NGHOST) * pd.mitot + NGHOST : nullptr;
            for (int i0 = 0; i0 < pd.mx; i0 += 64) {
                const int n = min(64, pd.mx - i0);
                const double v = lane < n ? (crow ? (double)row[i0 + lane] * crow[i0 + lane]
                                                  : (double)row[i0 + lane]) : 0.0;
                for (int k = 0; k < n; k++) tot = tot + lane_value(v, k);
            }
        }
    }
    if (lane == 0) out[0] = tot;
}

hipError_t launch_conck(int esize, const PatchDesc* patches, int npatch, const void* q,
                        double* out, hipStream_t st, const double* aux, int mcapa, int auxk) {
    if (npatch <= 0) return hipSuccess;
    if (esize == 8)
        hipLaunchKernelGGL(conck_kernel<double>, dim3(1), dim3(64), 0, st, patches, npatch, q, out,
                           aux, mcapa, auxk);
    else
        hipLaunchKernelGGL(conck_kernel<float>, dim3(1), dim3(64), 0, st, patches, npatch, q, out,
                           aux, mcapa, auxk);
    return hipGetLastError();
}

hipError_t launch_finereg(int solver, int esize, const QadArgs& a, const Physics& ph, hipStream_t st) {
    switch (solver) {
    case SOLVER_ADVECTION: return finereg_launch<Advection<double>>(esize, a, ph, st);
    case SOLVER_ACOUSTICS: return finereg_launch<Acoustics<double>>(esize, a, ph, st);
    case SOLVER_EULER: return finereg_launch<EulerRoe<double>>(esize, a, ph, st);
    case SOLVER_VCADV: return finereg_launch<VcAdvection<double>>(esize, a, ph, st);
    default: return hipErrorInvalidValue;
    }
}

hipError_t launch_update(int esize, const UpdateArgs& a, hipStream_t st) {
    const int up = (a.ncells + 255) / 256;
    if (up + a.ntiles <= 0) return hipSuccess;
    const dim3 grid((unsigned)(up + a.ntiles));
    if (esize == 8)
        hipLaunchKernelGGL(update_kernel<double>, grid, dim3(256), 0, st, a, up);
    else
        hipLaunchKernelGGL(update_kernel<float>, grid, dim3(256), 0, st, a, up);
    return hipGetLastError();
}

}  // namespace amrgpu
