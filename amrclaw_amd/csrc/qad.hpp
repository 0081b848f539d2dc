// qad.hpp -- the fine-side register kernel of a level step (qad + fluxad),
// templated on the Riemann solver: the library instantiates it for its own
// solvers (regs.hip) and a plug-in solver's translation unit for its solver
// (include/amrgpu_solver.hpp).  FP64 arithmetic in the reference's order:
// build with -ffp-contract=off.
#pragma once
#include <hip/hip_runtime.h>
#include <type_traits>
#include "lanes.hpp"
#include "regs.hpp"
#include "sweep.hpp"

namespace amrgpu {

// lane K of each group of G neighbouring lanes (2 or 4), read by the group
template <int G, int K>
__device__ __forceinline__ double group_lane(double v) {
    if constexpr (G == 1) return v;
    else if constexpr (G == 2) return dpp_move<K | K << 2 | (2 + K) << 4 | (2 + K) << 6>(v);
    else return dpp_move<K * 0x55>(v);
}
template <int G, int K = 0, class Add>
__device__ __forceinline__ void group_sum(int n, const Add& add) {
    if (K < n) add(std::integral_constant<int, K>{});
    if constexpr (K + 1 < G) group_sum<G, K + 1>(n, add);
}

// The fine-side register work of one level step, one register slot per
// group of G lanes, in the reference's order for that slot: qad.f:9-360 (the
// r Riemann problems between the saved coarse value and the fine grid's first
// ghost cells along one coarse segment, before the step) and then
// fluxad.f:36-92 (the r fine fluxes of the step through that segment).  `q` is
// the level's time-t array with its ghost cells; the fluxes come from the
// perimeter block the sweep wrote.
//
// Bound by latency: a level has some hundred to some ten thousand slots.  So
// the r problems of a slot are solved by neighbouring lanes at once and only
// their sum, the same additions in the same order, is serial: FP64 Euler, 39
// grids refined by 4 (about 1,000 slots), 20 us with one thread a slot, 8.0
// with four.
template <class Sol, typename S, int G>
__global__ __launch_bounds__(64) void finereg_kernel(QadArgs a, Physics ph) {
    constexpr int NV = Sol::NV, NW = Sol::NW;
    const int t = (blockIdx.x * 64 + threadIdx.x) / G, g = threadIdx.x % G;
    for (int i = blockIdx.x * 64 + threadIdx.x; i < a.ncfl; i += gridDim.x * 64) a.cfl_host[i] = a.cfl[i];
    if (t >= a.nitems) return;
    const QadItem it = a.items[t];
    const PatchDesc pd = a.patches[it.grid];
    const S* q = static_cast<const S*>(a.q) + pd.off;
    double* sv = a.reg + pd.reg_off;
    const double* qc = sv + (int64_t)NV * pd.lenbc;
    const double* per = a.reg + perim_offset(pd, NV);
    const bool xside = it.side == 1 || it.side == 3;
    const int r = xside ? a.raty : a.ratx;
    const double h = xside ? a.hy : a.hx;
    const int ixy = xside ? 1 : 2;
    // interface states: coarse is left on sides 1 and 4, right on 2 and 3
    const bool cleft = it.side == 1 || it.side == 4;
    // fluxad: perimeter side blocks 0 left, 1 top, 2 right, 3 bottom
    const int64_t side_off[4] = {0, (int64_t)NV * pd.my, (int64_t)NV * (pd.my + pd.mx),
                                 (int64_t)NV * (2 * pd.my + pd.mx)};
    const double* ps = per + side_off[it.side - 1];
    double acc[NV], qcv[NV];
#pragma unroll
    for (int m = 0; m < NV; m++) acc[m] = sv[(int64_t)(it.slot - 1) * NV + m];
#pragma unroll
    for (int m = 0; m < NV; m++) qcv[m] = qc[(int64_t)(it.slot - 1) * NV + m];
    for (int l0 = 0; l0 < (a.flux_form ? 0 : r); l0 += G) {
        const int f = (it.seg - 1) * r + min(l0 + g, r - 1) + 1;   // fine row (sides 1,3) or column
        int I, J;
        if (it.side == 1) { I = 0; J = f; }
        else if (it.side == 2) { I = f; J = pd.my + 1; }
        else if (it.side == 3) { I = pd.mx + 1; J = f; }
        else { I = f; J = 0; }
        const int64_t li = (int64_t)(J + 1) * pd.mitot + (I + 1);
        double ql[NV], qr[NV];
#pragma unroll
        for (int m = 0; m < NV; m++) {
            const double qf = (double)q[(int64_t)m * pd.plane + li];
            ql[m] = cleft ? qcv[m] : qf;
            qr[m] = cleft ? qf : qcv[m];
        }
        // aux of the two cells (qad.f:81-91, 160-185, 228-255, 300-330): the
        // coarse ring's value on the coarse side, on the fine side the ghost
        // cell's, or for an xleft / yleft component the fine face between
        // them (sides 1 and 4 take the first interior cell's; on sides 2
        // and 3 the face value is the ghost cell's, and it replaces the
        // coarse ring's value)
        constexpr int SNA = sol_naux<Sol>::value, NA = SNA > 0 ? SNA : 1;
        double al[NA], ar[NA];
        if constexpr (SNA > 0) {
            const double* fa = a.aux + pd.off * a.auxk;
            const double* ac = a.reg + aux_ring_offset(pd, NV) + (int64_t)(it.slot - 1) * a.naux;
            // the face cell on sides 1 (I = 1) and 4 (J = 1)
            const int64_t lface = it.side == 1 ? li + 1 : (it.side == 4 ? li + pd.mitot : li);
#pragma unroll
            for (int c = 0; c < SNA; c++) {
                const double vf = fa[(int64_t)c * pd.plane + li];
                const double vface = fa[(int64_t)c * pd.plane + lface];
                const bool face = (a.auxtype[c] == 1 && xside) || (a.auxtype[c] == 2 && !xside);
                if (cleft) {
                    al[c] = ac[c];
                    ar[c] = face ? vface : vf;
                } else {
                    al[c] = vf;
                    ar[c] = face ? vf : ac[c];
                }
            }
        }
        typename Sol::Cache cache = Sol::prep(ph, ixy, ql, qr);
        double wave[NW][NV], s[NW], amdq[NV], apdq[NV];
        Sol::rpn2(ph, ixy, ql, qr, SNA > 0 ? al : nullptr, SNA > 0 ? ar : nullptr, cache, wave, s,
                  amdq, apdq);
#pragma unroll
        for (int m = 0; m < NV; m++) {
            const double am = cleft ? amdq[m] * h * a.delt : -(amdq[m] * h * a.delt);
            const double ap = cleft ? apdq[m] * h * a.delt : -(apdq[m] * h * a.delt);
            group_sum<G>(r - l0, [&](auto k) {
                acc[m] = acc[m] + group_lane<G, decltype(k)::value>(am) +
                         group_lane<G, decltype(k)::value>(ap);
            });
        }
    }
    for (int l0 = 0; l0 < r; l0 += G) {
        const int f = (it.seg - 1) * r + min(l0 + g, r - 1) + 1;
#pragma unroll
        for (int m = 0; m < NV; m++) {
            const double v = ps[(int64_t)(f - 1) * NV + m] * a.delt * h;
            group_sum<G>(r - l0, [&](auto k) {
                acc[m] = acc[m] + group_lane<G, decltype(k)::value>(v);
            });
        }
    }
    if (g == 0) {
#pragma unroll
        for (int m = 0; m < NV; m++) sv[(int64_t)(it.slot - 1) * NV + m] = acc[m];
    }
}

template <class Sol, typename S>
void finereg_start(const QadArgs& a, const Physics& ph, hipStream_t st) {
    const int r = a.ratx > a.raty ? a.ratx : a.raty;
    const int lanes = r > 2 ? 4 : r;   // a slot
    const dim3 grid((unsigned)(((int64_t)a.nitems * lanes + 63) / 64));
    if (lanes == 4)
        hipLaunchKernelGGL((finereg_kernel<Sol, S, 4>), grid, dim3(64), 0, st, a, ph);
    else if (lanes == 2)
        hipLaunchKernelGGL((finereg_kernel<Sol, S, 2>), grid, dim3(64), 0, st, a, ph);
    else
        hipLaunchKernelGGL((finereg_kernel<Sol, S, 1>), grid, dim3(64), 0, st, a, ph);
}

template <class Sol>
hipError_t finereg_launch(int esize, const QadArgs& a, const Physics& ph, hipStream_t st) {
    if (a.nitems <= 0) return hipSuccess;
    if (esize == 8) finereg_start<Sol, double>(a, ph, st);
    else finereg_start<Sol, float>(a, ph, st);
    return hipGetLastError();
}

}  // namespace amrgpu
