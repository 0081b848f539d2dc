// FP64 instantiations of the 3-D step: IEEE division and square root, built
// without FMA contraction (bit-for-bit the reference's FP64 arithmetic).
#include "sweep3_launch.hpp"
#include "sweep3_pass.hpp"

namespace amrgpu {

hipError_t launch_sweep3_f64(int solver, const Sweep3Args& a, hipStream_t st) {
    return sweep3_launch<double, ExactMath<double>>(solver, a, st);
}

hipError_t launch_update3_f64(int nv, double* q, const double* face, const Patch3* patches,
                              const Block3* blocks, int nblocks, double dtdx, double dtdy,
                              double dtdz, hipStream_t st) {
    return update3_launch<double>(nv, q, face, patches, blocks, nblocks, dtdx, dtdy, dtdz, st);
}

template <class Sol, int D>
static hipError_t pass3_solve(const Pass3Args& a, hipStream_t st) {
    if (a.nwaves == 0) return hipSuccess;
    hipLaunchKernelGGL((pass3_solve_kernel<Sol, double, D>), dim3((a.nwaves + 3) / 4), dim3(256), 0,
                       st, a);
    return hipGetLastError();
}

hipError_t launch_pass3_solve_f64(int solver, int d, const Pass3Args& a, hipStream_t st) {
    using Adv = Advection3<double, ExactMath<double>>;
    using Eul = Euler3<double, ExactMath<double>>;
    if (solver == SOLVER_ADVECTION)
        return d == 1 ? pass3_solve<Adv, 1>(a, st) : (d == 2 ? pass3_solve<Adv, 2>(a, st) : pass3_solve<Adv, 3>(a, st));
    if (solver == SOLVER_EULER)
        return d == 1 ? pass3_solve<Eul, 1>(a, st) : (d == 2 ? pass3_solve<Eul, 2>(a, st) : pass3_solve<Eul, 3>(a, st));
    return hipErrorInvalidValue;
}

hipError_t launch_pass3_face_f64(int nv, const Pass3Args& a, hipStream_t st) {
    if (a.nblocks == 0) return hipSuccess;
    const dim3 grid((a.nblocks + 7) / 8 * 8);
    if (nv == 5) hipLaunchKernelGGL((pass3_face_kernel<5, double>), grid, dim3(256), 0, st, a);
    else if (nv == 1) hipLaunchKernelGGL((pass3_face_kernel<1, double>), grid, dim3(256), 0, st, a);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

}  // namespace amrgpu
