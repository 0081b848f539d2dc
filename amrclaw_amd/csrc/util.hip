// util.hip -- small device helpers used by the host library.
#include <hip/hip_runtime.h>
#include <cstdint>
#include "types.hpp"
#include "xfer.hpp"

namespace amrgpu {

// Fill kernel used instead of hipMemsetAsync so that the sequence stays
// valid inside captured graphs.
__global__ void fill_u64_kernel(unsigned long long* p, unsigned long long v, int64_t n) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

hipError_t launch_fill_u64(unsigned long long* p, unsigned long long v, int64_t n,
                           hipStream_t st) {
    if (n <= 0) return hipSuccess;
    int blocks = (int)((n + 255) / 256);
    hipLaunchKernelGGL(fill_u64_kernel, dim3(blocks), dim3(256), 0, st, p, v, n);
    return hipGetLastError();
}

// a few words from the device to pinned host memory
__global__ void copy_u64_kernel(unsigned long long* dst, const unsigned long long* src, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = src[i];
}

hipError_t launch_copy_u64(unsigned long long* dst, const unsigned long long* src, int n,
                           hipStream_t st) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(copy_u64_kernel, dim3((n + 255) / 256), dim3(256), 0, st, dst, src, n);
    return hipGetLastError();
}

// map[cell] = first + 1 of every record (MarchSvCell), on a cleared map
__global__ void sv_map_kernel(int32_t* map, const MarchSvCell* c, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) map[c[i].cell] = c[i].first + 1;
}

hipError_t launch_sv_map(int32_t* map, const MarchSvCell* c, int n, hipStream_t st) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(sv_map_kernel, dim3((n + 255) / 256), dim3(256), 0, st, map, c, n);
    return hipGetLastError();
}

// Pinned host slot (AoS, component fastest, FP64) <-> the grids' SoA arrays in
// storage precision, one element per thread: a wave moves 512 contiguous bytes
// of host memory.  Bound by PCIe (57 GB/s); the grid of a workgroup's first
// cell is found by bisection, the others' by walking on from it.
template <typename S, bool TO_DEV>
__global__ __launch_bounds__(256) void xfer_kernel(XferArgs a) {
    const int64_t first = a.e0 + (int64_t)blockIdx.x * 256;
    const int64_t e = first + threadIdx.x;
    XferGrid gr = a.one;
    const int64_t cell = e / a.nv;
    if (a.grids) {
        const int64_t c0 = first / a.nv;
        int lo = 0, hi = a.ngrids - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (a.grids[mid].cell0 <= c0) lo = mid;
            else hi = mid - 1;
        }
        while (lo + 1 < a.ngrids && a.grids[lo + 1].cell0 <= cell) lo++;
        gr = a.grids[lo];
    }
    if (e >= a.e1) return;
    const int64_t at = gr.off + (e - cell * a.nv) * gr.plane + (cell - gr.cell0);
    double* h = a.stage + (e - a.e0);
    if constexpr (TO_DEV) {
        const S v = (S)*h;
        static_cast<S*>(a.data)[at] = v;
        if (a.data2) static_cast<S*>(a.data2)[at] = v;
    } else {
        *h = (double)static_cast<const S*>(a.data)[at];
    }
}

hipError_t launch_xfer(bool to_dev, int esize, const XferArgs& a, hipStream_t st) {
    const int64_t n = a.e1 - a.e0;
    if (n <= 0) return hipSuccess;
    const dim3 grid((unsigned)((n + 255) / 256)), block(256);
    if (to_dev) {
        if (esize == 8) hipLaunchKernelGGL((xfer_kernel<double, true>), grid, block, 0, st, a);
        else hipLaunchKernelGGL((xfer_kernel<float, true>), grid, block, 0, st, a);
    } else {
        if (esize == 8) hipLaunchKernelGGL((xfer_kernel<double, false>), grid, block, 0, st, a);
        else hipLaunchKernelGGL((xfer_kernel<float, false>), grid, block, 0, st, a);
    }
    return hipGetLastError();
}

}  // namespace amrgpu
