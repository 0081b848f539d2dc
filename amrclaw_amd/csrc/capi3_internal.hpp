// capi3_internal.hpp -- state of the 3-D library (capi3.cpp) shared with the
// 3-D hierarchy code (capi3_amr.cpp).  Not part of the C ABI.
#pragma once
#include <hip/hip_runtime.h>
#include <vector>

#include "../../include/amrgpu3.h"
#include "sweep3.hpp"
#include "sweep3_pass.hpp"
#include "sweep3_tile.hpp"
#include "xfer.hpp"

namespace amrgpu {

// the fused step's tiles of a batch or level (sweep3_tile.hpp)
struct Tile3Plan {
    std::vector<Tile3> tiles;
    std::vector<Mark3> marks;     // each tile's marked faces, tile by tile
    size_t lds = 0;               // of the largest tile
    int xcd_start[TILE3_XCDS] = {}, xcd_count[TILE3_XCDS] = {};
};
// a marked face of a grid: lower face, normal to dir, of its 0-based cell
struct GridFace3 {
    int dir, x, y, z;
};
// the marked faces of a level's grids: their perimeters, if so, and others, each
// once
struct LevelFaces3 {
    bool perimeter = false;
    std::vector<std::vector<GridFace3>> others;
};
// device arrays of one fused step of a level
struct Fused3IO {
    const void* qin;              // time t, ghost cells filled
    void* qout;                   // time t + dt, with qin's ghost cells
    const Patch3* d_patches;
    int npatch;
    const Tile3* d_tiles;
    const Mark3* d_marks;
    const Tile3Plan* plan;
    void* face;                   // flux blocks: the marked faces are written
    unsigned long long* d_cfl;
};

// The two-pass FP64 step of a batch (sweep3_pass.hpp): the waves of each sweep,
// the face blocks, every grid's place in the work space, and the runs of grids
// that share it.  Built on first use, on the device until freed.
struct Pass3Run {
    int w0[3], w1[3], f0, f1;
};
struct Pass3Plan {
    bool built = false, ok = false;   // built and not ok: the phase kernels
    std::vector<Pass3Run> runs;
    int64_t ws_elems = 0;
    void* d_tables = nullptr;         // one allocation, these in it
    Pass3Wave* d_waves[3] = {};
    Block3* d_faces = nullptr;
    Pass3Ws* d_off = nullptr;
    void free() {
        hipFree(d_tables);
        *this = Pass3Plan();
    }
};

// device arrays of one step over a batch of grids
struct Step3IO {
    void* q;                      // solutions (compute precision)
    void* face;                   // flux blocks
    const Patch3* d_patches;
    Block3* d_blocks[4];          // x, y, z sweeps, update
    int nblocks[4];
    int npatch;
    unsigned long long* d_cfl;    // per-grid Courant number (double bits)
    const std::vector<Patch3>* patches;   // FP64: the host copies, and the batch's
    const std::vector<Block3>* blocks;
    Pass3Plan* pass;                      // two-pass plan (null: phase kernels)
};

bool ctx3_inited();
const amrgpu3_config& ctx3_cfg();
size_t ctx3_esize();
hipStream_t ctx3_stream();
int ctx3_plane_block();
XferRing& ctx3_xfer();
int ctx3_fail(int code, const char* fmt, ...);
hipError_t ctx3_h2d(void* dst, const void* src, size_t n);
hipError_t ctx3_d2h(void* dst, const void* src, size_t n);
// stepgrid.f (3-D) for every grid of the batch: clears d_cfl, launches the
// x-, y- and z-sweeps and the conservative update; esize 8 runs the FP64
// kernels whatever the library's precision (0: the library's)
int ctx3_step(const Step3IO& io, double dx, double dy, double dz, double dt, int esize = 0);
// the same step by the fused FP32 kernel (ctx3_fused: FP32 and the fused mode)
bool ctx3_fused();
int ctx3_step_fused(const Fused3IO& io, double dx, double dy, double dz, double dt);
void ctx3_plan_tiles(const std::vector<Patch3>& patches, const LevelFaces3& faces, Tile3Plan& plan);
// whether a level's step is better off fused than by its blocks' phase kernels
bool ctx3_fused_pays(const std::vector<Patch3>& patches, const std::vector<Block3>* blocks,
                     const Tile3Plan& plan);
// the work lists of a batch: per sweep (grid, plane block), largest first;
// update and totals (grid, 256 cells)
void ctx3_plan_blocks(const std::vector<Patch3>& patches, int plane_block,
                      std::vector<Block3> out[4]);
// releases the hierarchy state of capi3_amr.cpp (amrgpu3_finalize)
void amr3_release();

}  // namespace amrgpu
