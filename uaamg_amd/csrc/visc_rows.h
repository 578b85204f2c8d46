// The viscosity level above the coarsest as explicit rows, and its W-cycle
// visits in one launch (visc_rows_kernels.hip).
//
// A visit of that level is 24 dependent colour passes, a residual, a
// restriction, the coarsest solve and a prolongation over some thousand DOFs:
// as launches of about 5 us each nearly all of its time is launch and memory
// latency. Here the level's DOFs are rows sorted by (channel, colour), a row
// holding its 14 couplings, 1/diag, diag and the 14 neighbours' row numbers
// (96 bytes, read with wide coalesced loads), and one workgroup runs the
// whole visit with x in LDS.
#pragma once

#include "viscosity_kernels.h"

namespace uaamg {

struct ViscRowsView {
    int32_t n = 0;             // rows
    int32_t np = 0;            // row stride of coef and idx
    int32_t nc = 0;            // rows of the coarsest level
    int32_t start[7] = {};     // first row of group 2 * channel + (0 red, 1 black); start[6] = n
    float4* coef = nullptr;    // [4][np]: the 14 couplings in the operator's order, 1/diag, diag
    uint4* idx = nullptr;      // [2][np]: 16-bit row numbers of the 14 neighbours (n: none), the coarse row (nc: none)
    int32_t* pos = nullptr;    // [n] position in the level vector
    int32_t nsteps = 0;        // steps of one sweep
    int2* steps = nullptr;     // [2][nsteps]: the steps of an XYZ and of a ZYX sweep (visc_rows_steps)
    float* b = nullptr;        // [n] scratch: right-hand side by row
    float* r = nullptr;        // [n + 1] scratch: residual by row (the last stays 0)
    uint4* child = nullptr;    // [nc] 16-bit row numbers of a coarse row's eight children (n: none)
};

// Rows the kernel takes (x and the coarsest vector fit a workgroup's LDS, row
// numbers fit 16 bits). A colour pass over N rows streams 100 N / 6 bytes
// through one CU, so its time grows with N while the launched passes stay at
// about 5 us. Whole solves, rows / launches, with this level at 7428 rows: 677
// / 993 us, 11.9k: 1109 / 1507, 15.9k: 1379 / 1561, 19.0k: 1467 / 1622, 22.5k:
// 1662 / 1714, 25.0k: 1761 / 1730.
constexpr int64_t kViscRowsMax = 20480;

// Threads of a visit's workgroup and rows per step: 1024 where the coarsest
// rows fit 128 registers a thread (two of them), 512 beyond.
constexpr int kViscRowsWideNc = 1024;
inline int visc_rows_step(int nc) { return nc <= kViscRowsWideNc ? 1024 : 512; }

// A step is up to that many rows of one group: {first row, the group's end,
// plus kViscStepLast on a pass's last step (a barrier follows)}.
constexpr int kViscStepLast = 1 << 30;
constexpr int kViscMaxSteps = int(kViscRowsMax) / 512 + 6;

// allows the visit kernels the LDS of the largest level; before the first visit on a device
hipError_t visc_rows_init();

// device bytes of the view's arrays for n rows over nc coarse rows
size_t visc_rows_bytes(int64_t n, int64_t nc);

// Fills the arrays of R (allocated, R.n .. R.start set): F the level, Cl the
// coarsest level with DOF positions cpos. base: [nleaf_dof * 3][2], the first
// row of the brick's red and black DOFs. fmap / cmap: scratch of one float
// per brick entry of F and of Cl. Stream-ordered; create time only.
hipError_t launch_visc_rows_build(const ViscLevelView& F, const ViscLevelView& Cl, const ViscRowsView& R,
                                  const int32_t* base, const int32_t* cpos, float* fmap, float* cmap, hipStream_t s);

// nvisits visits of the level (the first from a zero guess when precon, else
// from x), with right-hand side b and the coarsest solves inside; the result
// goes to x. view (of n rows) and cview (of nc) are in device memory.
hipError_t launch_visc_rows_visit(const ViscRowsView* view, const ViscCoarsestView* cview, int n, int nc,
                                  const float* b, float* x, bool precon, int nvisits, hipStream_t s);
hipError_t launch_visc_rows_visit(const ViscRowsView* view, const ViscCoarsestView* cview, int n, int nc,
                                  const bf16* b, bf16* x, bool precon, int nvisits, hipStream_t s);

}  // namespace uaamg
