// Declarations of the hydrodynamics (HD) stage kernels: 1D, 2D or 3D boxes,
// periodic, outflow or reflective sides, PLM + HLLC/HLL + RK2/RK3, FP64.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/gpluto_amd.h"
#include "common.hpp"

namespace gpl {

struct HdBox {
  int nx, ny, nz;     // active zones (1 along unused directions)
  int ncell;
  int dims;           // DIMENSIONS
  int lo[3], hi[3];   // side types per direction: GPL_PERIODIC / GPL_OUTFLOW / GPL_REFLECTIVE
  double dx, dy, dz;
};

// One launch: a stage of a 2D or 3D box, or a whole step of a 1D box.  The
// inputs and outputs are distinct buffers, except that a cell's own U may be
// read from Uout (or U0) and written there.
struct HdBufs {
  const double *Vin;  // [5][n] primitives at the start
  double *Vout;       // [5][n] primitives after it
  const double *Uin;  // [5][n] conserved state at the start of the stage
  const double *U0;   // [5][n] conserved state at the start of the step
  double *Uout;       // [5][n] conserved state after it (1D: another buffer than Uin)
  double *cdt_part;   // per-block maxima of C_dt (hd_blocks entries)
  uint32_t *err;
  ZoneRep zr[3];      // zone-by-zone reports of the launch's stages (zr[s].err null: off)
};

constexpr int HD_ARRIVED = 17*32;

// NextTimeStep inside the launch that ends a step (update_stage.cpp:422-425,
// next_time_step.cpp:80,123-125, main.cpp:458): see step_control in hd_kernels.hip.
struct HdStep {
  StepCtl *ctl;
  unsigned *arrived;  // [HD_ARRIVED] arrival counters of the launch; zero between launches
  double cfl, cfl_max_var;
  int advance;        // 0: inv_dt only
  int ends_step;      // this launch is the last of its step
};

// One stage of a 2D or 3D box.
void hd_launch_stage(const HdBufs &b, const HdBox &g, const HdStep &st, RKW w, int first_stage,
                     int want_dt, int limiter, int solver, double gamma, double small_rho,
                     double small_prs, hipStream_t s);
// A whole step (nst stages) of a 1D box.
void hd_launch_step1d(const HdBufs &b, const HdBox &g, const HdStep &st, int nst, int limiter,
                      int solver, double gamma, double small_rho, double small_prs, hipStream_t s);

// blocks of a launch (one C_dt partial maximum each); nst: the stages of a step
int hd_blocks(const HdBox &g, int nst);

}  // namespace gpl
