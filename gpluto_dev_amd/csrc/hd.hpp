// Declarations of the hydrodynamics (HD) stage kernels: 1D, 2D or 3D boxes,
// periodic, outflow or reflective sides, PLM + HLLC/HLL + RK2/RK3, FP64.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <cmath>

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
  double *dU;         // [5][n] flux divergence and [n] C_dt of the directions so far
  double *Cdt;        // (hd_launch_sweep only)
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

// One direction of a stage of a 2D or 3D box that takes its stages by direction
// (hd_by_direction), 0 .. dims-1 in turn; launch_dt ends the step.
void hd_launch_sweep(int dir, const HdBufs &b, const HdBox &g, const StepCtl *ctl, RKW w, int first_stage,
                     int want_dt, int limiter, int solver, double gamma, double small_rho,
                     double small_prs, hipStream_t s);

constexpr int kHdCols = 64, kHdRows = 7;      // cells of a 3D block's planes

// Planes per block of a 3D march, rows per wave of a 2D one; the longest of
// lengths within 5%.
//  3D: the shortest rounds of one block per CU, a segment costing its planes and
//    about half of one more for its first face (128x96x112, us a stage: 149 at one
//    plane, 123 at 8, 103 at the 13 of one round).
//  2D: a wave solves 2 L + 1 faces in turn behind about five faces' worth of
//    launch and first loads; more waves than SIMDs cost about the root of their
//    number (511x333, us a stage at L = 1, 2, 3, 4, 8: 22, 21, 19, 23, 33;
//    512^2: 28, 26, 24, 28, 31; 2000x1800: 255, 205, 195, 195, 194).
inline int hd_march_cells(const HdBox &g)
{
  if (g.dims == 1) return 1;
  const bool d3 = g.dims == 3;
  const long long across = d3 ? (long long)((g.nx + kHdCols - 1)/kHdCols)*((g.ny + kHdRows - 1)/kHdRows) : (g.nx + 62)/63;
  const int n = d3 ? g.nz : g.ny;
  int best = 32;
  double tbest = 0.0;
  for (int l = 32; l >= 1; l--) {
    const long long items = across*((n + l - 1)/l);
    const double per = (double)items/1024;
    const double t = d3 ? (double)((items + 255)/256)*(l + 0.5) : (2*l + 6)*(per > 1.0 ? std::sqrt(per) : 1.0);
    if (l == 32 || t < 0.95*tbest) { best = l; tbest = t; }
  }
  return best;
}

// Whether a 2D or 3D box takes its stages direction by direction (k_hd_sweep).  The
// one-launch stages hold 64 x 7 columns of the x-y plane per block (3D) or 63
// columns per wavefront (2D); a box narrower than that leaves their lanes idle and
// makes their marches long.  Both sides in us a stage, as measured: a block's plane
// costs 7 in 3D; a row costs two solves, 1.4 together, in 2D, where wavefronts
// beyond one per SIMD add up to the power 2/3; the other way is launches (17, 13),
// then 0.125 and 0.085 per 1000 cells.  Stage, us, one launch / by direction:
// 8x16x1500 127 / 37, 20x100x100 50 / 42, 40x33x200 39 / 52, 64x8x24 16 / 17;
// 16x4096 20 / 16, 24x32768 93 / 81, 32x4096 20.5 / 21, 62x512 11.5 / 15.
inline bool hd_by_direction(const HdBox &g)
{
  if (g.dims == 1 || (g.dims == 2 && g.nx > 63)) return false;
  const int l = hd_march_cells(g);
  const double kcells = 1e-3*g.ncell;
  if (g.dims == 2) {
    const double per = (double)((g.ny + l - 1)/l)/1024, cells = 11.0 + 0.085*kcells;
    return (cells > 13.0 ? cells : 13.0) < 1.5*(2*l + 6)*(per > 1.0 ? std::cbrt(per*per) : 1.0);
  }
  const long long items = (long long)((g.nx + kHdCols - 1)/kHdCols)*((g.ny + kHdRows - 1)/kHdRows)*((g.nz + l - 1)/l);
  const double stage = 5.0 + 7.5*(double)((items + 255)/256)*(l + 0.5), cells = 15.0 + 0.125*kcells;
  return (cells > 17.0 ? cells : 17.0) < stage;
}

// threads of a block of a direction's sweep
inline int hd_sweep_block(const HdBox &g) { return g.ncell <= (1 << 16) ? 64 : 256; }

// threads of a 1D block
inline int hd_block1d(const HdBox &g) { return g.nx <= (1 << 14) ? 64 : 256; }

// blocks of a launch (one C_dt partial maximum each); nst: the stages of a step
inline int hd_blocks(const HdBox &g, int nst)
{
  if (g.dims == 1) {
    const int own = hd_block1d(g) - 4*nst;
    return (g.nx + own - 1)/own;
  }
  if (hd_by_direction(g)) return (int)(((long long)g.ncell + hd_sweep_block(g) - 1)/hd_sweep_block(g));
  const int l = hd_march_cells(g);
  if (g.dims == 2) return (((g.nx + 62)/63)*((g.ny + l - 1)/l) + 3)/4;
  return ((g.nx + kHdCols - 1)/kHdCols)*((g.ny + kHdRows - 1)/kHdRows)*((g.nz + l - 1)/l);
}

}  // namespace gpl
