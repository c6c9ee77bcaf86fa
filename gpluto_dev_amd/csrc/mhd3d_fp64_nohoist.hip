// The FP64 kernels that are faster without the compiler's machine-level loop
// hoisting: the RMHD sweeps, the van Leer sweeps and the edge EMFs.
//
// It moves the 64-bit literals of a march (two s_mov each, more than a hundred
// of them here) out of the loop, past the scalar registers there are, and
// stores the rest lane by lane in vector registers, which then overflow too:
// RMHD HLL z march 256 vector registers with 14 spilled against 224 without any,
// y 248 against 200.  us per launch
// with and without: van Leer y march of 75x90x61 35.1 -> 32.2, EMFs of 256^3
// 582 -> 573 and of RMHD 128^3 88 -> 80.  The MC sweeps of ideal MHD have the
// registers and stay with it (256^3 y march 709 with, 737 without).
#define GPL_MHD3D_NOHOIST
#include "mhd3d_kernels.hpp"

namespace gpl {
void mhd3d_launch_nohoist(int which, const Mhd3dBufs<double> &b, const Box3 &g, const StepCtl *ctl, RKW w,
                          int first_stage, int want_dt, int limiter, int solver, double gamma, hipStream_t s)
{
  const bool mc = limiter == MC_LIM;
  if (which == K_EMF) {
    if (mc) launch_emf<double, MC_LIM>(b, g, solver, s);
    else    launch_emf<double, VANLEER_LIM>(b, g, solver, s);
  } else if (b.phys == 1) {
    if (mc) launch_sweep_by<double, MC_LIM, 1>(which, b, g, ctl, w, first_stage, want_dt, solver, gamma, s);
    else    launch_sweep_by<double, VANLEER_LIM, 1>(which, b, g, ctl, w, first_stage, want_dt, solver, gamma, s);
  } else {
    launch_sweep_by<double, VANLEER_LIM, 0>(which, b, g, ctl, w, first_stage, want_dt, solver, gamma, s);
  }
}
}
