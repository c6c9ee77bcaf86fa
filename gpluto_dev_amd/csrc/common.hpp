// Declarations shared by every stage-update engine: the device-resident
// time-step control block, RK stage weights, kernel ids for timing, and the
// dt reduction kernel.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace gpl {

// Device-resident time-step control: the step loop never needs the host.
struct StepCtl {
  double dt;       // current time step (timeStep::dt)
  double time;     // timeStep::time
  double inv_dt;   // timeStep::invDt_hyp of the last stage-1 update
  long long nstep;
};

// RK weights of one stage: U = w0*U0 + w1*U + wR*R  (rk_step.cpp:20-51)
struct RKW { double w0, w1, wR; };

// Every kernel the library launches, for the per-kernel timing tables.
enum KernelId { K_SWEEP_X = 0, K_SWEEP_Y, K_SWEEP_Z, K_RHS, K_SWEEPX_F, K_SWEEPY_F, K_SWEEPZ_F,
                K_EMF, K_FINISH, K_DT, K_HD_X, K_HD_Y, K_HD_Z, K_SWEEPXY_F, K_COUNT };

// Zone-by-zone error reports: the reference's Data::err (Src/structs.hpp:678)
// as ConsToPrim3D writes it in every zone it converts (Src/mappers3D.cpp:115,
// 121, 173-176) and the flagged-zone counts Where() adds to Data::err_count
// (Src/debug_tools.cpp:587-593).  err is this stage's array over the device
// cells, count this stage's counter, total the running count; err == nullptr
// when the reports are off.
struct ZoneRep {
  uint32_t *err;
  unsigned long long *count, *total;
};

__device__ __forceinline__ void zone_report(const ZoneRep &z, size_t c, uint32_t e)
{
  if (!z.err) return;
  z.err[c] = e;
  if (e) { atomicAdd(z.count, 1ull); atomicAdd(z.total, 1ull); }
}

// OR e into a domain's error bits.  Only bits that are not there yet take an
// atomic: where a whole region reports (floors, or a run that has gone to NaN)
// every wavefront would otherwise queue on the one word, which cost more than
// the stage itself (64^3, every zone reporting: 373 us a step with an atomic
// per wavefront, 159 us with the load).
__device__ __forceinline__ void report_bits(uint32_t *err, uint32_t e)
{
  if (e && (__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & e) != e) atomicOr(err, e);
}

// counts[0..2] = 0 at the start of a step (Src/main.cpp:423); a kernel, so a
// captured step replays it
void launch_zone_reset(unsigned long long *counts, hipStream_t s);

// Cells per lane of a march along an extent of n cells, for `across` cells in
// the plane it crosses.  A lane solves L + 1 faces for its L cells, one after
// the other, and loads its window first (about half a face's time).  Long
// marches waste the fewest solves; on a small box they leave most of the chip
// idle.
//
// FP64: one wavefront's Riemann solve already fills a SIMD's issue slots about
// as well as two, so a launch takes ceil(blocks / CUs) (L + 1.5).  The shortest
// such time over L <= 16 is taken, L = 16 unless another is 5% shorter (a box
// that streams from HBM gains nothing from the model).  y and z march, us at
// L = 16 -> at the rule's L: 64^3 54 + 57 -> 23 + 25 (L = 4), RMHD HLLD
// 50x44x38 276 + 285 -> 59 + 59 (L = 2), 16^3 52 + 53 -> 11 + 12 (L = 1);
// 128^3 100 + 106 against 108 + 113 at 8 and 117 + 127 at 4.
//
// FP32: four wavefronts per SIMD hide the load latency, so L is the largest of
// 8, 4, 2, 1 that leaves 8192 wavefronts (512 for the last halving), and 16 where
// that leaves `waves16`, which differs by kernel: the z march loses at 16 even on
// large boxes (never: 0), the other two win once the chip is full (kWavesXY,
// kWaves2D).  z march and x+y kernel, us at 16 -> rule: 64^3 48 + 64 -> 16 + 20
// (L = 2), 128^3 81 + 110 -> 82 + 90 (L = 4), 192^3 280 + 270 -> 250 + 263 (L = 8).
// x+y kernel at 8 / 16: 208^3 379 / 378, 224^3 430 / 439, 400x300x100 685 / 698, 256^3
// 572 / 566, 320^3 2202 / 2130; z march 256^3 564 / 590, 320^3 1131 / 1168.
//
// The 2D y march: 512^2 FP64 67 -> 26 us (L = 4), 306x195 FP32 54 -> 9.5 (L = 1).
// FP32 step at the other lengths' best of 4 and 8 / at 16: 1024^2 219 / 246, 1500x1400
// 501 / 508, 2000x1500 658 / 649, 300x8000 579 / 570, 3000^2 2061 / 2000.
constexpr long long kWavesXY = 16384, kWaves2D = 2304;
inline int march_length(bool fp64, long long across, int n, long long waves16)
{
  if (!fp64) {
    if (waves16 && across*((n + 15)/16)/64 >= waves16) return 16;
    int l = 8;
    while (l > 1 && across*((n + l - 1)/l)/64 < (l > 2 ? 8192 : 512)) l /= 2;
    return l;
  }
  constexpr int kCUs = 256, kBlock = 256;
  int best = 16;
  double tbest = 0.0;
  for (int l = 16; l >= 1; l--) {
    const long long blocks = (across*((n + l - 1)/l) + kBlock - 1)/kBlock;
    const double t = (double)((blocks + kCUs - 1)/kCUs)*(l + 1.5);
    if (l == 16 || t < 0.95*tbest) { best = l; tbest = t; }
  }
  return best;
}

// Whole columns per block for a y or z sweep of columns of n cells (FP64), or 0
// for the march of `march` cells.  A block of c columns solves every face once,
// c*n lanes side by side; rows of fewer than 4 cells (32 bytes) waste too much of
// each cache line and blocks over 256 lanes stall on their barriers (64^3, y + z:
// 17 + 20 us with 4 columns, 21 + 24 with 2 and with 8).  In units of one wavefront's
// solve the busiest CU takes ceil(blocks / CUs) ceil(c n / 64) against the march's
// (L + 1.5) per wavefront; the columns are taken where that is 10% less.  Step, us,
// march -> columns: MHD HLLD 16^3 62 -> 55, 64^3 152 -> 138, 128x64^2 266 -> 242,
// 128^2x64 (ratio 0.91, refused) 500 -> 516; RMHD HLL 64^3 245 -> 199, HLLD 64^3
// 504 -> 376, HLLD van Leer RK3 50x44x38 455 -> 314.
//
// That holds while the rows of 4 to 8 cells are still cached when the next column
// block reads the rest of their lines: across z, whose rows lie a plane apart, less
// far than across y, and for RMHD's dearer solves further.  Above `full` cells a
// fifth is added, above `most` the columns are refused.  Sweep, us, columns / march:
// MHD z 192^2x20 (0.74 M cells) 55 / 52, 160^2x32 (0.82 M) 60 / 66, 192^2x28 (1.03 M)
// 84 / 74, 256^2x24 (1.6 M) 116 / 98, 400x300x20 (2.4 M) 206 / 139; MHD y 500x24x100 (1.2 M)
// 66 / 73, 256x24x256 (1.6 M) 93 / 82, 384x16x384 (2.4 M) 159 / 123; RMHD HLL z 192^2x32
// (1.2 M) 125 / 135, 256^2x24 167 / 158, y 384x16x384 199 / 214.
struct ColumnLimit { long long full, most; };
inline ColumnLimit column_limit(bool rmhd, bool z)
{
  if (rmhd) return z ? ColumnLimit{1300000, 1300000} : ColumnLimit{1LL << 40, 1LL << 40};
  return z ? ColumnLimit{650000, 850000} : ColumnLimit{1000000, 1300000};
}
inline int sweep_columns(int nx, int na, int n, int march, const ColumnLimit &lim)
{
  constexpr int kCUs = 256, kBlock = 256;
  const long long cells = (long long)nx*na*n, mb = ((long long)nx*na*((n + march - 1)/march) + kBlock - 1)/kBlock;
  if (cells > lim.most) return 0;
  const double far = cells > lim.full ? 1.2 : 1.0;
  double best = 0.9*(double)((mb + kCUs - 1)/kCUs)*(kBlock/64)*(march + 1.5);
  int x = 0;
  for (int c = 4; c <= 8 && c*n <= kBlock; c++) {
    const long long blocks = (long long)((nx + c - 1)/c)*na;
    const double t = far*(double)((blocks + kCUs - 1)/kCUs)*((c*n + 63)/64);
    if (t < best) { best = t; x = c; }
  }
  return x;
}

// Rows per block of the 3D x sweep: the fewest whose wavefronts on the busiest CU,
// ceil(blocks / CUs) ceil(rows nx / 64), are 5% fewer than with fewer rows, blocks
// of at most 256 lanes.  x sweep, us, one row -> this many: 20x70x90 20 -> 12
// (3 rows), 72x80x66 27 -> 22 (3), 79x94x65 (75x90x61 with ghosts) 32 -> 26 (3),
// 96^3 43 -> 38 (2).
inline int sweep_rows(int nx, long long nrows)
{
  constexpr int kCUs = 256, kBlock = 256;
  int rows = 1;
  double best = 0.0;
  for (int m = 1; m == 1 || m*nx <= kBlock; m++) {
    const long long blocks = (nrows + m - 1)/m;
    const double t = (double)((blocks + kCUs - 1)/kCUs)*((m*nx + 63)/64);
    if (m == 1 || t < 0.95*best) { best = t; rows = m; }
  }
  return rows;
}

// invDt_hyp = max over the partial maxima / DIMENSIONS; with advance != 0
// also NextTimeStep and time += dt on the device.
void launch_dt(const double *part, int nparts, double dims, StepCtl *ctl, double cfl,
               double cfl_max_var, int advance, hipStream_t s);

}  // namespace gpl
