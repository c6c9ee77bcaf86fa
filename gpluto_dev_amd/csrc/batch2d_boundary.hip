// Ghost-zone fill of the batched 2D MHD boxes with an outflow or reflective
// side: the reference's Boundary (Src/boundary.cpp:67-303) side by side,
// X1_BEG, X1_END, X2_BEG, X2_END, on every box of the batch.  A box is the reference's array for DIMENSIONS 2: cells
// 0 .. ntot-1 along each direction (two ghost layers, the active cells
// lo .. hi, two ghost layers) plus one spare layer holding the outermost face
// (index ntot) of each staggered component.  B1 and B2 live on faces, B3 is
// a cell variable.
//   periodic side: PeriodicBoundary (:502-669), images of cells and faces;
//   outflow side:  OutflowBoundary (:677-760), the edge layer's cells and
//                  tangential faces, then CT_FillStaggeredFields
//                  (Src/MHD/CT/ct_fill_mag_field.cpp:39-330) for the normal
//                  faces from div B = 0;
//   reflective side: ReflectiveBoundary (:931-1100), mirror images with the
//                  normal velocity and normal field negated (FlipSign :840-925);
// then the ghost cells' field average of B1, B2 (:275-303 with
// Src/MHD/CT/ct_field_average.cpp:182-184).
#include "batch2d.hpp"
#include "../../include/gpluto_amd.h"

namespace gpl {

namespace {

// Both sides of direction dir (blockIdx.z: lower, upper) of one box
// (blockIdx.y), one thread per transverse index a and both ghost layers.  As in
// the 3D fill (mhd3d_boundary.hip) the sides write different layers, read
// active ones, and what a ghost cell needs is computed from the source layers in
// registers: two launches a stage where a copy and a fill per side were eight
// (one 306 x 195 box: 44 us a stage in eight, 15 us in two, 12 us with every load
// before the first store).
template <typename R>
__global__ __launch_bounds__(256)
void k2_bnd_dir(const BoxDesc *__restrict__ box, int dir, int type_lo, int type_hi, R *__restrict__ V,
                double *__restrict__ Vs, size_t N)
{
  const BoxDesc d = box[blockIdx.y];
  const int upper = blockIdx.z, type = upper ? type_hi : type_lo;
  const int tr = 1 - dir;
  const int na = dir == 0 ? d.ny : d.nx;
  const int a = blockIdx.x*blockDim.x + threadIdx.x;
  if (a >= na) return;
  const size_t st = dir == 0 ? (size_t)d.nx : 1, sd = dir == 0 ? 1 : (size_t)d.nx;
  const size_t at = (size_t)d.off + a*st;
  const int lo = d.lo[dir], hi = d.hi[dir], n = hi - lo + 1;
  const int g0 = upper ? hi + 1 : 0;            // ghost layers g0, g0 + 1
  // source layer of ghost layer gi; reflective: the mirror image i0 - i,
  // i0 = 2*lo - 1 or 2*hi + 1 (Src/boundary.cpp:939-945)
  auto source = [&](int gi) {
    return type == GPL_PERIODIC ? gi + (upper ? -n : n)
         : type == GPL_REFLECTIVE ? (upper ? 2*hi + 1 : 2*lo - 1) - gi : (upper ? hi : lo);
  };
  double *Bt = Vs + tr*N, *Bn = Vs + dir*N;
  const bool cell = a <= na - 2;                // BOX_LOOP over the ghost box
  double e[2][2];                               // tangential faces on both ends of the ghost cells
  constexpr int VAR[6] = {0, 1, 2, 3, 6, 7};    // B1, B2 are the field average below
  R v[2][6];
  const int f0 = upper ? hi + 1 : 0;            // the normal faces f0 .. f0 + 2 bound the two ghost cells
  double f[3] = {0.0, 0.0, 0.0};
  // every load before the first store: the arrays are filled in place, so a store
  // would hold the loads after it back by a trip to memory each
#pragma unroll
  for (int l = 0; l < 2; l++) {
    const size_t cq = at + source(g0 + l)*sd;
    e[l][0] = Bt[cq];
    if (cell) {
      e[l][1] = Bt[cq + st];
#pragma unroll
      for (int q = 0; q < 6; q++) v[l][q] = V[VAR[q]*N + cq];
    }
  }
  if (cell) {
    if (type == GPL_PERIODIC) {
#pragma unroll
      for (int l = 0; l < 3; l++)
        f[l] = !upper && l == 2 ? Bn[at + lo*sd] : Bn[at + source(f0 + l)*sd];
    } else if (type == GPL_REFLECTIVE) {
      // mirrored about the boundary face and negated: face i from i0 - i + 1 on
      // the lower side, face i + 1 from i0 - i on the upper side
      f[upper ? 0 : 2] = Bn[at + (upper ? f0 : lo)*sd];
      f[upper ? 1 : 0] = -Bn[at + (upper ? source(hi + 1) : source(0) + 1)*sd];
      f[upper ? 2 : 1] = -Bn[at + (upper ? source(hi + 2) : source(1) + 1)*sd];
    } else {
      f[upper ? 0 : 2] = Bn[at + (upper ? hi + 1 : lo)*sd];
    }
  }
#pragma unroll
  for (int l = 0; l < 2; l++) {
    const size_t cp = at + (g0 + l)*sd;
    Bt[cp] = e[l][0];                           // one more face along it (BOX{I,J}_LOOP)
    if (cell) {
#pragma unroll
      for (int q = 0; q < 6; q++)
        V[VAR[q]*N + cp] = type == GPL_REFLECTIVE && VAR[q] == 1 + dir ? -v[l][q] : v[l][q];
    }
  }
  if (!cell) return;
  if (type == GPL_PERIODIC) {
    // BOX_LOOP on the lower side, one more face (the spare layer) on the upper
    Bn[at + f0*sd] = f[0];
    Bn[at + (f0 + 1)*sd] = f[1];
    if (upper) Bn[at + (f0 + 2)*sd] = f[2];
  } else if (type == GPL_REFLECTIVE) {
    Bn[at + (upper ? f0 + 1 : 0)*sd] = f[upper ? 1 : 0];
    Bn[at + (upper ? f0 + 2 : 1)*sd] = f[upper ? 2 : 1];
  } else {
    // outward from the boundary face with div B = 0; face areas of the uniform
    // Cartesian grid in 2D (Src/set_geometry.cpp:124,147)
    const double A[2] = {1.0*d.dy, d.dx*1.0};
#pragma unroll
    for (int l = 0; l < 2; l++) {
      const int c = upper ? l : 1 - l;          // the ghost cell crossed, outward
      // the transverse term, then the missing direction's 0.0 (x, y, z order)
      const double ta = A[tr]*e[c][1] - A[tr]*e[c][0];
      const double tb = 0.0;
      if (!upper) f[c] = (A[dir]*f[c + 1] + ta + tb)/A[dir];
      else        f[c + 1] = (A[dir]*f[c] - (ta + tb))/A[dir];
    }
    Bn[at + (upper ? f0 + 1 : 0)*sd] = f[upper ? 1 : 0];
    Bn[at + (upper ? f0 + 2 : 1)*sd] = f[upper ? 2 : 1];
  }
#pragma unroll
  for (int l = 0; l < 2; l++) {
    const size_t c = at + (g0 + l)*sd;
    V[(4 + dir)*N + c] = (R)(0.5*(f[l] + f[l + 1]));
    V[(4 + tr)*N + c] = (R)(0.5*(e[l][0] + e[l][1]));
  }
}

}  // namespace

template <typename R>
void batch2d_boundary(const BoxDesc *box, int nbox, int maxp, const int type[4], R *V, double *Vs,
                      size_t ncell, hipStream_t s)
{
  for (int dir = 0; dir < 2; dir++)
    hipLaunchKernelGGL((k2_bnd_dir<R>), dim3((maxp + 255)/256, nbox, 2), dim3(256), 0, s,
                       box, dir, type[2*dir], type[2*dir + 1], V, Vs, ncell);
}

template void batch2d_boundary<double>(const BoxDesc *, int, int, const int *, double *, double *,
                                       size_t, hipStream_t);
template void batch2d_boundary<float>(const BoxDesc *, int, int, const int *, float *, double *,
                                      size_t, hipStream_t);

}  // namespace gpl
