// Ghost-zone fill of a 3D MHD/RMHD box padded with ghost layers: the
// reference's Boundary (Src/boundary.cpp:67-303) side by side, X1_BEG ..
// X3_END, on the reference's own index ranges.  The padded box is the
// reference's array: cells 0 .. ntot-1 (two ghost layers, the active cells
// lo .. hi, two ghost layers) plus one spare layer that holds the outermost
// face (index ntot) of every staggered component.
//   periodic side: PeriodicBoundary (:502-669), images of cells and faces;
//   outflow side:  OutflowBoundary (:677-760), the edge layer's cells and
//                  tangential faces, then CT_FillStaggeredFields
//                  (Src/MHD/CT/ct_fill_mag_field.cpp:39-330) for the normal
//                  faces from div B = 0;
//   reflective side: ReflectiveBoundary (:931-1100), mirror images with the
//                  normal velocity and normal field negated (FlipSign);
// then the ghost cells' field average (:275-303 with
// Src/MHD/CT/ct_field_average.cpp:182-184).
#include "mhd3d.hpp"
#include "../../include/gpluto_amd.h"

namespace gpl {

namespace {

// Both sides of direction dir (blockIdx.y: lower, upper), one thread per
// transverse (a, b) of the padded box and both ghost layers.  The two sides
// write different layers and read active ones, and everything a ghost cell
// needs (its copied cells and tangential faces, the outflow side's normal faces
// outward from the boundary, the field average) is computed from the source
// layers in registers, so a direction is one launch without a barrier: three
// launches a stage where a copy and a fill per side were twelve.  These
// launches are latency, not bytes: 80 x 95 x 66, 81 us a stage in twelve,
// 32 us in three, 26 us with every load before the first store.  The directions
// stay in turn: a later one reads the ghosts of an earlier one in its corners.
template <typename R>
__global__ __launch_bounds__(256)
void k_bnd_dir(Box3 g, int dir, int type_lo, int type_hi, R *__restrict__ V, double *__restrict__ Vs)
{
  const int upper = blockIdx.y, type = upper ? type_hi : type_lo;
  const int t1 = (dir + 1) % 3, t2 = (dir + 2) % 3;
  const int P[3] = {g.nx, g.ny, g.nz};
  const int na = P[t1], nb = P[t2];
  const int t = blockIdx.x*blockDim.x + threadIdx.x;
  if (t >= na*nb) return;
  const int b = t / na, a = t - b*na;
  const size_t S[3] = {1, (size_t)g.nx, (size_t)g.nx*g.ny};
  const size_t N = (size_t)g.ncell, at = a*S[t1] + b*S[t2], s1 = S[t1], s2 = S[t2], sd = S[dir];
  const int lo = g.lo[dir], hi = g.hi[dir], n = hi - lo + 1;
  const int g0 = upper ? hi + 1 : 0;            // ghost layers g0, g0 + 1
  // source layer of ghost layer gi; reflective: the mirror image i0 - i,
  // i0 = 2*lo - 1 or 2*hi + 1 (Src/boundary.cpp:939-945)
  auto source = [&](int gi) {
    return type == GPL_PERIODIC ? gi + (upper ? -n : n)
         : type == GPL_REFLECTIVE ? (upper ? 2*hi + 1 : 2*lo - 1) - gi : (upper ? hi : lo);
  };
  double *B1 = Vs + t1*N, *B2 = Vs + t2*N, *Bn = Vs + dir*N;
  const bool cell = a <= na - 2 && b <= nb - 2; // BOX_LOOP over the ghost box
  double e1[2][2], e2[2][2];                    // tangential faces on both ends of the ghost cells
  constexpr int VAR[5] = {0, 1, 2, 3, 7};       // B1..3 are the field average below
  R v[2][5];
  const int f0 = upper ? hi + 1 : 0;            // the normal faces f0 .. f0 + 2 bound the two ghost cells
  double f[3] = {0.0, 0.0, 0.0};
  // every load before the first store: the arrays are filled in place, so a store
  // would hold the loads after it back by a trip to memory each
#pragma unroll
  for (int l = 0; l < 2; l++) {
    const size_t cq = at + source(g0 + l)*sd;
    if (b <= nb - 2) e1[l][0] = B1[cq];
    if (a <= na - 2) e2[l][0] = B2[cq];
    if (cell) {
      e1[l][1] = B1[cq + s1];
      e2[l][1] = B2[cq + s2];
#pragma unroll
      for (int q = 0; q < 5; q++) v[l][q] = V[VAR[q]*N + cq];
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
    // tangential components: one more face along the component (BOX{I,J,K}_LOOP)
    if (b <= nb - 2) B1[cp] = e1[l][0];
    if (a <= na - 2) B2[cp] = e2[l][0];
    if (cell) {
      // FlipSign (Src/boundary.cpp:840-925): a wall negates the normal velocity and field
#pragma unroll
      for (int q = 0; q < 5; q++)
        V[VAR[q]*N + cp] = type == GPL_REFLECTIVE && VAR[q] == 1 + dir ? -v[l][q] : v[l][q];
    }
  }
  if (!cell) return;
  if (type == GPL_PERIODIC) {
    // BOX_LOOP on the lower side, BOXI/J/K_LOOP (one more face, the spare
    // layer) on the upper side
    Bn[at + f0*sd] = f[0];
    Bn[at + (f0 + 1)*sd] = f[1];
    if (upper) Bn[at + (f0 + 2)*sd] = f[2];
  } else if (type == GPL_REFLECTIVE) {
    Bn[at + (upper ? f0 + 1 : 0)*sd] = f[upper ? 1 : 0];
    Bn[at + (upper ? f0 + 2 : 1)*sd] = f[upper ? 2 : 1];
  } else {
    // outward from the boundary face with div B = 0; face areas of the uniform
    // Cartesian grid (Src/set_geometry.cpp:124,147,166)
    const double A[3] = {1.0*g.dy*g.dz, g.dx*1.0*g.dz, g.dx*g.dy*1.0};
#pragma unroll
    for (int l = 0; l < 2; l++) {
      const int c = upper ? l : 1 - l;          // the ghost cell crossed, outward
      const double d1 = A[t1]*e1[c][1] - A[t1]*e1[c][0];
      const double d2 = A[t2]*e2[c][1] - A[t2]*e2[c][0];
      // the two transverse terms in x, y, z order: (t1, t2) is (y, z), (z, x), (x, y)
      const double ta = dir == 1 ? d2 : d1, tb = dir == 1 ? d1 : d2;
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
    V[(4 + t1)*N + c] = (R)(0.5*(e1[l][0] + e1[l][1]));
    V[(4 + t2)*N + c] = (R)(0.5*(e2[l][0] + e2[l][1]));
  }
}

}  // namespace

template <typename R>
void mhd3d_boundary(const Box3 &g, const int type[6], R *V, double *Vs, hipStream_t s)
{
  for (int dir = 0; dir < 3; dir++) {
    const int P[3] = {g.nx, g.ny, g.nz};
    const int na = P[(dir + 1) % 3], nb = P[(dir + 2) % 3];
    hipLaunchKernelGGL((k_bnd_dir<R>), dim3((na*nb + 255)/256, 2), dim3(256), 0, s,
                       g, dir, type[2*dir], type[2*dir + 1], V, Vs);
  }
}

template void mhd3d_boundary<double>(const Box3 &, const int *, double *, double *, hipStream_t);
template void mhd3d_boundary<float>(const Box3 &, const int *, float *, double *, hipStream_t);

}  // namespace gpl
