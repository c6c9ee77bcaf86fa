// HD stage update (PLM + HLLC/HLL + RK2/RK3) on 1D/2D/3D boxes with periodic,
// outflow or reflective sides, FP64, for gfx950.
//
// Device data model: V[5][n] (rho, v1..3, prs), U[5][n] (rho, m1..3, E), no
// ghost zones.  A neighbour outside the box is the wrapped cell (periodic), the
// nearest active cell (outflow: OutflowBoundary, boundary.cpp:677-760, copies the
// edge cell into every ghost zone) or the mirrored cell with its normal velocity
// negated (reflective: ReflectiveBoundary, boundary.cpp:931-1000, ghost i =
// vsign*Vc(i0 - i)), which is bitwise what the reference's ghost fill supplies to
// the sweep.
//
//  * 2D, 3D (k_hd_stage2d, k_hd_stage3d): a stage is one launch that marches rows
//    or planes; every face is solved about once and handed to its other cell by a
//    lane shuffle, through LDS or in registers, and dUc = rhs_x + rhs_y + rhs_z (update_stage.cpp:173-184,
//    272-284, 369-380), the RK combination (rk_step.cpp:366-374,509-518) and
//    ConsToPrim3D (mappers3D.cpp:104-194) follow in registers.
//  * 2D and 3D boxes too narrow to fill those kernels' lanes (hd_by_direction): one
//    launch per direction (k_hd_sweep), a thread per cell.
//  * 1D (k_hd_step1d): a whole step is one launch; a block recomputes the cells
//    that the later stages need beyond its own.
#include "hd.hpp"
#include "physics.hpp"

namespace gpl {

namespace {

// The cell that ghost index q of a direction reads, q within two cells of the
// box (further out: some cell, whose value nothing uses); flip: its normal
// velocity changes sign.
__device__ __forceinline__ int hd_source(int q, int n, int lo, int hi, bool &flip)
{
  flip = false;
  if (q < 0) {
    flip = lo == GPL_REFLECTIVE;
    q = lo == GPL_PERIODIC ? q + n : (lo == GPL_OUTFLOW ? 0 : -1 - q);
  } else if (q >= n) {
    flip = hi == GPL_REFLECTIVE;
    q = hi == GPL_PERIODIC ? q - n : (hi == GPL_OUTFLOW ? n - 1 : 2*n - 1 - q);
  }
  return q < 0 ? 0 : (q >= n ? n - 1 : q);
}

// base[idx] from a uniform base and a byte offset of type OFF: 32 bits (one
// scalar base per array slot and one offset per lane) while a slot is below
// 4 GiB, 64 bits above
template <typename OFF>
__device__ __forceinline__ double ldo(const double *base, OFF idx)
{
  return *(const double *)((const char *)base + idx*(OFF)sizeof(double));
}
template <typename OFF>
__device__ __forceinline__ void sto(double *base, OFF idx, double v)
{
  *(double *)((char *)base + idx*(OFF)sizeof(double)) = v;
}

template <int D, int SOLVER>
__device__ __forceinline__ void hd_riemann(const double *vl, const double *vr, double gamma,
                                           FaceFlux<double> &f)
{
  if constexpr (SOLVER == 2) hd_hllc<double, D>(vl, vr, gamma, f);
  else hd_hll<double, D>(vl, vr, gamma, f);
}

__device__ __forceinline__ double wave_max(double v)
{
  for (int o = 32; o > 0; o >>= 1) {
    const double w = __shfl_xor(v, o, 64);
    v = v >= w ? v : w;
  }
  return v;
}

// max over the block's values in every lane of wave 0 (red: one slot per wave)
__device__ __forceinline__ double block_max(double v, double *red)
{
  v = wave_max(v);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  const int nw = (blockDim.x + 63) >> 6;
  double m = red[0];
  for (int q = 1; q < nw; q++) m = m >= red[q] ? m : red[q];
  return m;
}

// Which block of a launch is the last to arrive, without a fence and without a
// queue on one address: a block counts itself into one of kSub counters (on
// lines of their own), the last of those into the common one.  `seen` is a value
// whose load or exchange has to have returned before the block counts: the
// increment is made to depend on it, which orders the two.  A device-scope
// release or acquire instead writes back or drops the XCD's whole L2, and one
// counter serialises its blocks (750 blocks of a 511x333 stage: 31 us with both,
// 24 without the fences, 19 with neither).  Called by one thread of a block.
constexpr unsigned kSub = 16, kLine = 32;      // kLine unsigneds: 128 B
static_assert((kSub + 1)*kLine == HD_ARRIVED, "the arrival counters");

template <typename T>
__device__ __forceinline__ bool arrive(unsigned *arrived, T seen)
{
  const unsigned c = blockIdx.x % kSub, mine = (gridDim.x + kSub - 1 - c)/kSub;   // blocks of counter c
  unsigned one = 1;
  asm volatile("" : "+v"(one) : "v"(seen));
  if (__hip_atomic_fetch_add(arrived + (1 + c)*kLine, one, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != mine - 1)
    return false;
  const unsigned counters = gridDim.x < kSub ? gridDim.x : kSub;
  return __hip_atomic_fetch_add(arrived, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == counters - 1;
}

// invDt_hyp = max(C_dt)/DIMENSIONS over the stage-1 partials (part[q] read with
// load), optionally NextTimeStep and time += dt; called by one whole block.
template <typename LOAD>
__device__ void step_control(const HdStep &st, double dt, int nparts, int dims, double *red, LOAD load)
{
  double m = -1.0;
  for (int q = threadIdx.x; q < nparts; q += blockDim.x) {
    const double p = load(q);
    m = m >= p ? m : p;
  }
  m = block_max(m, red);
  if (threadIdx.x == 0) {
    const double inv = m/(double)dims;
    st.ctl->inv_dt = inv;
    if (st.advance) {
      st.ctl->time += dt;
      const double dt_new = st.cfl/inv;
      st.ctl->dt = dt_new <= st.cfl_max_var*dt ? dt_new : st.cfl_max_var*dt;
      st.ctl->nstep += 1;
    }
    for (unsigned q = 0; q <= kSub; q++) st.arrived[q*kLine] = 0;
  }
}

// ---------------------------------------------------------------------------
// One stage of a 3D box.  Wave w of the block's eight owns row j0 + w of
// a plane: it solves the x faces of its 64 cells (the 65th of every row goes to
// wave 7's lanes, whose row is the next block's), the lower y face of its row,
// and the upper z face of its cells, whose window and lower flux it
// carries along the march of L planes.  The loads of plane k+1 are in flight
// while plane k is computed.
//
// What bounds it: about 160 B per cell and stage have to move (200 from the
// second stage on), and 3 x 330 VALU instructions per cell to issue.  One launch
// per direction with two face solves per cell and dU and C_dt through memory
// moved 480 B and issued twice the solves: 128x96x112, 184 us a stage in three
// launches, 103 in this one; 256^3, 2280 and 1150.  At 205 VGPRs one block fills a
// CU (two waves per SIMD), so its barriers are not hidden: 630 us is the bytes'.
//
// NextTimeStep rides in the last stage's launch: a block that has read dt counts
// itself in (arrive), and the last one, when nobody needs the old dt any more,
// reduces the partials that the first stage's launch left.  No block waits
// for another.
// ---------------------------------------------------------------------------
constexpr int TX = kHdCols, TY = kHdRows, NW = TY + 1;
constexpr int SW = TX + 4, SH = NW + 3;        // staged columns i0-2 .. i0+65, rows j0-2 .. j0+8

template <int LIM, int SOLVER, typename OFF>
__global__ __launch_bounds__(64*NW)
void k_hd_stage3d(HdBox g, int L, HdBufs b, HdStep st, RKW w, int first_stage, int want_cdt, int nparts,
                double gamma, double small_rho, double small_prs)
{
  __shared__ double sV[5][SH][SW];
  __shared__ double sY[6][NW][TX];             // flux and C_dt speed of the rows' lower y faces
  __shared__ double sX[6][TY];                 // and of the rows' 65th x face
  __shared__ double red[NW];
  __shared__ int s_last;
  const int tid = threadIdx.x, tx = tid & 63, wv = tid >> 6;
  const double dt = *(const volatile double *)&st.ctl->dt;   // read before this block counts as arrived
  const int nx = g.nx, ny = g.ny, nz = g.nz;
  const size_t n = (size_t)g.ncell;
  const int ntx = (nx + TX - 1)/TX, nty = (ny + TY - 1)/TY;
  const int bx = blockIdx.x % ntx, br = blockIdx.x / ntx, by = br % nty, seg = br / nty;
  const int i0 = bx*TX, j0 = by*TY, k0 = seg*L, k1 = k0 + L < nz ? k0 + L : nz;
  const int i = i0 + tx, j = j0 + wv;
  const bool own = wv < TY && i < nx && j < ny;
  const OFF plane = (OFF)nx*ny;
  // the cell of this thread's column (a ghost beyond the box: its source), and
  // the halo position that the first 236 threads load besides
  bool fx, fy, hx, hy;
  const int ci = hd_source(i, nx, g.lo[0], g.hi[0], fx), cj = hd_source(j, ny, g.lo[1], g.hi[1], fy);
  const OFF col = ci + (OFF)nx*cj;
  int hr, hc;
  if (tid < 2*SW)      { hr = tid / SW; hc = tid - hr*SW; }
  else if (tid < 3*SW) { hr = SH - 1;   hc = tid - 2*SW; }
  else { const int q = tid - 3*SW; hr = 2 + (q >> 2); hc = (q & 3) + ((q & 3) < 2 ? 0 : TX); }
  const bool halo = tid < 3*SW + 4*NW;
  const int hi_ = hd_source(i0 - 2 + hc, nx, g.lo[0], g.hi[0], hx);
  const int hj_ = hd_source(j0 - 2 + hr, ny, g.lo[1], g.hi[1], hy);
  const OFF hcol = hi_ + (OFF)nx*hj_;
  double pv[5];
  auto load_halo = [&](int k) {
    if (!halo) return;
    const OFF o = hcol + plane*k;
#pragma unroll
    for (int q = 0; q < 5; q++) pv[q] = ldo<OFF>(b.Vin + q*n, o);
    if (hx) pv[1] = -pv[1];
    if (hy) pv[2] = -pv[2];
  };
  // the cell of this thread's column in plane k, ghost planes included
  auto load_col = [&](int k, double *v) {
    bool fz;
    const int kk = hd_source(k, nz, g.lo[2], g.hi[2], fz);
    const OFF o = col + plane*kk;
#pragma unroll
    for (int q = 0; q < 5; q++) v[q] = ldo<OFF>(b.Vin + q*n, o);
    if (fx) v[1] = -v[1];
    if (fy) v[2] = -v[2];
    if (fz) v[3] = -v[3];
  };
  uint32_t e = 0;
  double cdt_max = -1.0;
  double vz[5], vz1[5], vz2[5], zl[5], Fz[5], cz = 0.0;   // V(k), V(k+1), V(k+2), vL(k+1), lower face
  {                                            // wave 7 only carries the planes it stages
    double a[5], c[5], vl[5], vr[5];
    load_col(k0 - 2, a);
    load_col(k0 - 1, c);
    load_col(k0, vz);
    load_col(k0 + 1, vz1);
#pragma unroll
    for (int q = 0; q < 5; q++) {
      vl[q] = c[q] + 0.5*plm_slope<double, LIM>(a[q], c[q], vz[q]);
      const double d = plm_slope<double, LIM>(c[q], vz[q], vz1[q]);
      vr[q] = vz[q] - 0.5*d;
      zl[q] = vz[q] + 0.5*d;
    }
    FaceFlux<double> f;
    hd_riemann<2, SOLVER>(vl, vr, gamma, f);
    if (own) e |= f.err;
#pragma unroll
    for (int q = 0; q < 5; q++) Fz[q] = f.f[q];
    cz = rmax(rabs(f.Sl), rabs(f.Sr));
  }
  const double dtdx = dt/g.dx, dtdy = dt/g.dy, dtdz = dt/g.dz;
  load_halo(k0);
  for (int k = k0; k < k1; k++) {
#pragma unroll
    for (int q = 0; q < 5; q++) {
      sV[q][wv + 2][tx + 2] = vz[q];
      if (halo) sV[q][hr][hc] = pv[q];
    }
    __syncthreads();
    if (k + 1 < k1) load_halo(k + 1);
    load_col(k + 2, vz2);
    const OFF o = col + plane*k;
    // x face i of row j; wave 7: face i0 + 64 of row j0 + tx
    double Fx[6];
    if (wv < TY || tx < TY) {
      const int r = (wv < TY ? wv : tx) + 2, c = wv < TY ? tx : TX;
      double vl[5], vr[5];
#pragma unroll
      for (int q = 0; q < 5; q++) {
        const double a0 = sV[q][r][c], a1 = sV[q][r][c + 1], a2 = sV[q][r][c + 2], a3 = sV[q][r][c + 3];
        vl[q] = a1 + 0.5*plm_slope<double, LIM>(a0, a1, a2);
        vr[q] = a2 - 0.5*plm_slope<double, LIM>(a1, a2, a3);
      }
      FaceFlux<double> f;
      hd_riemann<0, SOLVER>(vl, vr, gamma, f);
      if (i0 + c <= nx && j0 + r - 2 < ny) e |= f.err;
#pragma unroll
      for (int q = 0; q < 5; q++) Fx[q] = f.f[q];
      Fx[5] = rmax(rabs(f.Sl), rabs(f.Sr));
      if (wv == TY) {
#pragma unroll
        for (int q = 0; q < 6; q++) sX[q][tx] = Fx[q];
      }
    }
    __builtin_amdgcn_sched_barrier(0);         // one solve's registers at a time
    // y face j
    double Fy[6];
    {
      double vl[5], vr[5];
#pragma unroll
      for (int q = 0; q < 5; q++) {
        const double a0 = sV[q][wv][tx + 2], a1 = sV[q][wv + 1][tx + 2];
        const double a2 = sV[q][wv + 2][tx + 2], a3 = sV[q][wv + 3][tx + 2];
        vl[q] = a1 + 0.5*plm_slope<double, LIM>(a0, a1, a2);
        vr[q] = a2 - 0.5*plm_slope<double, LIM>(a1, a2, a3);
      }
      FaceFlux<double> f;
      hd_riemann<1, SOLVER>(vl, vr, gamma, f);
      if (i < nx && j <= ny) e |= f.err;
#pragma unroll
      for (int q = 0; q < 5; q++) Fy[q] = f.f[q];
      Fy[5] = rmax(rabs(f.Sl), rabs(f.Sr));
#pragma unroll
      for (int q = 0; q < 6; q++) sY[q][wv][tx] = Fy[q];
    }
    __builtin_amdgcn_sched_barrier(0);
    double u_in[5], u0[5];
    if (own) {
#pragma unroll
      for (int q = 0; q < 5; q++) u_in[q] = ldo<OFF>(b.Uin + q*n, o);
      if (!first_stage) {
#pragma unroll
        for (int q = 0; q < 5; q++) u0[q] = ldo<OFF>(b.U0 + q*n, o);
      }
    }
    __syncthreads();
    double du[5], cd = 0.0;
    if (wv < TY) {                             // whole waves: the shuffle
#pragma unroll
      for (int q = 0; q < 6; q++) {
        double up = __shfl_down(Fx[q], 1, 64);
        if (tx == TX - 1) up = sX[q][wv];
        const double uy = sY[q][wv + 1][tx];
        if (q < 5) {
          double r = -dtdx*(up - Fx[q]);
          r += 0.0;
          du[q] = r;
          r = -dtdy*(uy - Fy[q]);
          r += 0.0;
          du[q] += r;
        } else {
          cd = 0.5*(Fx[5] + up)/g.dx;          // rhs.cpp:523,756,981
          cd += 0.5*(Fy[5] + uy)/g.dy;
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      {                                        // z face k + 1
        double vl[5], vr[5];
#pragma unroll
        for (int q = 0; q < 5; q++) {
          const double d = plm_slope<double, LIM>(vz[q], vz1[q], vz2[q]);
          vl[q] = zl[q];
          vr[q] = vz1[q] - 0.5*d;
          zl[q] = vz1[q] + 0.5*d;
        }
        FaceFlux<double> f;
        hd_riemann<2, SOLVER>(vl, vr, gamma, f);
        if (own) e |= f.err;
#pragma unroll
        for (int q = 0; q < 5; q++) {
          double r = -dtdz*(f.f[q] - Fz[q]);
          r += 0.0;
          du[q] += r;
          Fz[q] = f.f[q];
        }
        const double cm = rmax(rabs(f.Sl), rabs(f.Sr));
        cd += 0.5*(cz + cm)/g.dz;
        cz = cm;
      }
      if (own) {
        double u[5], vn[5];
#pragma unroll
        for (int q = 0; q < 5; q++)
          u[q] = first_stage ? u_in[q] + w.wR*du[q] : w.w0*u0[q] + w.w1*u_in[q] + w.wR*du[q];
        const uint32_t ce = hd_cons_to_prim(u, gamma - 1.0, small_rho, small_prs, vn);
        e |= ce;
        zone_report(b.zr[0], o, ce);
#pragma unroll
        for (int q = 0; q < 5; q++) { sto<OFF>(b.Uout + q*n, o, u[q]); sto<OFF>(b.Vout + q*n, o, vn[q]); }
        if (want_cdt) cdt_max = cdt_max >= cd ? cdt_max : cd;
      }
    }
#pragma unroll
    for (int q = 0; q < 5; q++) { vz[q] = vz1[q]; vz1[q] = vz2[q]; }
  }
  report_bits(b.err, e);
  if (want_cdt) {
    const double m = block_max(cdt_max, red);
    if (tid == 0) b.cdt_part[blockIdx.x] = m;
  }
  if (st.ends_step) {
    __syncthreads();                           // every wave has read dt
    if (tid == 0) s_last = arrive(st.arrived, dt);
    __syncthreads();
    if (s_last) step_control(st, dt, nparts, 3, red, [&](int q) { return b.cdt_part[q]; });
  }
}

// ---------------------------------------------------------------------------
// One stage of a 2D box.  A wavefront owns 63 columns and marches L rows of
// them, with no barrier: it solves the 64 lower x faces of a row (the last one
// is the upper face of column 62) and takes the upper one by a lane shuffle, and
// carries its columns' window and lower y flux from row to row.  Side columns
// come from the row just loaded by the neighbours (L1).
//
// What bounds it: the latency of one lane's solves on small boxes, 160 to 200 B
// per cell and stage on large ones (2000x1800: 365 us a stage in two launches with
// two solves per face, 195 in this one; 511x333: 25 and 19).
// ---------------------------------------------------------------------------
template <int LIM, int SOLVER, typename OFF>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3)))
void k_hd_stage2d(HdBox g, int L, HdBufs b, HdStep st, RKW w, int first_stage, int want_cdt, int nparts,
                  double gamma, double small_rho, double small_prs)
{
  __shared__ double red[4];
  __shared__ int s_last;
  const int tid = threadIdx.x, tx = tid & 63, wv = tid >> 6;
  const double dt = *(const volatile double *)&st.ctl->dt;   // read before this block counts as arrived
  const int nx = g.nx, ny = g.ny;
  const size_t n = (size_t)g.ncell;
  const int ntx = (nx + 62)/63, gw = blockIdx.x*4 + wv, seg = gw / ntx;
  const int f = (gw - seg*ntx)*63 + tx;        // the lane's face: the lower one of cell f
  const int s0 = seg*L, s1 = s0 + L < ny ? s0 + L : ny;
  uint32_t e = 0;
  double cdt_max = -1.0;
  if (s0 < ny) {                               // whole waves
    const bool own = tx < 63 && f < nx;
    OFF xc[4];                                 // columns f-2 .. f+1
    bool xf[4];
#pragma unroll
    for (int o = 0; o < 4; o++) xc[o] = hd_source(f + o - 2, nx, g.lo[0], g.hi[0], xf[o]);
    auto row_of = [&](int r, bool &flip) { return (OFF)nx*hd_source(r, ny, g.lo[1], g.hi[1], flip); };
    auto load_own = [&](int r, double *v) {
      bool fy;
      const OFF o = xc[2] + row_of(r, fy);
#pragma unroll
      for (int q = 0; q < 5; q++) v[q] = ldo<OFF>(b.Vin + q*n, o);
      if (fy) v[2] = -v[2];
    };
    double vc[5], v1[5], yl[5], Fy[5], cy;     // V(r), V(r+1), vL(r+1), the lower y flux
    {
      double a[5], c[5], vl[5], vr[5];
      load_own(s0 - 2, a);
      load_own(s0 - 1, c);
      load_own(s0, vc);
      load_own(s0 + 1, v1);
#pragma unroll
      for (int q = 0; q < 5; q++) {
        vl[q] = c[q] + 0.5*plm_slope<double, LIM>(a[q], c[q], vc[q]);
        const double d = plm_slope<double, LIM>(c[q], vc[q], v1[q]);
        vr[q] = vc[q] - 0.5*d;
        yl[q] = vc[q] + 0.5*d;
      }
      FaceFlux<double> ff;
      hd_riemann<1, SOLVER>(vl, vr, gamma, ff);
      if (own) e |= ff.err;
#pragma unroll
      for (int q = 0; q < 5; q++) Fy[q] = ff.f[q];
      cy = rmax(rabs(ff.Sl), rabs(ff.Sr));
    }
    const double dtdx = dt/g.dx, dtdy = dt/g.dy;
    for (int r = s0; r < s1; r++) {
      const OFF row = (OFF)nx*r, o = xc[2] + row;
      double v2[5], u_in[5], u0[5];
      load_own(r + 2, v2);
      double vl[5], vr[5], du[5], cd = 0.0;
#pragma unroll
      for (int q = 0; q < 5; q++) {            // x face f
        double a0 = ldo<OFF>(b.Vin + q*n, xc[0] + row), a1 = ldo<OFF>(b.Vin + q*n, xc[1] + row);
        double a2 = vc[q], a3 = ldo<OFF>(b.Vin + q*n, xc[3] + row);
        if (q == 1) {
          a0 = xf[0] ? -a0 : a0;
          a1 = xf[1] ? -a1 : a1;
          a2 = xf[2] ? -a2 : a2;
          a3 = xf[3] ? -a3 : a3;
        }
        vl[q] = a1 + 0.5*plm_slope<double, LIM>(a0, a1, a2);
        vr[q] = a2 - 0.5*plm_slope<double, LIM>(a1, a2, a3);
      }
      if (own) {
#pragma unroll
        for (int q = 0; q < 5; q++) u_in[q] = ldo<OFF>(b.Uin + q*n, o);
        if (!first_stage) {
#pragma unroll
          for (int q = 0; q < 5; q++) u0[q] = ldo<OFF>(b.U0 + q*n, o);
        }
      }
      {
        FaceFlux<double> ff;
        hd_riemann<0, SOLVER>(vl, vr, gamma, ff);
        if (f <= nx) e |= ff.err;
#pragma unroll
        for (int q = 0; q < 5; q++) {
          double rr = -dtdx*(__shfl_down(ff.f[q], 1, 64) - ff.f[q]);
          rr += 0.0;
          du[q] = rr;
        }
        const double cm = rmax(rabs(ff.Sl), rabs(ff.Sr));
        cd = 0.5*(cm + __shfl_down(cm, 1, 64))/g.dx;     // rhs.cpp:523,756,981
      }
#pragma unroll
      for (int q = 0; q < 5; q++) {            // y face r + 1
        const double d = plm_slope<double, LIM>(vc[q], v1[q], v2[q]);
        vl[q] = yl[q];
        vr[q] = v1[q] - 0.5*d;
        yl[q] = v1[q] + 0.5*d;
        vc[q] = v1[q];
        v1[q] = v2[q];
      }
      {
        FaceFlux<double> ff;
        hd_riemann<1, SOLVER>(vl, vr, gamma, ff);
        if (own) e |= ff.err;
#pragma unroll
        for (int q = 0; q < 5; q++) {
          double rr = -dtdy*(ff.f[q] - Fy[q]);
          rr += 0.0;
          du[q] += rr;
          Fy[q] = ff.f[q];
        }
        const double cm = rmax(rabs(ff.Sl), rabs(ff.Sr));
        cd += 0.5*(cy + cm)/g.dy;
        cy = cm;
      }
      if (own) {
        double u[5], vn[5];
#pragma unroll
        for (int q = 0; q < 5; q++)
          u[q] = first_stage ? u_in[q] + w.wR*du[q] : w.w0*u0[q] + w.w1*u_in[q] + w.wR*du[q];
        const uint32_t ce = hd_cons_to_prim(u, gamma - 1.0, small_rho, small_prs, vn);
        e |= ce;
        zone_report(b.zr[0], o, ce);
#pragma unroll
        for (int q = 0; q < 5; q++) { sto<OFF>(b.Uout + q*n, o, u[q]); sto<OFF>(b.Vout + q*n, o, vn[q]); }
        if (want_cdt) cdt_max = cdt_max >= cd ? cdt_max : cd;
      }
    }
  }
  report_bits(b.err, e);
  if (want_cdt) {
    const double m = block_max(cdt_max, red);
    if (tid == 0) b.cdt_part[blockIdx.x] = m;
  }
  if (st.ends_step) {
    __syncthreads();                           // every wave has read dt
    if (tid == 0) s_last = arrive(st.arrived, dt);
    __syncthreads();
    if (s_last) step_control(st, dt, nparts, 2, red, [&](int q) { return b.cdt_part[q]; });
  }
}

// ---------------------------------------------------------------------------
// One direction of a 2D or 3D stage, one thread per cell: it reconstructs cells
// -1, 0, +1, solves both faces of its cell and forms rhs; dU and Cdt carry the sums
// to the last direction, which applies the RK combination and ConsToPrim.  Every face
// is solved twice and dU, Cdt go through memory, but no lane is idle however
// narrow the box; hd_by_direction draws the line to the kernels above.
// ---------------------------------------------------------------------------
template <int D, bool LAST, int LIM, int SOLVER>
__global__ __launch_bounds__(256)
void k_hd_sweep(HdBox g, HdBufs b, const StepCtl *__restrict__ ctl, RKW w, int first_stage, int want_cdt,
                double gamma, double small_rho, double small_prs)
{
  __shared__ double red[4];
  const int c = blockIdx.x*blockDim.x + threadIdx.x;
  double cdt_max = -1.0;
  uint32_t e = 0;
  if (c < g.ncell) {
    const size_t n = (size_t)g.ncell;
    const int nd = D == 0 ? g.nx : (D == 1 ? g.ny : g.nz);
    const int sd = D == 0 ? 1 : (D == 1 ? g.nx : g.nx*g.ny);
    const int p = D == 0 ? c % g.nx : (D == 1 ? (c/g.nx) % g.ny : c/(g.nx*g.ny));
    double v[5][5];                 // [cell -2..+2][variable]
#pragma unroll
    for (int o = 0; o < 5; o++) {
      bool flip;
      const int i = c + (hd_source(p + o - 2, nd, g.lo[D], g.hi[D], flip) - p)*sd;
#pragma unroll
      for (int q = 0; q < 5; q++) v[o][q] = b.Vin[q*n + i];
      if (flip) v[o][1 + D] = -v[o][1 + D];
    }
    double lo_l[5], lo_r[5], hi_l[5], hi_r[5];
#pragma unroll
    for (int q = 0; q < 5; q++) {
      const double d0 = plm_slope<double, LIM>(v[1][q], v[2][q], v[3][q]);
      lo_l[q] = v[1][q] + 0.5*plm_slope<double, LIM>(v[0][q], v[1][q], v[2][q]);
      lo_r[q] = v[2][q] - 0.5*d0;
      hi_l[q] = v[2][q] + 0.5*d0;
      hi_r[q] = v[3][q] - 0.5*plm_slope<double, LIM>(v[2][q], v[3][q], v[4][q]);
    }
    FaceFlux<double> lo, hi;
    hd_riemann<D, SOLVER>(lo_l, lo_r, gamma, lo);
    hd_riemann<D, SOLVER>(hi_l, hi_r, gamma, hi);
    e |= lo.err | hi.err;           // a face's bits come from both of its cells
    const double ddx = D == 0 ? g.dx : (D == 1 ? g.dy : g.dz), dtdx = ctl->dt/ddx;
    double du[5];
#pragma unroll
    for (int q = 0; q < 5; q++) {
      double r = -dtdx*(hi.f[q] - lo.f[q]);
      r += 0.0;
      du[q] = D == 0 ? r : b.dU[q*n + c] + r;
    }
    double cd = 0.0;
    if (want_cdt) {
      cd = 0.5*(rmax(rabs(lo.Sl), rabs(lo.Sr)) + rmax(rabs(hi.Sl), rabs(hi.Sr)))/ddx;   // rhs.cpp:523,756,981
      if (D > 0) cd = b.Cdt[c] + cd;
    }
    if (!LAST) {
#pragma unroll
      for (int q = 0; q < 5; q++) b.dU[q*n + c] = du[q];
      if (want_cdt) b.Cdt[c] = cd;
    } else {
      double u[5], vn[5];
#pragma unroll
      for (int q = 0; q < 5; q++) {
        const size_t o = q*n + c;
        u[q] = first_stage ? b.Uin[o] + w.wR*du[q] : w.w0*b.U0[o] + w.w1*b.Uin[o] + w.wR*du[q];
      }
      const uint32_t ce = hd_cons_to_prim(u, gamma - 1.0, small_rho, small_prs, vn);
      e |= ce;
      zone_report(b.zr[0], c, ce);
#pragma unroll
      for (int q = 0; q < 5; q++) { b.Uout[q*n + c] = u[q]; b.Vout[q*n + c] = vn[q]; }
      cdt_max = cd;
    }
  }
  report_bits(b.err, e);
  if (LAST && want_cdt) {
    const double m = block_max(cdt_max, red);
    if (threadIdx.x == 0) b.cdt_part[blockIdx.x] = m;
  }
}

// ---------------------------------------------------------------------------
// A whole step of a 1D box: NST stages with everything between them in
// registers and LDS.  A block's B threads hold its own cells and 2 NST more on
// either side; after stage s the outer 2 s cells of either side are no longer
// right and nothing that is kept depends on them.  Outflow and reflective
// ghosts are refilled from the block's own cells between the stages.
//
// A 1D box is latency: three dependent launches a step (two stages and the dt
// reduction) took 18.2 us for 4096 cells, this one 9.8.  Blocks of one
// wavefront up to 16384 cells, of four above, where the redundant cells (8 or 12
// of the block's) cost more than the barriers.
//
// NextTimeStep: the last block to finish reduces the partial maxima.  They are
// exchanged and read with device-scope atomics, each before its block counts as
// arrived (arrive); no block waits for another.
// ---------------------------------------------------------------------------
template <int LIM, int SOLVER, int NST, int B>
__global__ __launch_bounds__(B)
void k_hd_step1d(HdBox g, HdBufs b, HdStep st, double gamma, double small_rho, double small_prs)
{
  constexpr int H = 2*NST, T = B - 2*H;
  __shared__ double sV[5][B], sL[5][B], sF[6][B];
  __shared__ double red[(B + 63)/64];
  __shared__ int s_last;
  const int t = threadIdx.x, nx = g.nx;
  const size_t n = (size_t)nx;
  const int q0 = blockIdx.x*T - H, i = q0 + t;        // this thread's cell, ghosts included
  // every wave uses dt in the first stage, before the barriers of the second, so
  // before the block counts itself in
  const double dt = st.ctl->dt, dtdx = dt/g.dx;
  const bool periodic = g.lo[0] == GPL_PERIODIC;
  // the cell to start from; a periodic ghost is an image and evolves like it,
  // other ghosts are refilled from cell src (position sp) before each stage
  bool flip = false;
  int src = i;
  if (periodic) src = ((i % nx) + nx) % nx;
  else src = hd_source(i, nx, g.lo[0], g.hi[0], flip);
  const bool ghost = !periodic && (i < 0 || i >= nx);
  int sp = src - q0;
  if (sp < 0 || sp >= B) sp = t;                      // beyond what the block's cells depend on
  const bool own = t >= H && t < B - H && i < nx;
  double v[5], u0[5], u[5];
#pragma unroll
  for (int q = 0; q < 5; q++) { v[q] = b.Vin[q*n + src]; u0[q] = b.Uin[q*n + src]; u[q] = u0[q]; }
  if (flip) v[1] = -v[1];
  const RKW ws[3] = {{0.0, 0.0, 1.0},
                     NST == 3 ? RKW{0.75, 0.25, 0.25} : RKW{0.5, 0.5, 0.5},
                     {1.0/3.0, 2.0/3.0, 2.0/3.0}};
  const int tm = t > 0 ? t - 1 : 0, tp = t < B - 1 ? t + 1 : B - 1;
  uint32_t e = 0;
  double cdt_max = -1.0;
#pragma unroll
  for (int s = 0; s < NST; s++) {
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 5; q++) sV[q][t] = v[q];
    __syncthreads();
    if (s > 0 && ghost) {
#pragma unroll
      for (int q = 0; q < 5; q++) v[q] = sV[q][sp];
      if (flip) v[1] = -v[1];
    }
    if (s > 0 && !periodic) {
      __syncthreads();
#pragma unroll
      for (int q = 0; q < 5; q++) sV[q][t] = v[q];
      __syncthreads();
    }
    double vr[5], vl[5];
#pragma unroll
    for (int q = 0; q < 5; q++) {
      const double d = plm_slope<double, LIM>(sV[q][tm], v[q], sV[q][tp]);
      vr[q] = v[q] - 0.5*d;                           // this cell's side of its lower face
      sL[q][t] = v[q] + 0.5*d;
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 5; q++) vl[q] = sL[q][tm];
    FaceFlux<double> f;
    hd_riemann<0, SOLVER>(vl, vr, gamma, f);
    const double cm = rmax(rabs(f.Sl), rabs(f.Sr));
    // the faces of the block's own cells
    if (t >= H && t <= B - H && i <= nx) e |= f.err;
#pragma unroll
    for (int q = 0; q < 5; q++) sF[q][t] = f.f[q];
    sF[5][t] = cm;
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 5; q++) {
      double du = -dtdx*(sF[q][tp] - f.f[q]);
      du += 0.0;
      u[q] = s == 0 ? u0[q] + ws[0].wR*du : ws[s].w0*u0[q] + ws[s].w1*u[q] + ws[s].wR*du;
    }
    if (s == 0 && own) cdt_max = 0.5*(cm + sF[5][tp])/g.dx;
    const uint32_t ce = hd_cons_to_prim(u, gamma - 1.0, small_rho, small_prs, v);
    if (own) {
      e |= ce;
      zone_report(b.zr[s], (size_t)i, ce);
    }
  }
  if (own) {
#pragma unroll
    for (int q = 0; q < 5; q++) { b.Uout[q*n + i] = u[q]; b.Vout[q*n + i] = v[q]; }
  }
  report_bits(b.err, e);
  const double m = block_max(cdt_max, red);
  if (t == 0) {
    const unsigned long long was =
        __hip_atomic_exchange((unsigned long long *)b.cdt_part + blockIdx.x, __double_as_longlong(m),
                              __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s_last = arrive(st.arrived, was);
  }
  __syncthreads();
  if (s_last)
    step_control(st, dt, gridDim.x, 1, red, [&](int q) {
      return __hip_atomic_load(b.cdt_part + q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    });
}

template <int LIM, int SOLVER>
void stage_t(const HdBufs &b, const HdBox &g, const HdStep &st, RKW w, int first_stage, int want_dt,
             double gamma, double small_rho, double small_prs, hipStream_t s)
{
  const int nb = hd_blocks(g, 0), L = hd_march_cells(g);
  auto go = [&](auto kernel, int threads) {
    hipLaunchKernelGGL(kernel, dim3(nb), dim3(threads), 0, s, g, L, b, st, w, first_stage, want_dt, nb,
                       gamma, small_rho, small_prs);
  };
  const bool wide = g.ncell >= 1 << 29;        // an array slot of 4 GiB or more
  if (g.dims == 2)
    wide ? go(k_hd_stage2d<LIM, SOLVER, size_t>, 256) : go(k_hd_stage2d<LIM, SOLVER, unsigned>, 256);
  else
    wide ? go(k_hd_stage3d<LIM, SOLVER, size_t>, 64*NW) : go(k_hd_stage3d<LIM, SOLVER, unsigned>, 64*NW);
}

template <int LIM, int SOLVER>
void sweep_t(int dir, const HdBufs &b, const HdBox &g, const StepCtl *ctl, RKW w, int first_stage, int want_dt,
             double gamma, double small_rho, double small_prs, hipStream_t s)
{
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(hd_blocks(g, 0)), dim3(hd_sweep_block(g)), 0, s, g, b, ctl, w, first_stage,
                       want_dt, gamma, small_rho, small_prs);
  };
  if (dir == 0)         go(k_hd_sweep<0, false, LIM, SOLVER>);
  else if (dir == 2)    go(k_hd_sweep<2, true, LIM, SOLVER>);
  else if (g.dims == 2) go(k_hd_sweep<1, true, LIM, SOLVER>);
  else                  go(k_hd_sweep<1, false, LIM, SOLVER>);
}

template <int LIM, int SOLVER, int NST>
void step1d_t(const HdBufs &b, const HdBox &g, const HdStep &st, double gamma, double small_rho,
              double small_prs, hipStream_t s)
{
  const int nb = hd_blocks(g, NST);
  if (hd_block1d(g) == 64)
    hipLaunchKernelGGL((k_hd_step1d<LIM, SOLVER, NST, 64>), dim3(nb), dim3(64), 0, s, g, b, st, gamma,
                       small_rho, small_prs);
  else
    hipLaunchKernelGGL((k_hd_step1d<LIM, SOLVER, NST, 256>), dim3(nb), dim3(256), 0, s, g, b, st, gamma,
                       small_rho, small_prs);
}

}  // namespace

void hd_launch_stage(const HdBufs &b, const HdBox &g, const HdStep &st, RKW w, int first_stage,
                     int want_dt, int limiter, int solver, double gamma, double small_rho,
                     double small_prs, hipStream_t s)
{
  if (limiter == MC_LIM) {
    if (solver == 2) stage_t<MC_LIM, 2>(b, g, st, w, first_stage, want_dt, gamma, small_rho, small_prs, s);
    else             stage_t<MC_LIM, 1>(b, g, st, w, first_stage, want_dt, gamma, small_rho, small_prs, s);
  } else {
    if (solver == 2) stage_t<VANLEER_LIM, 2>(b, g, st, w, first_stage, want_dt, gamma, small_rho, small_prs, s);
    else             stage_t<VANLEER_LIM, 1>(b, g, st, w, first_stage, want_dt, gamma, small_rho, small_prs, s);
  }
}

void hd_launch_sweep(int dir, const HdBufs &b, const HdBox &g, const StepCtl *ctl, RKW w, int first_stage,
                     int want_dt, int limiter, int solver, double gamma, double small_rho,
                     double small_prs, hipStream_t s)
{
  if (limiter == MC_LIM) {
    if (solver == 2) sweep_t<MC_LIM, 2>(dir, b, g, ctl, w, first_stage, want_dt, gamma, small_rho, small_prs, s);
    else             sweep_t<MC_LIM, 1>(dir, b, g, ctl, w, first_stage, want_dt, gamma, small_rho, small_prs, s);
  } else {
    if (solver == 2) sweep_t<VANLEER_LIM, 2>(dir, b, g, ctl, w, first_stage, want_dt, gamma, small_rho, small_prs, s);
    else             sweep_t<VANLEER_LIM, 1>(dir, b, g, ctl, w, first_stage, want_dt, gamma, small_rho, small_prs, s);
  }
}

template <int NST>
static void step1d_n(const HdBufs &b, const HdBox &g, const HdStep &st, int limiter, int solver,
                     double gamma, double small_rho, double small_prs, hipStream_t s)
{
  if (limiter == MC_LIM) {
    if (solver == 2) step1d_t<MC_LIM, 2, NST>(b, g, st, gamma, small_rho, small_prs, s);
    else             step1d_t<MC_LIM, 1, NST>(b, g, st, gamma, small_rho, small_prs, s);
  } else {
    if (solver == 2) step1d_t<VANLEER_LIM, 2, NST>(b, g, st, gamma, small_rho, small_prs, s);
    else             step1d_t<VANLEER_LIM, 1, NST>(b, g, st, gamma, small_rho, small_prs, s);
  }
}

void hd_launch_step1d(const HdBufs &b, const HdBox &g, const HdStep &st, int nst, int limiter,
                      int solver, double gamma, double small_rho, double small_prs, hipStream_t s)
{
  if (nst == 3) step1d_n<3>(b, g, st, limiter, solver, gamma, small_rho, small_prs, s);
  else          step1d_n<2>(b, g, st, limiter, solver, gamma, small_rho, small_prs, s);
}

}  // namespace gpl
