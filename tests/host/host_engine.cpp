// The library's host side (C ABI, engines, transfers) on the CPU: linked with
// gpl_api.cpp, engine_*.cpp, host_copy.cpp and dbl_io.cpp in place of the HIP
// runtime and of the kernels.  "Device" memory is host memory, streams are the
// calling thread, kernel launches are recorded and compute nothing, except the
// field gather.  A test can let allocations fail.
#include "../../gpluto_dev_amd/csrc/batch2d.hpp"
#include "../../gpluto_dev_amd/csrc/c2p_net.hpp"
#include "../../gpluto_dev_amd/csrc/diagnostics.hpp"
#include "../../gpluto_dev_amd/csrc/engine.hpp"
#include "../../gpluto_dev_amd/csrc/hd.hpp"
#include "../../gpluto_dev_amd/csrc/mhd3d.hpp"

#include <dirent.h>
#include <stdlib.h>
#include <string.h>
#include <sys/mman.h>

#include <algorithm>
#include <map>
#include <vector>

namespace {

struct Launch { int kernel, value[8]; };       // what a launcher was asked for
std::vector<Launch> launches;
std::map<void *, size_t> live_dev, live_pin;
size_t dev_limit = ~size_t(0), pin_limit = ~size_t(0);
int threads_seen = 0, copies = 0;
const void *hd_arrived = nullptr, *hd_u[2] = {};

size_t held(const std::map<void *, size_t> &m)
{
  size_t s = 0;
  for (const auto &p : m) s += p.second;
  return s;
}
hipError_t last = hipSuccess;
hipError_t fail(hipError_t e) { last = e; return e; }

hipError_t take(std::map<void *, size_t> &live, size_t limit, void **p, size_t n)
{
  if (held(live) + n > limit) { *p = nullptr; return fail(hipErrorOutOfMemory); }
  // zero pages, none of them there before it is touched
  *p = mmap(nullptr, n ? n : 1, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0);
  if (*p == MAP_FAILED) { *p = nullptr; return fail(hipErrorOutOfMemory); }
  live[*p] = n;
  return hipSuccess;
}
hipError_t give(std::map<void *, size_t> &live, void *p)
{
  if (!p) return hipSuccess;
  const auto at = live.find(p);
  if (at == live.end()) return fail(hipErrorInvalidValue);
  munmap(p, at->second ? at->second : 1);
  live.erase(at);
  return hipSuccess;
}
int threads_now()
{
  int n = 0;
  if (DIR *d = opendir("/proc/self/task")) {
    while (dirent *e = readdir(d)) n += e->d_name[0] != '.';
    closedir(d);
  }
  return n;
}
// handles: a byte each
template <typename H> hipError_t make(H *h) { *h = (H)malloc(1); return hipSuccess; }
template <typename H> hipError_t drop(H h) { free((void *)h); return hipSuccess; }

}  // namespace

// --------------------------------------------------------------------------
// the HIP runtime calls that the host side makes
// --------------------------------------------------------------------------
extern "C" {
hipError_t hipMalloc(void **p, size_t n) { return take(live_dev, dev_limit, p, n); }
hipError_t hipFree(void *p) { return give(live_dev, p); }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return take(live_pin, pin_limit, p, n); }
hipError_t hipHostFree(void *p) { return give(live_pin, p); }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind)
{
  memcpy(d, s, n);
  copies++;
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t)
{
  memcpy(d, s, n);
  copies++;
  return hipSuccess;
}
hipError_t hipMemset(void *d, int v, size_t n) { memset(d, v, n); return hipSuccess; }
hipError_t hipGetLastError(void) { const hipError_t e = last; last = hipSuccess; return e; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return make(s); }
hipError_t hipStreamDestroy(hipStream_t s) { return drop(s); }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) { return make(g); }
hipError_t hipEventCreate(hipEvent_t *e) { return make(e); }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return make(e); }
hipError_t hipEventDestroy(hipEvent_t e) { return drop(e); }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { threads_seen = std::max(threads_seen, threads_now()); return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { *ms = 1.f; return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *, char *, size_t) { return make(e); }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t g) { return drop(g); }
hipError_t hipGraphExecDestroy(hipGraphExec_t e) { return drop(e); }
}

// --------------------------------------------------------------------------
// the kernels' launchers
// --------------------------------------------------------------------------
namespace gpl {

void launch_zone_reset(unsigned long long *, hipStream_t) {}
void launch_dt(const double *, int nparts, double, StepCtl *, double, double, int, hipStream_t)
{
  launches.push_back({K_DT, {nparts}});
}

template <typename R>
void mhd3d_launch(int which, const Mhd3dBufs<R> &b, const Box3 &, const StepCtl *, RKW, int, int, int, int,
                  double, double, double, hipStream_t)
{
  launches.push_back({which, {b.march[0], b.march[1], b.rows, b.cols[0], b.cols[1], b.emf_march}});
}
template void mhd3d_launch<double>(int, const Mhd3dBufs<double> &, const Box3 &, const StepCtl *, RKW, int, int,
                                   int, int, double, double, double, hipStream_t);
template void mhd3d_launch<float>(int, const Mhd3dBufs<float> &, const Box3 &, const StepCtl *, RKW, int, int,
                                  int, int, double, double, double, hipStream_t);
template <typename R> void mhd3d_boundary(const Box3 &, const int *, R *, double *, hipStream_t) {}
template void mhd3d_boundary<double>(const Box3 &, const int *, double *, double *, hipStream_t);
template void mhd3d_boundary<float>(const Box3 &, const int *, float *, double *, hipStream_t);
template <typename R>
void mhd3d_dump_gather(const Box3 &, const int *, const int *, const R *, const double *, double *, hipStream_t) {}
template void mhd3d_dump_gather<double>(const Box3 &, const int *, const int *, const double *, const double *,
                                        double *, hipStream_t);
template void mhd3d_dump_gather<float>(const Box3 &, const int *, const int *, const float *, const double *,
                                       double *, hipStream_t);
int mhd3d_blocks(const Box3 &g) { return (g.ncell + 255)/256; }
int mhd3d_march_blocks(const Box3 &g, int march)
{
  return (int)(((long long)g.nx*g.ny*((g.nz + march - 1)/march) + 255)/256);
}

// kernel ids of the 2D launches: 100 + phase
template <typename R>
void batch2d_launch(int phase, const Batch2dBufs<R> &b, RKW, int, int, int, int, int march, int blocks, double,
                    double, double, hipStream_t)
{
  launches.push_back({100 + phase, {march, blocks, b.tile_lanes}});
}
template void batch2d_launch<double>(int, const Batch2dBufs<double> &, RKW, int, int, int, int, int, int, double,
                                     double, double, hipStream_t);
template void batch2d_launch<float>(int, const Batch2dBufs<float> &, RKW, int, int, int, int, int, int, double,
                                    double, double, hipStream_t);
template <typename R>
void batch2d_boundary(const BoxDesc *, int, int, const int *, R *, double *, size_t, hipStream_t) {}
template void batch2d_boundary<double>(const BoxDesc *, int, int, const int *, double *, double *, size_t, hipStream_t);
template void batch2d_boundary<float>(const BoxDesc *, int, int, const int *, float *, double *, size_t, hipStream_t);
template <typename R>
void batch2d_dump_gather(const BoxDesc &, const int *, const R *, const double *, size_t, double *, hipStream_t) {}
template void batch2d_dump_gather<double>(const BoxDesc &, const int *, const double *, const double *, size_t,
                                          double *, hipStream_t);
template void batch2d_dump_gather<float>(const BoxDesc &, const int *, const float *, const double *, size_t,
                                         double *, hipStream_t);
void batch2d_launch_dt(const double *, const int *, int, StepCtl *, double, double, int, hipStream_t) {}

// HD launches: 200 a stage, 201 a 1D step, 210 + direction a sweep
static void hd_seen(const HdBufs &b, const HdStep &st)
{
  hd_arrived = st.arrived;
  hd_u[0] = b.U0;
  hd_u[1] = b.Uout;
}
void hd_launch_stage(const HdBufs &b, const HdBox &, const HdStep &st, RKW, int, int, int, int, double, double,
                     double, hipStream_t)
{
  hd_seen(b, st);
  launches.push_back({200, {}});
}
void hd_launch_step1d(const HdBufs &b, const HdBox &, const HdStep &st, int, int, int, double, double, double,
                      hipStream_t)
{
  hd_seen(b, st);
  launches.push_back({201, {}});
}

void hd_launch_sweep(int dir, const HdBufs &, const HdBox &, const StepCtl *, RKW, int, int, int, int, double, double,
                     double, hipStream_t)
{
  launches.push_back({210 + dir, {}});
}

template <typename R>
void launch_diagnostics(const DiagBox &, const R *, const double *, double *, double *, hipStream_t) {}
template void launch_diagnostics<double>(const DiagBox &, const double *, const double *, double *, double *, hipStream_t);
template void launch_diagnostics<float>(const DiagBox &, const float *, const double *, double *, double *, hipStream_t);
int net_pack_upload(const float *, float *, NetPack *, hipStream_t) { return GPL_EUNSUPPORTED; }

hipError_t launch_fields_gather(const FieldGeom &g, const std::vector<FieldOut> &out, size_t t0, size_t count,
                                double *dst, hipStream_t)
{
  const size_t n = (size_t)g.n[0]*g.n[1]*g.n[2];
  for (size_t t = t0; t < t0 + count; t++) {
    const size_t q = t/n, e = t % n, r = e/g.n[0];
    const int i = (int)(e % g.n[0]), j = (int)(r % g.n[1]), k = (int)(r/g.n[1]);
    const size_t o = g.off + (size_t)(i + g.lo[0]) +
                     (size_t)g.sx*((size_t)(j + g.lo[1]) + (size_t)g.sy*(k + g.lo[2]));
    dst[t - t0] = out[q].f32 ? (double)((const float *)out[q].src)[o] : ((const double *)out[q].src)[o];
  }
  return hipSuccess;
}

}  // namespace gpl

// --------------------------------------------------------------------------
// for the tests
// --------------------------------------------------------------------------
extern "C" {
// bytes that device / pinned allocations may hold from now on
void he_limits(size_t dev, size_t pin) { dev_limit = dev; pin_limit = pin; }
size_t he_held(int pinned) { return held(pinned ? live_pin : live_dev); }
void he_set_last_error(int e) { last = (hipError_t)e; }
int he_last_error() { return (int)last; }
int he_copies() { const int n = copies; copies = 0; return n; }
int he_threads(int reset) { const int n = threads_seen; if (reset) threads_seen = 0; return n; }
int he_launches(int *out, int most)            // rows of 9, the newest `most`; clears the record
{
  const int n = (int)launches.size(), k = n < most ? n : most;
  for (int q = 0; q < k; q++) memcpy(out + 9*q, &launches[n - k + q], 9*sizeof(int));
  launches.clear();
  return k;
}
const void *he_hd_arrived() { return hd_arrived; }
const void *he_hd_u(int which) { return hd_u[which]; }

// the learned con2prim start is left out of this build
int gpl_c2p_net_size(void) { return 0; }
int gpl_c2p_net_make_data(int, uint64_t, int, double, double *, float *, float *) { return GPL_EUNSUPPORTED; }
int gpl_c2p_net_pairs(int, const double *, const double *, int, double, float *, float *) { return GPL_EUNSUPPORTED; }
int gpl_c2p_net_fit(int, uint64_t, const float *, const float *, int, int, int, float, float *, float *)
{
  return GPL_EUNSUPPORTED;
}
int gpl_c2p_net_train(int, uint64_t, int, int, int, float, double, float *, float *) { return GPL_EUNSUPPORTED; }
int gpl_c2p_net_grad(int, const float *, const float *, const float *, int, float *, float *) { return GPL_EUNSUPPORTED; }
int gpl_c2p_net_infer(int, const float *, const float *, int, float *) { return GPL_EUNSUPPORTED; }
int gpl_c2p_solve(int, const float *, const double *, int, double, double *, int *, uint32_t *, double *, int *)
{
  return GPL_EUNSUPPORTED;
}
int gpl_c2p_solve_noalloc(int, const float *, const double *, int, double, double *, int *, uint32_t *, int *)
{
  return GPL_EUNSUPPORTED;
}
}
