// Device-to-host transfer of state arrays: see host_copy.hpp.
#include "host_copy.hpp"
#include "../../include/gpluto_amd.h"

#include <sched.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <thread>

namespace gpl {

namespace {

// cores this thread may run on
int cores()
{
  cpu_set_t set;
  return sched_getaffinity(0, sizeof(set), &set) == 0 ? CPU_COUNT(&set) : 1;
}

// Moves chunks from pinned memory to the caller's arrays: the calling thread and
// up to kHelpers more, each taking pieces of the chunk on offer.  No more threads
// than cores: one without a core of its own only takes turns with the others.
// Helpers that cannot be started are simply missing.
class Movers {
public:
  explicit Movers(size_t total)
  {
    // a helper pays for itself from some megabytes on
    const int most = total >= (size_t(32) << 20) ? kHelpers : (total >= (size_t(4) << 20) ? 2 : 0);
    const int want = most == 0 ? 0 : std::min(most, cores() - 1);
    try {
      helpers.reserve(want);
      for (int q = 0; q < want; q++) helpers.emplace_back([this] { serve(); });
    } catch (...) {
    }
  }
  ~Movers()
  {
    {
      std::lock_guard<std::mutex> l(m);
      quit = true;
    }
    cv.notify_all();
    for (auto &t : helpers) t.join();
  }
  void move(void *dst, const void *src, size_t bytes)
  {
    if (helpers.empty()) { memcpy(dst, src, bytes); return; }
    {
      std::lock_guard<std::mutex> l(m);
      to = (char *)dst; from = (const char *)src; size = bytes;
      // enough pieces for every thread, of 256 KiB at least: a chunk of 1 MiB in one
      // piece left the helpers idle (HD 511x333 278 -> 335 us a download, 270 in four)
      piece = std::min(std::max(bytes/16, kPiece/4), kPiece);
      next.store(0);
      busy = (int)helpers.size();
      round++;
    }
    cv.notify_all();
    work();
    std::unique_lock<std::mutex> l(m);
    idle.wait(l, [this] { return busy == 0; });
  }

private:
  static constexpr int kHelpers = 7;
  static constexpr size_t kPiece = size_t(1) << 20;
  void work()
  {
    for (;;) {
      const size_t o = next.fetch_add(piece);
      if (o >= size) return;
      memcpy(to + o, from + o, size - o < piece ? size - o : piece);
    }
  }
  void serve()
  {
    unsigned long seen = 0;
    std::unique_lock<std::mutex> l(m);
    for (;;) {
      cv.wait(l, [&] { return quit || round != seen; });
      if (quit) return;
      seen = round;
      l.unlock();
      work();
      l.lock();
      if (--busy == 0) idle.notify_one();
    }
  }
  std::vector<std::thread> helpers;
  std::mutex m;
  std::condition_variable cv, idle;
  std::atomic<size_t> next{0};
  char *to = nullptr;
  const char *from = nullptr;
  size_t size = 0, piece = kPiece;
  unsigned long round = 0;
  int busy = 0;
  bool quit = false;
};

// part of a run of fields that are adjacent at the caller's and, unless the gather
// kernel collects them, on the device
struct Piece {
  const double *src;
  double *dst;
  size_t count, at;  // doubles; offset in its slot
};

}  // namespace

HostCopy::~HostCopy()
{
  if (pin) (void)hipHostFree(pin);
  for (hipEvent_t e : done) if (e) (void)hipEventDestroy(e);
}

bool HostCopy::pinned(size_t bytes)
{
  if (pin_cap >= bytes) return true;
  if (pin) (void)hipHostFree(pin);
  pin = nullptr;
  pin_cap = 0;
  if (hipHostMalloc((void **)&pin, bytes, hipHostMallocDefault) != hipSuccess) {
    pin = nullptr;
    (void)hipGetLastError();                   // dealt with by the caller: not for a later check to find
    return false;
  }
  pin_cap = bytes;
  return true;
}

bool HostCopy::reserve(size_t slot, int slots)
{
  if (!pinned(slots*slot*sizeof(double))) return false;
  for (int q = 0; q < slots; q++)
    if (!done[q] && hipEventCreateWithFlags(&done[q], hipEventDisableTiming) != hipSuccess) {
      done[q] = nullptr;
      (void)hipGetLastError();
      return false;
    }
  return true;
}

void HostCopy::prepare(size_t total)
{
  // touched here: a page's first access costs more than its copy
  if (total <= kSmall && pinned(total*sizeof(double))) memset(pin, 0, total*sizeof(double));
}

int HostCopy::fetch_small(const FieldGeom &g, const std::vector<FieldOut> &out, hipStream_t s)
{
  const size_t n = (size_t)g.n[0]*g.n[1]*g.n[2], nf = out.size();
  if (launch_fields_gather(g, out, 0, nf*n, pin, s) != hipSuccess || hipStreamSynchronize(s) != hipSuccess)
    return GPL_EHIP;
  for (size_t q = 0; q < nf;) {
    size_t run = 1;                            // arrays that follow one another at the caller's
    while (q + run < nf && out[q + run].dst == out[q].dst + run*n) run++;
    memcpy(out[q].dst, pin + q*n, run*n*sizeof(double));
    q += run;
  }
  return 0;
}

int HostCopy::fetch_whole(const FieldGeom &g, const std::vector<FieldOut> &out, hipStream_t s)
{
  const size_t n = (size_t)g.n[0]*g.n[1]*g.n[2];
  for (size_t q = 0; q < out.size();) {
    size_t run = 1;                            // fields that follow one another on both sides
    while (q + run < out.size() && out[q + run].dst == out[q].dst + run*n &&
           (const double *)out[q + run].src == (const double *)out[q].src + run*n)
      run++;
    if (hipMemcpyAsync(out[q].dst, (const double *)out[q].src + g.off, run*n*sizeof(double),
                       hipMemcpyDeviceToHost, s) != hipSuccess)
      return GPL_EHIP;
    q += run;
  }
  return hipStreamSynchronize(s) == hipSuccess ? 0 : GPL_EHIP;
}

int HostCopy::fetch_rows(const FieldGeom &g, const std::vector<FieldOut> &out, hipStream_t s)
{
  // whole stored rows of a plane at a time, about 2 MiB or one row
  const int most = (int)(kRows/(size_t)g.sx), rows = most < 1 ? 1 : (most < g.n[1] ? most : g.n[1]);
  std::vector<double> buf((size_t)rows*g.sx);
  for (const FieldOut &f : out) {
    const size_t es = f.f32 ? sizeof(float) : sizeof(double);
    for (int k = 0; k < g.n[2]; k++)
      for (int j0 = 0; j0 < g.n[1]; j0 += rows) {
        const int m = g.n[1] - j0 < rows ? g.n[1] - j0 : rows;
        const size_t at = g.off + (size_t)g.sx*((size_t)(j0 + g.lo[1]) + (size_t)g.sy*(k + g.lo[2]));
        if (hipMemcpyAsync(buf.data(), (const char *)f.src + at*es, (size_t)m*g.sx*es, hipMemcpyDeviceToHost,
                           s) != hipSuccess ||
            hipStreamSynchronize(s) != hipSuccess)
          return GPL_EHIP;
        for (int j = 0; j < m; j++) {
          double *d = f.dst + ((size_t)k*g.n[1] + j0 + j)*g.n[0];
          const size_t o = (size_t)j*g.sx + g.lo[0];
          if (f.f32) for (int i = 0; i < g.n[0]; i++) d[i] = (double)((const float *)buf.data())[o + i];
          else       memcpy(d, buf.data() + o, (size_t)g.n[0]*sizeof(double));
        }
      }
  }
  return 0;
}

int HostCopy::fetch(const FieldGeom &g, const std::vector<FieldOut> &out, hipStream_t s)
{
  const size_t n = (size_t)g.n[0]*g.n[1]*g.n[2], total = n*out.size();
  if (!total) return 0;
  bool gather = !g.whole;
  for (const FieldOut &f : out) gather = gather || f.f32;
  const bool fits = out.size() <= kFields;     // the gather kernel's set
  if (total <= kSmall && fits && pinned(total*sizeof(double))) return fetch_small(g, out, s);
  // a larger state in slots of an eighth of it, 1 MiB at least, 16 MiB at most
  const size_t slot = std::min(std::max((total + 7)/8, kSmall), kChunk);
  const int slots = (int)std::min((total + slot - 1)/slot, (size_t)kSlots);
  if (total <= kSmall || (gather && !fits) || !reserve(slot, slots))
    return gather ? fetch_rows(g, out, s) : fetch_whole(g, out, s);
  // groups of pieces, one group per slot
  std::vector<std::vector<Piece>> groups;
  size_t used = slot;
  for (const FieldOut &f : out) {
    const double *src = gather ? nullptr : (const double *)f.src + g.off;
    for (size_t e = 0; e < n;) {
      if (used == slot) { groups.emplace_back(); used = 0; }
      const size_t c = std::min(n - e, slot - used);
      Piece *last = groups.back().empty() ? nullptr : &groups.back().back();
      if (last && last->dst + last->count == f.dst + e && (gather || last->src + last->count == src + e))
        last->count += c;
      else
        groups.back().push_back({gather ? nullptr : src + e, f.dst + e, c, used});
      e += c;
      used += c;
    }
  }
  const int ng = (int)groups.size();
  Movers movers(total*sizeof(double));
  auto send = [&](int k) -> bool {
    double *hp = pin + (size_t)(k % kSlots)*slot;
    if (gather) {
      const size_t t0 = (size_t)k*slot;
      if (launch_fields_gather(g, out, t0, std::min(slot, total - t0), hp, s) != hipSuccess) return false;
    } else {
      for (const Piece &p : groups[k])
        if (hipMemcpyAsync(hp + p.at, p.src, p.count*sizeof(double), hipMemcpyDeviceToHost, s) != hipSuccess)
          return false;
    }
    return hipEventRecord(done[k % kSlots], s) == hipSuccess;
  };
  bool ok = true;
  int sent = 0;
  for (int k = 0; k < ng && ok; k++) {
    while (ok && sent < ng && sent < k + kSlots) { ok = send(sent); sent++; }
    ok = ok && hipEventSynchronize(done[k % kSlots]) == hipSuccess;
    if (!ok) break;
    const double *hp = pin + (size_t)(k % kSlots)*slot;
    for (const Piece &p : groups[k]) movers.move(p.dst, hp + p.at, p.count*sizeof(double));
  }
  if (!ok) (void)hipStreamSynchronize(s);     // nothing is in flight into the buffers afterwards
  return ok ? 0 : GPL_EHIP;
}

}  // namespace gpl
