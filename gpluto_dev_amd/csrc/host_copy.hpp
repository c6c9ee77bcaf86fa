// Device-to-host transfer of state arrays into a caller's (pageable) arrays.
//
// A field is one variable over the active zones, i fastest.
//  * Up to 1 MiB (kSmall) one kernel writes every field into a pinned buffer, made
//    with the context; one wait, then the caller's arrays.  Copies of the fields
//    by themselves cost 5 to 20 us each, and some runs of them 60 to 100: us a
//    download, 1D 100 zones 40 -> 15, 4096 zones 150 -> 27, 10^3 MHD 65 -> 21, 16^3 300
//    -> 41, 18x17x16 77 -> 46, 60^2 mixed with ghosts 97 -> 38.  Vc of HD, stored as it
//    leaves, takes the launch too: one copy of 1052 zones is 11 us or, after another
//    context's large transfers, 45; the launch 15 both times (4096 zones 16 and 20).
//  * Above, the fields are cut into chunks of an eighth of the state, 1 to 16 MiB; a
//    chunk is copied into one of kSlots pinned buffers (where the stored array is FP32
//    or holds ghost layers, written there by the gather kernel), and while later chunks
//    are on their way, helper threads move it to the caller's arrays.  256^3, the
//    eleven arrays of Vc and Vs (1.48 GB): 422 ms with pageable copies into host
//    vectors and element loops, 27.6 this way (a pinned copy alone is 26); 128^3 55 ->
//    3.7.  Chunks below 1 MiB cost more in waits than they overlap (24^3 196 -> 126
//    us).  A device buffer between gather and copy is no faster: Vc, Vs and Uc of
//    192^3 mixed 21.4 ms with, 20.4 without, 128^3 mixed with ghosts 6.5 and 6.3, 24^3
//    mixed 115 and 94 us.
//
// The buffers belong to one context (no sharing between contexts or threads): the
// small one is allocated with it, the others at its first larger transfer, at most
// kSlots chunks of 16 MiB, and are freed with it; no device memory.  Where they cannot
// be had (a limit on locked memory) the transfer does without: pageable copies,
// unpacked on the host where a gather would be needed.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <vector>

namespace gpl {

// Where the active zones lie in a stored array: element (i, j, k) at
// off + (i + lo[0]) + sx*((j + lo[1]) + sy*(k + lo[2])).
struct FieldGeom {
  size_t off;
  int sx, sy;
  int lo[3], n[3];
  bool whole;        // the array is the active zones and nothing else
};

struct FieldOut {
  const void *src;   // device array, at element 0 of the box's storage (before off)
  bool f32;          // float, else double
  double *dst;       // host array of n[0]*n[1]*n[2] doubles
};

class HostCopy {
public:
  ~HostCopy();
  // Every field of `out` to the host, behind the work already on the stream;
  // returns when the arrays are filled.  0 or GPL_EHIP.
  int fetch(const FieldGeom &g, const std::vector<FieldOut> &out, hipStream_t s);
  // Before the first transfer of at most `total` doubles: a small state's buffer
  void prepare(size_t total);

private:
  static constexpr int kSlots = 4;
  static constexpr size_t kChunk = size_t(1) << 21;   // doubles per slot at most: 16 MiB
  static constexpr size_t kSmall = size_t(1) << 17;   // doubles of a small state at most: 1 MiB
  static constexpr size_t kRows = size_t(1) << 18;    // doubles of fetch_rows' host buffer
  bool pinned(size_t bytes);
  bool reserve(size_t chunk, int slots);
  int fetch_small(const FieldGeom &g, const std::vector<FieldOut> &out, hipStream_t s);
  int fetch_whole(const FieldGeom &g, const std::vector<FieldOut> &out, hipStream_t s);   // no gather needed
  int fetch_rows(const FieldGeom &g, const std::vector<FieldOut> &out, hipStream_t s);
  double *pin = nullptr;
  size_t pin_cap = 0;                                  // bytes
  hipEvent_t done[kSlots] = {};
};

// dst[t] = element t0 + t of the fields laid one after the other, in FP64, for t <
// count; at most kFields of them.  dst: pinned host memory.
constexpr int kFields = 24;
hipError_t launch_fields_gather(const FieldGeom &g, const std::vector<FieldOut> &out, size_t t0, size_t count,
                                double *dst, hipStream_t s);

}  // namespace gpl
