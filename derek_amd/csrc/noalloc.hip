// Allocation-free overlap, for callers that cannot call hipMalloc (code under
// HIP graph capture, tight serving loops, harnesses that forbid it): the
// split-K partial sums of S = X^H Y go to a buffer that derek_hip_init
// allocates (kNoAllocScratchElems double2, 32 MiB) instead of one the call
// would have to.  Every partial the reduction reads is written by the product
// kernel of the same call, so nothing has to be cleared between calls.
//
// Order.  The operands are the caller's and nothing else in the library touches
// them or the buffer, so the kernels go to the caller's stream: X and Y are
// written before and S is read and the memory reused after, as with any kernel
// launched there.  (Left on the context's non-blocking stream the overlap ran
// beside both, and with one buffer for every context beside the overlaps of
// other contexts: wrong sums.)  A caller that has asked for the context's stream
// may order its work on that, so from then on the kernels run there, between
// two waits on events made at init: after what the caller's stream holds, before
// what it is given next.
// A pass of 1503 x 10: 11 us on the caller's stream, 35 us with the two
// waits (a hop between two queues takes about 12 us).
#include "context.hpp"

namespace derek {

void NoAlloc::init() {
  work = dmalloc<double2>(kNoAllocScratchElems);
  DEREK_HIP(hipEventCreateWithFlags(&ready, hipEventDisableTiming));
  DEREK_HIP(hipEventCreateWithFlags(&done, hipEventDisableTiming));
  // the overlap kernels' resident-slot queries run here, not inside the
  // allocation-free call
  (void)overlap_work_elems(1, 1, 1, 1);
}

NoAlloc::~NoAlloc() {
  if (pending) (void)(last ? hipEventSynchronize(done) : hipStreamSynchronize(nullptr));
  dfree(work);
  for (hipEvent_t e : {ready, done})
    if (e) (void)hipEventDestroy(e);
}

// `to` waits for the latest overlap on a caller's stream
void NoAlloc::order(hipStream_t to) {
  if (!last) DEREK_HIP(hipEventRecord(ready, nullptr));
  DEREK_HIP(hipStreamWaitEvent(to, last ? done : ready, 0));
}

void NoAlloc::share(hipStream_t s) {
  if (pending) order(s);
  pending = false;
  shared = true;
}

void NoAlloc::sync() {
  if (!pending) return;
  DEREK_HIP(last ? hipEventSynchronize(done) : hipStreamSynchronize(nullptr));
  pending = false;
}

namespace {
// the context's device current for the scope (the null stream is the current device's)
struct OnDevice {
  int prev = -1;
  explicit OnDevice(int dev) {
    int cur = 0;
    DEREK_HIP(hipGetDevice(&cur));
    if (cur == dev) return;
    DEREK_HIP(hipSetDevice(dev));
    prev = cur;
  }
  ~OnDevice() {
    if (prev >= 0) (void)hipSetDevice(prev);
  }
};

// the null stream takes no part in a capture
bool capturing(hipStream_t s) {
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  if (s) DEREK_HIP(hipStreamIsCapturing(s, &st));
  return st != hipStreamCaptureStatusNone;
}
}  // namespace

void overlap_noalloc(derek_ctx* c, hipStream_t caller, int64_t npw, int m, int n, const double2* X, const double2* Y,
                     double2* S) {
  const int64_t mn = (int64_t)m * n;
  DEREK_REQUIRE(mn <= kNoAllocScratchElems, "overlap_noalloc: m * n = " + std::to_string(mn) +
                                                " exceeds the scratch capacity of " +
                                                std::to_string(kNoAllocScratchElems) + " complex values");
  const int64_t max_chunks = kNoAllocScratchElems / mn;
  const bool herm = (X == Y) && (m == n);
  const OnDevice on(c->device);
  NoAlloc& w = c->noalloc;
  // launched directly: the profiler's event pool may create events
  auto product = [&](hipStream_t s) {
    overlap<double>(X, npw, 0, Y, npw, 0, m, n, npw, nullptr, S, m, 0, 1, w.work, kNoAllocScratchElems, herm, s, 0,
                    max_chunks);
  };
  if (w.shared) {
    // recorded into a graph on the context's stream, the order on it is the graph's
    const bool wait = caller ? caller != c->s : !capturing(c->s);
    if (wait) {
      DEREK_HIP(hipEventRecord(w.ready, caller));
      DEREK_HIP(hipStreamWaitEvent(c->s, w.ready, 0));
    }
    product(c->s);
    if (wait) {
      DEREK_HIP(hipEventRecord(w.done, c->s));
      DEREK_HIP(hipStreamWaitEvent(caller, w.done, 0));
    }
    return;
  }
  const bool recorded = capturing(caller);
  // the buffer is one stream's at a time
  if (!recorded && w.pending && w.last != caller) w.order(caller);
  product(caller);
  if (recorded) return;
  if (caller) DEREK_HIP(hipEventRecord(w.done, caller));
  w.last = caller;
  w.pending = true;
}

}  // namespace derek
