// sfft_pool.hip -- scratch memory of the entry points that have no plan (dense FFT, truth
// spectrum, filter design, synthesis, metric), kept between calls.
//
// Allocating a few arrays of n points costs far more than the kernels between them (n = 2^22:
// the kernels of a truth spectrum took 130 us and its calls 0.5-4.5 ms, those of a filter design
// 0.4 ms and 3-7 ms; each hipMalloc or miss of the runtime's stream-ordered pool is 0.1 ms and
// more, and that pool gives its memory back at every synchronisation).  Here each device has a
// list of idle blocks.  A block is handed out in stream order: it carries the event its last
// user recorded when it returned the block, and the next user's stream waits for that event on
// the device, whichever stream and thread it is.  At most kKeepBytes stay idle on a device;
// blocks beyond that, and blocks that kKeepUses allocations in a row had no use for, go back to
// the runtime, and all idle blocks do when device memory cannot be allocated (dev_alloc) and when
// the caller asks for it (sfft_release_scratch).
#include <algorithm>
#include <cstdint>
#include <map>
#include <mutex>
#include <vector>

#include "sfft_internal.h"

namespace sfft {

constexpr size_t kKeepBytes = (size_t)1 << 30;   // five arrays of 2^22 complex128, with room
constexpr uint64_t kKeepUses = 512;
constexpr size_t kRound = (size_t)1 << 16;       // block sizes are multiples of this

namespace {
struct Block {
  void* p = nullptr;
  size_t bytes = 0;
  int dev = 0;
  hipEvent_t ev = nullptr;   // recorded by the last user
  uint64_t used = 0;         // allocation count when it was last returned
};
std::mutex g_mu;
std::vector<Block> g_idle;
std::map<void*, Block> g_out;   // handed out
uint64_t g_uses = 0;

// gives a block back to the runtime in st's order, after its last user's work
void give_back(const Block& b, hipStream_t st) {
  (void)hipStreamWaitEvent(st, b.ev, 0);
  (void)hipFreeAsync(b.p, st);
  (void)hipEventDestroy(b.ev);
}
}  // namespace

static bool capturing(hipStream_t st) {
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(st, &cap) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return cap != hipStreamCaptureStatusNone;
}

hipError_t work_alloc(void** p, size_t bytes, hipStream_t st) {
  *p = nullptr;
  int dev = 0;
  // a stream that is being captured takes the allocation into its graph
  if (capturing(st) || hipGetDevice(&dev) != hipSuccess) return hipMallocAsync(p, bytes, st);
  const size_t need = (bytes + kRound - 1) / kRound * kRound;
  std::lock_guard<std::mutex> lock(g_mu);
  ++g_uses;
  // the smallest block that is large enough and not more than twice as large
  int best = -1;
  for (int i = 0; i < (int)g_idle.size(); ++i)
    if (g_idle[i].dev == dev && g_idle[i].bytes >= need && g_idle[i].bytes <= 2 * need &&
        (best < 0 || g_idle[i].bytes < g_idle[best].bytes))
      best = i;
  Block b;
  if (best >= 0) {
    b = g_idle[best];
    const hipError_t e = hipStreamWaitEvent(st, b.ev, 0);
    if (e != hipSuccess) return e;   // (the block stays idle)
    g_idle.erase(g_idle.begin() + best);
  } else {
    b.bytes = need;
    b.dev = dev;
    hipError_t e = hipEventCreateWithFlags(&b.ev, hipEventDisableTiming);
    if (e != hipSuccess) return e;
    e = hipMallocAsync(&b.p, need, st);
    if (e != hipSuccess) {   // what is idle here may be what is missing
      (void)hipGetLastError();
      for (size_t i = g_idle.size(); i-- > 0;)
        if (g_idle[i].dev == dev) {
          give_back(g_idle[i], st);
          g_idle.erase(g_idle.begin() + i);
        }
      (void)hipStreamSynchronize(st);
      e = hipMallocAsync(&b.p, need, st);
    }
    if (e != hipSuccess) {
      (void)hipEventDestroy(b.ev);
      return e;
    }
  }
  g_out[b.p] = b;
  *p = b.p;
  return hipSuccess;
}

void work_free(void* p, hipStream_t st) {
  if (!p) return;
  std::lock_guard<std::mutex> lock(g_mu);
  auto it = g_out.find(p);
  if (it == g_out.end()) {   // allocated while the stream was being captured
    (void)hipFreeAsync(p, st);
    return;
  }
  Block b = it->second;
  g_out.erase(it);
  if (hipEventRecord(b.ev, st) != hipSuccess) {
    (void)hipGetLastError();
    (void)hipStreamSynchronize(st);
    (void)hipFreeAsync(b.p, st);
    (void)hipEventDestroy(b.ev);
    return;
  }
  b.used = g_uses;
  g_idle.push_back(b);
  size_t idle = 0;
  for (const Block& x : g_idle)
    if (x.dev == b.dev) idle += x.bytes;
  // oldest first (the list is in the order of return)
  for (size_t i = 0; i < g_idle.size();) {
    const Block& x = g_idle[i];
    if (x.dev == b.dev && (idle > kKeepBytes || g_uses - x.used > kKeepUses)) {
      idle -= x.bytes;
      give_back(x, st);
      g_idle.erase(g_idle.begin() + i);
    } else {
      ++i;
    }
  }
}

// the bytes given back; on a stream of its own (the default one may not be used while another
// thread captures)
static size_t work_trim() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return 0;
  std::lock_guard<std::mutex> lock(g_mu);
  const bool any = std::any_of(g_idle.begin(), g_idle.end(),
                               [&](const Block& b) { return b.dev == dev; });
  hipStream_t st = nullptr;
  if (!any || hipStreamCreateWithFlags(&st, hipStreamNonBlocking) != hipSuccess) return 0;
  size_t bytes = 0;
  for (size_t i = g_idle.size(); i-- > 0;)
    if (g_idle[i].dev == dev) {
      bytes += g_idle[i].bytes;
      give_back(g_idle[i], st);
      g_idle.erase(g_idle.begin() + i);
    }
  (void)hipStreamSynchronize(st);   // (the runtime gives its pool's memory back here)
  (void)hipStreamDestroy(st);
  return bytes;
}

hipError_t dev_alloc(void** p, size_t bytes) {
  hipError_t e = hipMalloc(p, bytes);
  if (e == hipSuccess) return e;
  if (work_trim()) e = hipMalloc(p, bytes);
  (void)hipGetLastError();   // (reported by the status alone)
  return e;
}

}  // namespace sfft

extern "C" size_t sfft_release_scratch(void) { return sfft::work_trim(); }
