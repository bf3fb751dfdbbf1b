// Device scratch buffers owned by the library, one per (device, stream, purpose).  Work on one stream is ordered, so
// consecutive calls can share a buffer; calls on different streams never do.
//
// A buffer only grows, and growing never frees: a HIP graph captured on the stream holds the old buffer's address, and
// replaying that graph must keep working.  The old buffer is therefore retired, not freed; retired buffers stay
// allocated (and valid for such graphs) until release_stream_workspaces() is called for the stream -- by the owner of
// a private stream (an operator handle, a module) right before it destroys the stream, after destroying its graphs.
// Buffers of caller-owned streams live until the process ends.  Growing allocates, which cannot happen while the
// stream is being captured into a graph: run a shape once eagerly before capturing it.
#include <map>
#include <mutex>
#include <set>
#include <tuple>
#include <vector>

#include "internal.h"

namespace mi {

namespace {
struct Buf {
  void *ptr = nullptr;
  size_t bytes = 0;
  std::vector<void *> retired;  // smaller predecessors that a captured graph may still name
};
std::mutex g_mutex;
std::map<std::tuple<int, hipStream_t, int>, Buf> g_bufs;
long g_allocations = 0;  // hipMalloc calls made here since the library was loaded (read by the tests)
}  // namespace

int stream_workspace(hipStream_t st, int purpose, size_t bytes, void **out, bool zero_fresh) {
  int dev = 0;
  MI_HIP(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lock(g_mutex);
  Buf &b = g_bufs[std::make_tuple(dev, st, purpose)];
  if (b.bytes < bytes) {
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    (void)hipStreamIsCapturing(st, &cs);
    MI_REQUIRE(cs == hipStreamCaptureStatusNone, MI_HIP_ERROR,
               "a scratch buffer has to grow while its stream is being captured: run the same shape once eagerly "
               "before capturing it");
    const size_t want = (bytes + 255) & ~(size_t)255;
    void *fresh = nullptr;
    MI_HIP(hipMalloc(&fresh, want));
    ++g_allocations;
    if (zero_fresh) {  // on the stream, ahead of the first kernel to use it (the stream is not being captured)
      const hipError_t e = hipMemsetAsync(fresh, 0, want, st);
      if (e != hipSuccess) {
        (void)hipFree(fresh);
        MI_HIP(e);
      }
    }
    if (b.ptr)
      b.retired.push_back(b.ptr);
    b.ptr = fresh;
    b.bytes = want;
  }
  *out = b.ptr;
  return MI_SUCCESS;
}

namespace {
std::mutex g_scratch_use[WS_COUNT];  // taken before g_mutex, never after it
std::set<hipStream_t> g_replay_in_order;
}  // namespace

void stream_replays_in_order(hipStream_t st) {
  std::lock_guard<std::mutex> lock(g_mutex);
  g_replay_in_order.insert(st);
}

int ScratchBytes::get(hipStream_t st, int purpose, size_t bytes) {
  stream = st;
  size_t want = 1 << 16;
  while (want < bytes)
    want *= 2;
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  const bool capturing = hipStreamIsCapturing(st, &cs) == hipSuccess && cs != hipStreamCaptureStatusNone;
  bool kept = st != hipStreamPerThread && want <= ((size_t)64 << 20);
  if (kept && capturing) {
    int dev = 0;
    MI_HIP(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lock(g_mutex);
    const auto it = g_bufs.find(std::make_tuple(dev, st, purpose));
    kept = g_replay_in_order.count(st) && it != g_bufs.end() && it->second.bytes >= want;
  }
  if (kept) {
    use = std::unique_lock<std::mutex>(g_scratch_use[purpose]);
    return stream_workspace(st, purpose, want, &ptr);
  }
  MI_HIP(hipMallocAsync(&ptr, bytes, st));
  own = true;
  return MI_SUCCESS;
}

int ScratchBytes::release() {
  if (use.owns_lock())
    use.unlock();
  if (own) {
    own = false;
    MI_HIP(hipFreeAsync(ptr, stream));
  }
  return MI_SUCCESS;
}

long workspace_allocations() {
  std::lock_guard<std::mutex> lock(g_mutex);
  return g_allocations;
}

void release_stream_workspaces(hipStream_t st) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess)
    return;
  std::lock_guard<std::mutex> lock(g_mutex);
  g_replay_in_order.erase(st);
  for (auto it = g_bufs.begin(); it != g_bufs.end();) {
    if (std::get<0>(it->first) == dev && std::get<1>(it->first) == st) {
      (void)hipStreamSynchronize(st);
      for (void *p : it->second.retired)
        (void)hipFree(p);
      if (it->second.ptr)
        (void)hipFree(it->second.ptr);
      it = g_bufs.erase(it);
    } else {
      ++it;
    }
  }
}

}  // namespace mi
