// Device memory of the library's own: the records through which workgroups of one launch hand partial tiles to each
// other (the split division of the attention kernel, the K-split shares of the persistent GEMM, the K ranges of small
// products) and the arrival counters that go with them.  One set per (device, stream): launches on one stream run one after
// the other and can share it, launches on different streams get different sets, and so do the launches that were recorded on a
// stream (scratch_sets.h).  A set is created at the first launch that needs one, grown when a later launch needs more, and kept
// until ll_release_stream_memory or the end of the process.  The counters are zero whenever no launch is running: every kernel
// that uses them leaves them at zero.
#include <map>
#include <mutex>

#include "ll_common.h"
#include "gemm_split.h"

namespace ll {

static std::mutex g_scratch_mutex;
static std::map<std::pair<int, hipStream_t>, ScratchSets> g_scratch;

// The memory of small products (gemm_w4a4_small_kernel) is a set of its own: launches of the other kernels that are
// recorded keep using the set above at every replay, on whatever stream that is, and an ordinary linear layer beside
// them must not meet them there.  No recorded launch uses this one.  One size holds every small product, so it never grows.
static std::map<std::pair<int, hipStream_t>, StreamScratch> g_small_scratch;

// Memory is set up and freed as if no stream were being captured: while one is, in the global mode, either call is refused and
// spoils the recording, on whatever stream it is made.
struct RelaxedCapture {
  hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
  const bool exchanged = hipThreadExchangeStreamCaptureMode(&mode) == hipSuccess;
  ~RelaxedCapture() {
    if (exchanged) (void)hipThreadExchangeStreamCaptureMode(&mode);
  }
};

static void free_scratch(StreamScratch& w) {
  const RelaxedCapture relaxed;
  if (w.records) (void)hipFree(w.records);  // waits for the launches that still use it
  if (w.counters) (void)hipFree(w.counters);
  w = StreamScratch{};
}

// Records and counters of the sizes in w, the counters zero for the work that follows on `stream`.
static hipError_t allocate_scratch(StreamScratch& w, hipStream_t stream) {
  const RelaxedCapture relaxed;
  hipError_t e = hipMalloc(reinterpret_cast<void**>(&w.records), w.record_bytes);
  if (e == hipSuccess) e = hipMalloc(reinterpret_cast<void**>(&w.counters), w.n_counters * sizeof(int));
  if (e == hipSuccess) e = hipMemsetAsync(w.counters, 0, w.n_counters * sizeof(int), stream);
  if (e != hipSuccess) free_scratch(w);
  return e;
}

int stream_scratch(int dev, hipStream_t stream, size_t record_bytes, size_t counters, bool may_allocate, StreamScratch& out,
                   bool* missing, const char* what) {
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (missing) *missing = false;
  if (!may_allocate) {  // the stream is being captured
    const auto it = g_scratch.find({dev, stream});
    const StreamScratch* w = it == g_scratch.end() ? nullptr : it->second.for_recording(record_bytes, counters);
    if (w) out = *w;
    else if (missing) *missing = true;
    return LL_OK;
  }
  ScratchSets& sets = g_scratch[{dev, stream}];
  StreamScratch grown;
  if (!sets.for_launch(record_bytes, counters, grown)) {
    free_scratch(sets.ordinary);
    const size_t want_bytes = grown.record_bytes;
    if (const hipError_t e = allocate_scratch(grown, stream); e != hipSuccess) {
      set_error("%s: cannot set up %zu bytes for partial results: %s", what, want_bytes, hipGetErrorString(e));
      if (sets.empty()) g_scratch.erase({dev, stream});
      return LL_ELAUNCH;
    }
    sets.ordinary = grown;
  }
  out = sets.ordinary;
  return LL_OK;
}

bool small_product_scratch(int dev, hipStream_t stream, int cus, StreamScratch& out) {
  if (stream_is_capturing(stream)) return false;
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  StreamScratch& w = g_small_scratch[{dev, stream}];
  if (!w.records) {
    w.record_bytes = (size_t)small_product_units(cus) * kSmallRecordBytes;
    w.n_counters = (size_t)small_product_units(cus);
    const hipError_t e = allocate_scratch(w, stream);
    if (e != hipSuccess) {
      (void)hipGetLastError();  // the caller has a way without the memory
      g_small_scratch.erase({dev, stream});
      return false;
    }
  }
  out = w;
  return true;
}

int release_stream_scratch(int dev, hipStream_t stream) {
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (const auto small = g_small_scratch.find({dev, stream}); small != g_small_scratch.end()) {
    free_scratch(small->second);
    g_small_scratch.erase(small);
  }
  const auto it = g_scratch.find({dev, stream});
  if (it == g_scratch.end()) return LL_OK;
  free_scratch(it->second.ordinary);
  free_scratch(it->second.recorded);
  for (StreamScratch& old : it->second.retired) free_scratch(old);
  g_scratch.erase(it);
  return LL_OK;
}

bool stream_is_capturing(hipStream_t stream) {
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream, &status) != hipSuccess) {
    (void)hipGetLastError();
    return true;
  }
  return status != hipStreamCaptureStatusNone;
}

int compute_units_of(int dev, int& cus, const char* what) {
  static std::atomic<int> cached[64];
  if (dev >= 0 && dev < 64 && (cus = cached[dev].load(std::memory_order_relaxed)) > 0) return LL_OK;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) {
    set_error("%s: cannot read the number of compute units of device %d", what, dev);
    return LL_ELAUNCH;
  }
  if (dev >= 0 && dev < 64) cached[dev].store(cus, std::memory_order_relaxed);
  return LL_OK;
}

}  // namespace ll

extern "C" int ll_release_stream_memory(void* stream) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) {
    ll::set_error("ll_release_stream_memory: hipGetDevice failed");
    return LL_ELAUNCH;
  }
  return ll::release_stream_scratch(dev, static_cast<hipStream_t>(stream));
}
