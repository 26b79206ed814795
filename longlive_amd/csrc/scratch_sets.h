// The sets of device memory of one (device, stream) pair: which of them a launch gets.  Host arithmetic without a GPU call, so
// that the CPU tests run it too.
#pragma once
#include <stddef.h>
#include <stdint.h>

#include <vector>

namespace ll {

// Records for partial tiles and arrival counters.
struct StreamScratch {
  uint8_t* records = nullptr;
  size_t record_bytes = 0;
  int* counters = nullptr;  // zero whenever no launch is running
  size_t n_counters = 0;
};

// A recorded graph uses the addresses it was recorded with at every replay, on whatever stream that is, and so beside the
// ordinary launches of the stream it was recorded on: two launches that meet in one set count their arrivals in the same
// words and add up each other's parts.  A set therefore serves either ordinary launches, which the stream keeps apart, or
// recorded ones.  A recorded set is never freed for a larger one: graphs may still be replayed that use it.
struct ScratchSets {
  StreamScratch ordinary;
  StreamScratch recorded;
  std::vector<StreamScratch> retired;  // recorded ones that a later recording found too small

  static bool holds(const StreamScratch& w, size_t record_bytes, size_t counters) {
    return w.record_bytes >= record_bytes && w.n_counters >= counters;
  }
  // The set for a launch that is being recorded, which may not allocate: the one of earlier recordings, or else the one that an
  // ordinary launch or a reserve call left, which the recordings then keep.  Null if neither is large enough.
  const StreamScratch* for_recording(size_t record_bytes, size_t counters) {
    if (!holds(recorded, record_bytes, counters)) {
      if (!holds(ordinary, record_bytes, counters)) return nullptr;
      if (recorded.records) retired.push_back(recorded);
      recorded = ordinary;
      ordinary = StreamScratch{};
    }
    return &recorded;
  }
  // The set for an ordinary launch, which is stream_scratch's to allocate.  False: too small; `grown` has the sizes to allocate.
  bool for_launch(size_t record_bytes, size_t counters, StreamScratch& grown) const {
    grown = StreamScratch{};
    if (holds(ordinary, record_bytes, counters)) return true;
    grown.record_bytes = record_bytes > ordinary.record_bytes ? record_bytes : ordinary.record_bytes;
    grown.n_counters = counters > ordinary.n_counters ? counters : ordinary.n_counters;
    if (grown.n_counters < 4096) grown.n_counters = 4096;
    return false;
  }
  bool empty() const { return !ordinary.records && !recorded.records && retired.empty(); }
};

}  // namespace ll
