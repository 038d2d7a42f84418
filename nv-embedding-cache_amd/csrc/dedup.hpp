// dedup.hpp -- key dedup and dedup-ordered gather (device buffers, caller workspace).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <cstddef>

#include "kernels/dedup_launch.hpp"

namespace nve_amd {

size_t dedup_workspace_bytes(int64_t n);

// The sort first assumes that the keys differ only below this bit (rows of
// tables up to 2^27: three 9-bit passes) and learns whether they did from the
// span computed on the way, so no host round trip sits between the key
// preparation and the sort; a batch whose keys differ higher up is sorted
// again on its exact bits.
constexpr int kSpecSortBits = 27;
inline bool dedup_spec_failed(const DedupHead& h) { return (h.span >> kSpecSortBits) != 0; }

// Sorted unique keys, counts, stable inverse map and exclusive offsets (all of
// the key type); returns the number of unique keys (synchronizes the stream).
// pos_key (optional, n entries): the unique index of each position of the
// dedup order.  later: instead of waiting for the head (a stream
// synchronization), return -1; the caller holds a PendingHead, reads it once it
// has queued what follows (from the same thread, before another dedup) and, if
// dedup_spec_failed, runs again with exact = true.  exact: read the key span
// back first and sort on exactly its bits (never needs a second run).
// pg (optional): also each dedup position's gradient row and weight (the
// backprop's per-position step, done on the way).
int64_t dedup_run(int key_bytes, int64_t n, const void* keys, void* unique, void* counts,
                  void* inverse, void* offsets, void* ws, size_t ws_bytes, hipStream_t s,
                  uint32_t* pos_key = nullptr, bool later = false, bool exact = false,
                  const PositionGrad* pg = nullptr);
// The head of this thread's last dedup_run on stream s (synchronizes it).
DedupHead dedup_head(hipStream_t s);

// The head of a dedup_run with `later` on stream s, which kernels still to run
// write to this thread's pinned memory.  Left unread (a launch behind the dedup
// failed), it waits for the stream, so that no write to it is pending when the
// thread's next dedup, on whatever stream, has its head there.
class PendingHead {
 public:
  explicit PendingHead(hipStream_t s) : stream_(s) {}
  PendingHead(const PendingHead&) = delete;
  PendingHead& operator=(const PendingHead&) = delete;
  ~PendingHead() {
    if (!read_) (void)hipStreamSynchronize(stream_);
  }
  DedupHead read() {
    const DedupHead h = dedup_head(stream_);
    read_ = true;
    return h;
  }

 private:
  hipStream_t stream_;
  bool read_ = false;
};

// out[i] = table row keys[i] for keys in [0, num_rows), each distinct row read
// from the table once (asynchronous).
void dedup_gather_run(int key_bytes, int64_t n, const void* keys, const uint8_t* table,
                      int64_t num_rows, int64_t row_bytes, void* out, int64_t out_stride, void* ws,
                      size_t ws_bytes, hipStream_t s);

}  // namespace nve_amd
