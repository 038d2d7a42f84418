// The training backprop's host code (csrc/backprop.cpp, csrc/dedup.cpp) over a
// pretended device, on the CPU: a dedup's head is written to pinned memory only
// when its stream is waited for, and a launch behind the dedup can be made to
// fail.  However the backprop ends, no such write may be left: it would land in
// the head of the thread's next dedup.
#include <cstdio>
#include <cstring>
#include <vector>

#include "backprop.hpp"
#include "dedup.hpp"
#include "kernels/backprop_launch.hpp"
#include "kernels/cache_launch.hpp"
#include "kernels/dedup_launch.hpp"
#include "kernels/launch.hpp"
#include "kernels/sort_launch.hpp"
#include "layers.hpp"
#include "runtime.hpp"

struct Write {
  hipStream_t stream;
  nve_amd::DedupHead* to;
  nve_amd::DedupHead value;
};
static std::vector<Write> pending;
static int fail_at;  // 1: the small dedup, 2: the pieces, 3: the crossing keys
alignas(64) static unsigned char slots[nve_amd::kPinnedSlots][nve_amd::kPinnedSlotBytes];

extern "C" {
hipError_t hipStreamSynchronize(hipStream_t s) {
  std::vector<Write> left;
  for (const Write& w : pending) {
    if (w.stream == s) *w.to = w.value;
    else left.push_back(w);
  }
  pending.swap(left);
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorName(hipError_t) { return "error"; }
const char* hipGetErrorString(hipError_t) { return "a launch that was made to fail"; }
}

namespace nve_amd {
void* pinned_slot(PinnedSlot use) { return slots[use]; }
void read_small(void* host, const void*, size_t bytes, hipStream_t s) {
  std::memset(pinned_slot(kReadSlot), 0xff, bytes);
  (void)hipStreamSynchronize(s);
  std::memset(host, 0, bytes);
}
bool carries_rows(int) { return false; }
hipError_t launch_gather(const GatherLaunch&, hipStream_t) { return hipSuccess; }
hipError_t launch_fill_u64(uint64_t*, int64_t, uint64_t, hipStream_t) { return hipSuccess; }
int64_t run_state_words(int64_t n) { return n + 3; }
int64_t dedup_span_parts(int64_t) { return 1; }
size_t hash_dedup_slots(int64_t) { return 1024; }
size_t radix_sort_temp_bytes(int64_t) { return 1024; }
hipError_t radix_sort_pairs(uint64_t*, uint32_t*, uint64_t*, uint32_t*, int64_t, int, int, void*, int*, hipStream_t,
                            const RadixSource*, uint64_t*, int64_t, const PositionGrad*) {
  return hipSuccess;
}
hipError_t launch_dedup_prep(const void*, int, int64_t, int, uint64_t*, uint32_t*, hipStream_t) { return hipSuccess; }
static hipError_t queue_head(int64_t n, const DedupOut& o, hipStream_t s) {
  pending.push_back({s, o.host_head, DedupHead{(uint32_t)n, 0, 0}});
  return fail_at == 1 ? hipErrorInvalidValue : hipSuccess;
}
hipError_t launch_dedup_runs(const uint64_t*, const uint32_t*, int64_t n, const uint64_t*, uint64_t*, bool,
                             const DedupOut& o, hipStream_t s) {
  return queue_head(n, o, s);
}
hipError_t launch_dedup_small(const void*, int64_t n, const DedupOut& o, hipStream_t s) { return queue_head(n, o, s); }
hipError_t launch_hash_dedup_gather(const void*, int, int64_t, const uint8_t*, int64_t, int64_t, void*, int64_t, void*,
                                    uint32_t*, uint32_t*, hipStream_t) {
  return hipSuccess;
}
hipError_t key_span(const uint64_t*, int64_t, unsigned long long*, hipStream_t) { return hipSuccess; }
hipError_t launch_bag_denom(const void*, int, int64_t, int64_t, const void*, int, int, float*, hipStream_t) {
  return hipSuccess;
}
hipError_t launch_piece_pool(const PieceArgs&, int, int, hipStream_t s) {
  // another read of this thread meanwhile, as a callback could make it
  unsigned char word[8];
  read_small(word, nullptr, 8, reinterpret_cast<hipStream_t>((char*)s + 1));
  return fail_at == 2 ? hipErrorInvalidValue : hipSuccess;
}
hipError_t launch_piece_combine(const PieceArgs&, int, hipStream_t) {
  return fail_at == 3 ? hipErrorInvalidValue : hipSuccess;
}
}  // namespace nve_amd

int main() {
  using namespace nve_amd;
  int bad = 0;
  for (int64_t n : {int64_t(10), int64_t(5000)}) {
    std::vector<unsigned char> ws(backprop_workspace_bytes(n, 0, 4));
    std::vector<int64_t> keys(n), unique(n);
    std::vector<float> in(n * 4), out(n * 4);
    int turn = 0;
    for (fail_at = 0; fail_at <= 3; ++fail_at) {
      const hipStream_t s = reinterpret_cast<hipStream_t>(slots[0] + 64 * ++turn);  // a stream of its own each time
      bool threw = false;
      int64_t got = -1;
      try {
        got = pooling_backprop_run(8, n, keys.data(), NVE_POOL_CONCATENATE, 0, nullptr, 0, 0, nullptr, 0, in.data(),
                                   kF32, 4, unique.data(), out.data(), ws.data(), ws.size(), s, false);
      } catch (const Error&) {
        threw = true;
      }
      if (threw != (fail_at != 0) || (!threw && got != n)) bad = 1, std::printf("n %ld fail %d: wrong end\n", (long)n, fail_at);
      if (!pending.empty()) bad = 1, std::printf("n %ld fail %d: a write to the head is left\n", (long)n, fail_at);
      pending.clear();
    }
  }
  if (!bad) std::printf("pending head ok\n");
  return bad;
}
