// dedup_launch.hpp -- host launchers of the dedup kernels (dedup.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "backprop_launch.hpp"

namespace nve_amd {

// The unique count and the key span of a dedup, side by side.
struct DedupHead {
  uint32_t total;           // unique keys
  uint32_t pad;
  unsigned long long span;  // OR over the keys of key ^ key[0] (sort keys): the bits where they differ
};

// Where a dedup's outputs go: unique keys, counts, inverse (optional) and offsets
// of the key type, pos_key (optional) the unique index of every dedup position, the head
// (and a copy in pinned host memory, optional); with pg.rows, each dedup
// position's gradient row and weight.
struct DedupOut {
  int key_bytes;
  void* unique;
  void* counts;
  void* inverse;
  void* offsets;
  uint32_t* pos_key;
  DedupHead* head;
  DedupHead* host_head;
  PositionGrad pg;
};

// Words of the key-span parts that the radix sort writes for n keys
// (radix_span_parts(n)).
int64_t dedup_span_parts(int64_t n);
// Whether a sort of the caller's keys (RadixSource) with gradient rows carries
// rows in place of positions.
bool carries_rows(int mode);
// k64[i] = key i as an unsigned sort key (sign bit flipped when flip != 0), v[i] = i.
hipError_t launch_dedup_prep(const void* keys, int key_bytes, int64_t n, int flip, uint64_t* k64,
                             uint32_t* v, hipStream_t stream);
// Every output from the sorted keys ks (values vs: positions, or with `carried`
// their gradient rows); head.span = the OR of the span parts (0 without
// span_part).  state: run_state_words(n) words, all 0.
int64_t run_state_words(int64_t n);
hipError_t launch_dedup_runs(const uint64_t* ks, const uint32_t* vs, int64_t n, const uint64_t* span_part,
                             uint64_t* state, bool carried, const DedupOut& out, hipStream_t stream);
// Sort and outputs of at most kSmallDedupKeys keys in one launch (head.span 0).
constexpr int64_t kSmallDedupKeys = 4096;
hipError_t launch_dedup_small(const void* keys, int64_t n, const DedupOut& out, hipStream_t stream);

// Hash slots for a batch of n keys: a power of two, at least 2n (and 1024).
size_t hash_dedup_slots(int64_t n);
// Bytes per hash-table key: 4 when every row index fits 32 bits, else 8.
size_t hash_dedup_key_bytes(int64_t num_rows);
// out row i = table row keys[i] for keys in [0, num_rows) (others untouched),
// deduplicated by hashing.  Scratch: tab (hash_dedup_slots(n) 8-byte slots:
// key and owner position when hash_dedup_key_bytes(num_rows) is 4, else the
// key), owner (one word per slot, 8-byte keys only) and slot_of (n words:
// each position's owner, or with 8-byte keys its slot).  Three launches,
// asynchronous.
hipError_t launch_hash_dedup_gather(const void* keys, int key_bytes, int64_t n, const uint8_t* table,
                                    int64_t num_rows, int64_t row_bytes, void* out, int64_t out_stride,
                                    void* tab, uint32_t* owner, uint32_t* slot_of, hipStream_t stream);

}  // namespace nve_amd
