// sort_launch.hpp -- stable radix sort, exclusive scan and key-span helpers.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <utility>

#include "backprop_launch.hpp"

namespace nve_amd {

// Bytes of temporary storage radix_sort_pairs needs for n pairs; it also
// covers exclusive_scan_u32 of up to n elements.
size_t radix_sort_temp_bytes(int64_t n);
// Bytes of temporary storage exclusive_scan_u32 needs for m elements.
size_t scan_temp_bytes(int64_t m);

// The caller's keys as the first pass's input: keys of key_bytes bytes at
// `keys` (sign bit flipped when flip != 0), values = positions; span_part
// (optional, radix_span_parts(n) words) receives ORs of key ^ key[0] whose OR is
// that of all keys.
struct RadixSource {
  const void* keys;
  int key_bytes;
  int flip;
  uint64_t* span_part;
};
int64_t radix_span_parts(int64_t n);

// Stable ascending sort of (keys[i], vals[i]) on bits [begin_bit, end_bit) of
// the keys (digits of 8 or 9 bits from begin_bit).  Ping-pongs between (keys, vals) and
// (keys_alt, vals_alt); *result_in_alt says which pair holds the result.
// With src, the first pass reads src instead of keys / vals (which it never
// reads); at least one pass must then run (n >= 2, end_bit > begin_bit), else
// hipErrorInvalidValue.  clear (optional): clear_words words set to 0 on the
// way, when a pass runs.  pg (optional, a pooled mode): pg->by_key is filled on
// the way too, and with src and weight_from_row(pg->mode) the values are the
// positions' gradient rows (also Concatenate: the positions).
hipError_t radix_sort_pairs(uint64_t* keys, uint32_t* vals, uint64_t* keys_alt, uint32_t* vals_alt,
                            int64_t n, int begin_bit, int end_bit, void* temp, int* result_in_alt,
                            hipStream_t stream, const RadixSource* src = nullptr, uint64_t* clear = nullptr,
                            int64_t clear_words = 0, const PositionGrad* pg = nullptr);

// In-place exclusive scan of m uint32 (total, if non-null, gets the sum);
// temp holds scan_temp_bytes(m) bytes.
hipError_t exclusive_scan_u32(uint32_t* data, int64_t m, uint32_t* total, void* temp,
                              hipStream_t stream);

// *out |= OR over i of (keys[i] ^ keys[0]); *out must start at 0.
hipError_t key_span(const uint64_t* keys, int64_t n, unsigned long long* out, hipStream_t stream);

}  // namespace nve_amd
