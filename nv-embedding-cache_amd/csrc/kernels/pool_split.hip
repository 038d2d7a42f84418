// pool_split.hip -- the sliced find-and-pool kernels (pool_slices.cuh) over
// fp32 and fp16 rows, and the rule that chooses them.
#include "pool_slices.cuh"

namespace nve_amd {

// Groups of g lanes that share a bag.  A workgroup of the split kernel is at least
// a wave, and a wave does the work of 64 rows for a bag of 33 to 64 keys, whatever
// its length: it pays while the bags alone would not fill the chip.  From two waves
// per SIMD of whole bags (131,072 lanes) on, a group per bag is faster: bags of ~35
// weighted keys over 128-byte rows, 16,384 of them 13.2 and 8.4 us, over 256-byte rows,
// 8,192 bags 11.8 and 7.4; with half as many bags of ~64 keys unweighted 8.3 and 9.2.
// Byte rows of 129 to 512 bytes take twice the lanes in whole bags (4,096 bags of ~40
// weighted 264-byte rows 19.3 and 14.4 us).
// Groups of 32 lanes cut such a bag in two; with weights and up to 48 keys a group
// per bag is faster at any number of bags (512-byte rows, ~35 keys, 1,024 bags 7.1 and
// 5.0 us; 64 bags of ~63 keys 5.3 and 5.9).
// Over a cache many bags of up to 48 keys are left to the general kernel, which cuts
// them into less than a wave, where its loads are as wide: 32,000 bags of ~36 keys
// over 128-byte rows 32.2 us in whole waves and 27.2 there with weights, 27.5 and 26.6
// without; 16,384 bags of ~40 keys 19.0 and 16.8, 16.4 and 16.9.
static int slice_groups(const PoolLaunch& a, int g) {
  const int gpb = pool_groups_per_bag(a, g);
  if (a.force_split != 0 || gpb == 1 || gpb * g > 64) return gpb;
  const int64_t avg = a.keys_per_bag > 0 ? a.keys_per_bag : a.num_keys / a.num_bags;
  const int64_t simd_waves = 1024 * 64;  // lanes of a wave per SIMD
  const int64_t bytes = a.count * value_elem_bytes(a.stored_dtype);
  int whole = g;  // lanes of a bag that is not shared: byte rows are then cut finer
  while (value_elem_bytes(a.stored_dtype) == 1 && whole * 8 < bytes && whole < 64) whole *= 2;
  const int64_t lanes = a.num_bags * whole;
  if (a.src.cache_data != nullptr) {
    const bool wide = ((uint64_t)a.src.table | (uint64_t)a.src.cache_data | a.src.row_bytes | (uint64_t)bytes |
                       (uint64_t)a.out | (uint64_t)a.out_stride) % 16 == 0;
    const bool many = avg <= 48 && lanes >= (a.weighted && bytes > 64 ? 2 : 3) * simd_waves;
    return many && wide ? gpb : 64 / g;
  }
  return (avg <= 64 && lanes >= 2 * simd_waves) || (avg <= 48 && g == 32 && a.weighted) ? 1 : 64 / g;
}

// The slices of a launch's rows, or false where the general kernel serves it:
// quantized rows over several tables or a cache, short bags over a cache
// (12.8 us for 8,192 bags of 32 keys, all hits, as a short kernel that probed without
// a round ahead took; one that probes ahead has not been measured),
// tables without a row count or with more rows than a 32-bit index holds, rows
// under 32 bytes (a lane group of 8 would be mostly idle) or wider than the
// zero row, and bags cut into chunks by fewer lanes than a wave.
bool pool_slices(const PoolLaunch& a, PoolSlices* g) {
  const int es = value_elem_bytes(a.stored_dtype);
  const bool cache = a.src.cache_data != nullptr;
  if (!a.src.load_indices) return false;
  if (a.stored_dtype != kF16 && a.stored_dtype != kF32 && !is_rowwise(a.stored_dtype)) return false;
  if (is_rowwise(a.stored_dtype) && (cache || a.num_tables > 0)) return false;
  if (a.out_dtype != kF16 && a.out_dtype != kF32) return false;
  if (a.src.row_bytes == 0 || a.src.row_bytes > 0xffffffffull) return false;  // 32-bit row stride
  if (a.count <= 0 || a.count > 0x7fffffff / es) return false;
  // whole elements: the rows' and the output's
  const uint64_t oes = a.out_dtype == kF16 ? 2 : 4;
  const auto whole = [](uint64_t p, uint64_t n) { return p % n == 0; };
  if (!whole(a.src.row_bytes, (uint64_t)es) || !whole((uint64_t)a.out, oes) || !whole((uint64_t)a.out_stride, oes))
    return false;
  if (a.num_tables > 0) {
    if (!whole((uint64_t)a.out_table_stride, oes)) return false;
    for (int t = 0; t < a.num_tables; ++t)
      if (a.tables[t] == nullptr || a.table_rows[t] == 0 || a.table_rows[t] >= kMaxIndexRows ||
          !whole((uint64_t)a.tables[t], (uint64_t)es))
        return false;
  } else if (cache) {
    // 32-bit row codes: cache slots and backing rows below 2^31
    if (a.src.num_sets == 0 || a.src.num_sets * 8 >= 0x80000000ull) return false;
    if (a.src.table != nullptr && (a.src.num_rows == 0 || a.src.num_rows >= 0x80000000ull)) return false;
    if (a.key_bytes == 4 && a.src.num_sets > 0xffffffffull) return false;
    if (!whole((uint64_t)a.src.table, (uint64_t)es) || !whole((uint64_t)a.src.cache_data, (uint64_t)es)) return false;
  } else if (a.src.table == nullptr || a.src.num_rows == 0 || a.src.num_rows >= kMaxIndexRows ||
             !whole((uint64_t)a.src.table, (uint64_t)es)) {
    return false;
  }
  const int64_t area = a.count * es;
  if (area < 32 || area > kZeroRowBytes) return false;
  const auto cut = [&](int vb) {
    const int64_t slices = (area + vb - 1) / vb;
    g->vb = vb;
    g->g = 8;
    while (g->g < slices && g->g < 64) g->g *= 2;
    g->columns = (int)((slices + g->g - 1) / g->g);
    g->gpb = slice_groups(a, g->g);
  };
  cut(area > 64 ? 16 : area > 32 ? 8 : 4);
  // Bytes widen to 16 values a lane in a 16-byte slice: 8-byte slices halve the
  // lane's work and double the waves, as long as they fit one column.  Long
  // bags have their waves from the split and keep 16-byte slices past 128 bytes
  // (int8 rows of 512 values, 64 bags of 500: 11.4 us, 13.1 with 8-byte slices;
  // 16,384 bags of 30: 54.0 and 49.1 us).
  if (es == 1 && area > 64 && area <= 512 && (g->gpb == 1 || area <= 128)) {
    const bool whole = g->gpb == 1;
    cut(8);
    if (whole) g->gpb = 1;
  }
  if (g->columns > 65535) return false;
  if (g->gpb == 1) {
    // several tables: table t holds bags t * bags_per_table ...
    if (a.num_tables > 0 && a.num_bags != a.num_tables * a.bags_per_table) return false;
    return !cache && a.num_bags <= 0x7fffffffLL * (256 / g->g);
  }
  return a.num_tables == 0 && g->gpb * g->g >= 64 && a.num_bags <= 0x7fffffffLL;
}

hipError_t launch_pool_slices(const PoolLaunch& a, const PoolSlices& g, hipStream_t stream) {
  switch (a.stored_dtype) {
    case kF16: return launch_slices_sdt<kF16>(a, g, stream);
    case kF32: return launch_slices_sdt<kF32>(a, g, stream);
    case kXI8AF32:
    case kXE4M3F32: return launch_pool_slices_ext(a, g, stream);
    default: return launch_pool_slices_quant(a, g, stream);
  }
}

}  // namespace nve_amd
