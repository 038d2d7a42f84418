// pool_split.hip -- the sliced find-and-pool kernels (pool_slices.cuh) over
// fp32 and fp16 rows, and the rule that chooses them.
#include "pool_slices.cuh"

namespace nve_amd {

// The slices of a launch's rows, or false where the general kernel serves it:
// quantized rows over several tables or a cache, short bags over a cache
// (measured as fast there: 12.8 us for 8,192 bags of 32 keys, all hits),
// tables without a row count or with more rows than a 32-bit index holds, rows
// under 32 bytes (a lane group of 8 would be mostly idle) or wider than the
// zero row, and bags cut into
// chunks by fewer lanes than a wave.
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
    g->gpb = pool_groups_per_bag(a, g->g);
    if (a.force_split == 0 && g->gpb > 1 && g->gpb * g->g < 64) g->gpb = 64 / g->g;  // whole waves
  };
  cut(area > 64 ? 16 : area > 32 ? 8 : 4);
  // Bytes widen to 16 values a lane in a 16-byte slice: 8-byte slices halve the
  // lane's work and double the waves, as long as they fit one column.  Long
  // bags have their waves from the split and keep 16-byte slices past 128 bytes
  // (int8 rows of 512 values, 64 bags of 500: 11.4 us, 13.1 with 8-byte slices;
  // 16,384 bags of 30: 54.0 and 49.1 us).
  if (es == 1 && area > 64 && area <= 512 && (g->gpb == 1 || area <= 128)) cut(8);
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
