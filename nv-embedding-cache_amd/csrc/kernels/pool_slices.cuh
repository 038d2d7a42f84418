// pool_slices.cuh -- find-and-pool over linear tables (and, for long bags, over
// a set-associative cache) without the general pool_kernel's generality
// (64-bit address shuffles, hit masks, a 1 KB argument block):
//  * pool_split_kernel: long bags (the GPULayer benchmark: a few hundred bags
//    of ~1K keys), one workgroup per bag;
//  * pool_short_kernel: short bags (DLRM-style jagged batches, one or many
//    tables), one lane group per bag.
//
// Reference behaviour restated: find_and_combine (cuda_ops/find_and_combine_kernel.cuh:40-154)
// over a linear table (GPULayer, gpu_embedding_layer.cu:153-189).
//
// A row's value area is cut into slices of VB bytes, one per lane of a G-lane
// group (G = 8..64).  VB is 16 for fp16 / fp32 rows past 64 bytes, for byte rows of
// 65 to 512 bytes 8 where a group has the bag to itself (a byte widens to a value,
// so that a 16-byte slice is 16 of them), 8 or 4 for narrower rows; also for
// rows at any alignment (odd widths, quantized rows with their scale behind
// the values): gfx950 loads 16 bytes from any address, and the last slice of a
// width that is no multiple of VB starts VB bytes before the end, so it
// overlaps its neighbour (both lanes add the same values and store the same
// bits) and no lane reads outside the row.  Rows wider than 64 slices take one
// workgroup column (blockIdx.y) per 64 slices.
//
// Bound: the lines moved into the CUs, in small launches the latency of few waves.
// The plain read kernel (launch_read_ceiling) takes random 256-byte rows at 16.7
// TB/s from a table in L2 (4 MB), at 9.3 to 7.3 from the MALL (16 to 200 MB) and at 5.9
// from HBM (4 GB); batches of Zipf keys lie between the first two: 200-byte rows (2.6
// lines of 128 bytes) at 12 TB/s by lines, 26 tables as below at 12, 132-byte int8 rows
// (2.0 lines) at 8.5 (what holds those back has not been taken apart).  Measured against loads as narrow as the row's own alignment
// (pool_kernel): 16,384 bags of ~30 weighted 200-byte fp16 rows 20.9 -> 13.5 us
// (8-byte loads, 25 of 32 lanes before), the same bags of 132-byte int8 rows
// 23.6 -> 14.8 us (4-byte loads and a scale load per lane and row before),
// 26 tables of 8,192 bags of ~20 256-byte rows 112 -> 101 us.
//
// Same decomposition and summation order as pool_kernel's paths, so where both cut
// a row into the same lane groups and a bag into the same chunks (fp16 / fp32 rows
// of whole 16-byte slices) the two produce the same bits: a long bag cut into gpb
// contiguous key chunks, one chunk per G-lane group, each group accumulating
// its chunk in key order; an xor butterfly inside each wave; the waves'
// partial rows added in wave order through LDS.  A bag that one group adds has
// the bits of its key order in either.  What is leaner:
//  * the lane that resolves a key forms its row's address; both halves travel by
//    one DPP row_newbcast each, inside the 16 lanes of a row, which is why the rows
//    of a wider group resolve the same 16 keys (over a cache, where a probe is
//    dear, each its own: spread_keys);
//  * a quantized row's scale and offset are loaded once per key, by the lane
//    that resolves the key, and travel the same way;
//  * the butterfly uses DPP row_ror and v_permlane16_swap / v_permlane32_swap
//    (gfx950): a + (a of lane l ^ m), formed as the sum of the two swapped
//    halves, which is the same float addition;
//  * G, VB and the weighting fixed at compile time;
//  * the cross-wave sum is unrolled so its LDS reads are all in flight.
#pragma once

#include <type_traits>

#include "device_common.cuh"
#include "lane_moves.cuh"
#include "pool_launch.hpp"

namespace nve_amd {

namespace {

constexpr uint64_t kMaxIndexRows = 0xffffffffull;  // rows a 32-bit index addresses

// VB bytes from any address (one global_load of VB bytes).
typedef uint32_t u32x4_any __attribute__((ext_vector_type(4), aligned(1)));
typedef uint32_t u32x2_any __attribute__((ext_vector_type(2), aligned(1)));
typedef uint32_t u32_any __attribute__((aligned(1)));

template <int VB>
__device__ __forceinline__ Vec<VB> load_slice(uint64_t addr) {
  Vec<VB> v;
  if constexpr (VB == 16) {
    const u32x4_any x = gload<u32x4_any>(addr);
    v.w[0] = x.x;
    v.w[1] = x.y;
    v.w[2] = x.z;
    v.w[3] = x.w;
  } else if constexpr (VB == 8) {
    const u32x2_any x = gload<u32x2_any>(addr);
    v.w[0] = x.x;
    v.w[1] = x.y;
  } else {
    static_assert(VB == 4, "slices of 4, 8 or 16 bytes");
    v.w[0] = gload<u32_any>(addr);
  }
  return v;
}

// The scale (and offset) of a row whose values end at p, at any alignment.
template <int SDT>
__device__ __forceinline__ Meta load_meta_any(uint64_t p) {
  Meta m{1.0f, 0.0f};
  if constexpr (SDT == kQU8F32 || SDT == kXI8AF32) {
    const u32x2_any x = gload<u32x2_any>(p);
    m.s = __uint_as_float(x.x);
    m.o = __uint_as_float(x.y);
  } else if constexpr (SDT == kQI8F32 || SDT == kXE4M3F32) {
    m.s = __uint_as_float(gload<u32_any>(p));
  } else if constexpr (SDT == kQU8F16) {
    const uint32_t x = gload<u32_any>(p);
    m.s = h2f((uint16_t)(x & 0xffffu));
    m.o = h2f((uint16_t)(x >> 16));
  } else if constexpr (SDT == kQI8F16) {
    m.s = h2f(gload<uint16_t>(p));  // quantized rows have an even width
  }
  return m;
}

// E values (as f32 or RNE f16) at p, aligned to one output element.  One store
// per lane streams past L2 (as store_out); several go through it.
template <int E>
__device__ __forceinline__ void store_slice(uint64_t p, const float* v, bool out_f16) {
  if (out_f16) {
    if constexpr (E == 1) {
      *reinterpret_cast<gptr_w<uint16_t>>(p) = f2h(v[0]);
    } else {
      uint32_t w[E / 2];
#pragma unroll
      for (int i = 0; i < E / 2; ++i) w[i] = (uint32_t)f2h(v[2 * i]) | ((uint32_t)f2h(v[2 * i + 1]) << 16);
      if constexpr (E == 2) {
        *reinterpret_cast<gptr_w<u32_any>>(p) = w[0];
      } else if constexpr (E == 4) {
        __builtin_nontemporal_store(u32x2_any{w[0], w[1]}, reinterpret_cast<gptr_w<u32x2_any>>(p));
      } else if constexpr (E == 8) {
        __builtin_nontemporal_store(u32x4_any{w[0], w[1], w[2], w[3]}, reinterpret_cast<gptr_w<u32x4_any>>(p));
      } else {
#pragma unroll
        for (int i = 0; i < E / 8; ++i)
          reinterpret_cast<gptr_w<u32x4_any>>(p)[i] =
              u32x4_any{w[4 * i], w[4 * i + 1], w[4 * i + 2], w[4 * i + 3]};
      }
    }
  } else if constexpr (E == 1) {
    *reinterpret_cast<gptr_w<float>>(p) = v[0];
  } else if constexpr (E == 2) {
    __builtin_nontemporal_store(u32x2_any{__float_as_uint(v[0]), __float_as_uint(v[1])},
                                reinterpret_cast<gptr_w<u32x2_any>>(p));
  } else {
#pragma unroll
    for (int i = 0; i < E / 4; ++i) {
      const u32x4_any x{__float_as_uint(v[4 * i]), __float_as_uint(v[4 * i + 1]), __float_as_uint(v[4 * i + 2]),
                        __float_as_uint(v[4 * i + 3])};
      if constexpr (E == 4)
        __builtin_nontemporal_store(x, reinterpret_cast<gptr_w<u32x4_any>>(p));
      else
        reinterpret_cast<gptr_w<u32x4_any>>(p)[i] = x;
    }
  }
}

// a + (a of lane l ^ M), the same float addition as a + __shfl_xor(a, M)
// (addition commutes exactly, so both partners get the same bits).
template <int M>
__device__ __forceinline__ float xor_add(float a) {
  if constexpr (M == 32) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(a), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
  } else if constexpr (M == 16) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(a), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
  } else {
    static_assert(M == 8, "lane groups of 8 to 64 lanes");
    return a + __uint_as_float(dpp_mov<kDppRowRor8>(__float_as_uint(a)));
  }
}

template <int G, int M = G>
__device__ __forceinline__ void butterfly(float* acc, int e, float& wsum, bool weighted) {
  if constexpr (M < 64) {
    for (int c = 0; c < e; ++c) acc[c] = xor_add<M>(acc[c]);
    if (weighted) wsum = xor_add<M>(wsum);
    butterfly<G, 2 * M>(acc, e, wsum, weighted);
  }
}

// What a lane holds of the key it resolved.  A key without a row has the zero
// row's address, zero metadata and weight 0 for its (zero) values, while its
// own weight still counts in the weight sum; so nothing has to be selected
// per row: a slot past the end of the bag adds zeros.
struct LaneKey {
  uint64_t addr;
  float w;   // weight of the row's values
  float ws;  // the key's share of the weight sum
  Meta m;
};

// Keys a group takes per round, one per lane; the 16-lane rows of a wider
// group all resolve the same 16 keys, so that one DPP move broadcasts a value
// (from lane 17 to a group of 32 takes three or four instructions, which cost
// weighted 512-byte rows 20 %).
template <int G>
constexpr int kRound = G < 16 ? G : 16;

// U keys of a round, from its key J0 on, after their broadcast.  EARLY: their
// metadata too, which the lane that resolved the key has loaded.
template <int SDT, int U, bool W>
struct BatchKeys {
  uint64_t addr[U];
  float w[U];
  float ws[U];
  Meta m[Fmt<SDT>::meta != 0 ? U : 1];
};

template <int G, int J>
__device__ __forceinline__ float group_bcastf(float v) {
  return __uint_as_float(group_bcast<G, J>(__float_as_uint(v)));
}

template <int SDT, int K, int U, bool W, bool EARLY, int J0, int u = 0>
__device__ __forceinline__ void group_bcast_batch(const LaneKey& k, BatchKeys<SDT, U, W>& b) {
  if constexpr (u < U) {
    static_assert(J0 + u < K, "broadcast source outside the group");
    const uint32_t lo = group_bcast<K, J0 + u>((uint32_t)k.addr);
    const uint32_t hi = group_bcast<K, J0 + u>((uint32_t)(k.addr >> 32));
    b.addr[u] = ((uint64_t)hi << 32) | lo;
    // kept as one register pair: taken apart, adding the lane's offset takes
    // two 64-bit additions and their zero-extensions instead of one addition
    asm("" : "+v"(b.addr[u]));
    if constexpr (W) {
      b.w[u] = group_bcastf<K, J0 + u>(k.w);
      b.ws[u] = group_bcastf<K, J0 + u>(k.ws);
    }
    if constexpr (Fmt<SDT>::meta != 0 && EARLY) {
      b.m[u].s = group_bcastf<K, J0 + u>(k.m.s);
      if constexpr (SDT == kQU8F32 || SDT == kXI8AF32 || SDT == kQU8F16)
        b.m[u].o = group_bcastf<K, J0 + u>(k.m.o);
      else
        b.m[u].o = 0.0f;
    }
    group_bcast_batch<SDT, K, U, W, EARLY, J0, u + 1>(k, b);
  }
}

// acc += row, or acc = fma(row, wt, acc) when weighted, for one slice of a
// stored row.  f16 slices accumulate with one v_fma_mix_f32 per element (same
// bits as widening then adding).  A key without a row adds the zero row (zero
// metadata, wt = 0): adding +0 leaves acc unchanged (acc starts at +0 and a
// round-to-nearest sum is -0 only when both terms are), and wt = 0 keeps a
// non-finite weight of such a key out of the sum.
template <int SDT, int VB, bool W, int E>
__device__ __forceinline__ void add_slice(float (&acc)[E], const Vec<VB>& v, const Meta& m, float wt) {
  if constexpr (SDT == kF16) {
#pragma unroll
    for (int c = 0; c < E / 2; ++c) {
      if constexpr (W) {
        acc[2 * c] = fma_half_lo(v.w[c], wt, acc[2 * c]);
        acc[2 * c + 1] = fma_half_hi(v.w[c], wt, acc[2 * c + 1]);
      } else {
        acc[2 * c] = acc_half_lo(acc[2 * c], v.w[c]);
        acc[2 * c + 1] = acc_half_hi(acc[2 * c + 1], v.w[c]);
      }
    }
  } else {
    float x[E];
    decode<SDT, VB>(v, m, x);
#pragma unroll
    for (int c = 0; c < E; ++c) acc[c] = W ? __builtin_fmaf(x[c], wt, acc[c]) : acc[c] + x[c];
  }
}

// The rows of U keys of a round, from its key J0 on: every load in flight, then
// added in key order.  value_bytes: the place of the metadata in a row.
template <int SDT, int VB, int K, int U, bool W, bool EARLY, int J0>
__device__ __forceinline__ void add_batch(const LaneKey& k, uint32_t off, uint32_t value_bytes, float (&acc)[VB / Fmt<SDT>::esize],
                                          float& wsum) {
  BatchKeys<SDT, U, W> b;
  group_bcast_batch<SDT, K, U, W, EARLY, J0>(k, b);
  Vec<VB> v[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    v[u] = load_slice<VB>(b.addr[u] + off);
    // the zero row has zeros behind its kZeroRowBytes too
    if constexpr (Fmt<SDT>::meta != 0 && !EARLY) b.m[u] = load_meta_any<SDT>(b.addr[u] + value_bytes);
  }
  __builtin_amdgcn_sched_barrier(0);  // no addition moves up between the loads
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if constexpr (W) wsum += b.ws[u];
    add_slice<SDT, VB, W>(acc, v[u], b.m[Fmt<SDT>::meta != 0 ? u : 0], W ? b.w[u] : 1.0f);
  }
}

// The kernels' arguments: only what these shapes read (PoolLaunch carries a
// table array for multi-table launches; a smaller kernarg segment is quicker
// to set up per launch).
struct SplitArgs {
  const void* keys;
  const void* offsets;  // null: fixed hotness
  const void* weights;
  const uint8_t* table;
  void* out;
  int64_t num_keys;
  int64_t hotness;
  uint64_t row_bytes;
  uint64_t num_rows;
  int64_t count;
  int64_t out_stride;
  int key_bytes;
  int weight_dtype;
  int mean;
  int out_dtype;
  int gpb_shift;
};

// Long bags over a set-associative cache (with or without a backing table):
// the split kernel's arguments plus the cache.
struct SplitCacheArgs : SplitArgs {
  const uint8_t* cache_data;
  const void* cache_tags;
  uint64_t num_sets;
  unsigned long long* miss_counter;  // optional, kMissStripes * kMissStripeWords words
};

// The address of a key's row in a cache-backed table: the cache slot
// set * 8 + way on a hit (the lowest way whose rebuilt key tag * num_sets + set
// equals the key, as resolve_row), else the backing table's row when it holds
// the key, else 0.  *miss reports a cache miss.
template <typename A>
__device__ __forceinline__ uint64_t cache_row(const A& a, int64_t key, bool* miss) {
  uint32_t set, mask = 0;
  if (a.key_bytes == 4) {
    const uint32_t uk = (uint32_t)(int32_t)key;
    const uint32_t ns = (uint32_t)a.num_sets;
    set = uk % ns;
    const uint4* tp = reinterpret_cast<const uint4*>(reinterpret_cast<const int32_t*>(a.cache_tags) +
                                                     (uint64_t)set * 8);
    const uint4 t0 = tp[0];
    const uint4 t1 = tp[1];
    const uint32_t t[8] = {t0.x, t0.y, t0.z, t0.w, t1.x, t1.y, t1.z, t1.w};
#pragma unroll
    for (int w = 0; w < 8; ++w) mask |= (uint32_t)(t[w] * ns + set == uk) << w;
  } else {
    const uint64_t uk = (uint64_t)key;
    set = (uint32_t)(uk % a.num_sets);
    const uint4* tp = reinterpret_cast<const uint4*>(reinterpret_cast<const int64_t*>(a.cache_tags) +
                                                     (uint64_t)set * 8);
    uint64_t t[8];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const uint4 q = tp[c];
      t[2 * c] = (uint64_t)q.x | ((uint64_t)q.y << 32);
      t[2 * c + 1] = (uint64_t)q.z | ((uint64_t)q.w << 32);
    }
#pragma unroll
    for (int w = 0; w < 8; ++w) mask |= (uint32_t)(t[w] * a.num_sets + set == uk) << w;
  }
  *miss = mask == 0;
  const uint32_t rb32 = (uint32_t)a.row_bytes;  // launcher: row_bytes < 2^32, slots and rows < 2^31
  if (mask) return (uint64_t)a.cache_data + (uint64_t)(set * 8u + (uint32_t)__builtin_ctz(mask)) * rb32;
  if (a.table != nullptr && (uint64_t)key < a.num_rows) return (uint64_t)a.table + (uint64_t)(uint32_t)key * rb32;
  return 0;
}

// Adds the workgroup's per-lane miss counts to its word of the striped miss
// counter with one atomic (every thread of the workgroup calls it).
__device__ __forceinline__ void add_group_misses(unsigned long long* counter, uint32_t misses) {
  __shared__ uint32_t wave_misses[16];
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) misses += __shfl_xor(misses, o);
  if ((threadIdx.x & 63) == 0) wave_misses[threadIdx.x >> 6] = misses;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t m = 0;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) m += wave_misses[w];
    if (m) atomicAdd(counter + (blockIdx.x & (kMissStripes - 1)) * kMissStripeWords, (unsigned long long)m);
  }
}

// This lane's slice of every row: bytes [off, off + VB) of the value area; a
// lane past its end (in_row false) reads the last slice and stores nothing.
struct Slice {
  uint32_t off;
  bool in_row;
};
template <int VB, int G>
__device__ __forceinline__ Slice lane_slice(uint32_t value_bytes, int gl, uint32_t column) {
  const uint32_t at = (column * G + (uint32_t)gl) * VB;
  Slice s;
  s.in_row = at < value_bytes;
  s.off = at < value_bytes - VB ? at : value_bytes - VB;  // launcher: VB <= value_bytes <= the zero row
  return s;
}

// part[q] = the keys that row q of each G-lane group resolved (G a multiple of
// 16), in every row of the group.
template <int G>
__device__ __forceinline__ void spread_rows(uint32_t v, uint32_t (&part)[G / 16]) {
  if constexpr (G == 64) {
    const auto h = __builtin_amdgcn_permlane32_swap(v, v, false, false);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const auto r = __builtin_amdgcn_permlane16_swap(h[q], h[q], false, false);
      part[2 * q] = r[0];
      part[2 * q + 1] = r[1];
    }
  } else if constexpr (G == 32) {
    const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    part[0] = r[0];
    part[1] = r[1];
  } else {
    part[0] = v;
  }
}
template <int G, bool W>
__device__ __forceinline__ void spread_keys(const LaneKey& k, LaneKey (&part)[G / 16]) {
  uint32_t lo[G / 16], hi[G / 16], w[G / 16], ws[G / 16];
  spread_rows<G>((uint32_t)k.addr, lo);
  spread_rows<G>((uint32_t)(k.addr >> 32), hi);
  if constexpr (W) {
    spread_rows<G>(__float_as_uint(k.w), w);
    spread_rows<G>(__float_as_uint(k.ws), ws);
  }
#pragma unroll
  for (int q = 0; q < G / 16; ++q) {
    part[q] = LaneKey{((uint64_t)hi[q] << 32) | lo[q], 0.0f, 0.0f, Meta{0.0f, 0.0f}};
    if constexpr (W) {
      part[q].w = __uint_as_float(w[q]);
      part[q].ws = __uint_as_float(ws[q]);
    }
  }
}

template <int SDT, int VB, int G, bool W, bool CACHE = false>
__global__ __launch_bounds__(1024) void pool_split_kernel(
    std::conditional_t<CACHE, SplitCacheArgs, SplitArgs> a) {
  constexpr int ES = Fmt<SDT>::esize;
  constexpr int E = VB / ES;
  constexpr int K = kRound<G>;
  // rows in flight: fewer with 16 values a lane or weights and a cache, whose
  // batch would leave the registers of a 1024-thread workgroup
  constexpr int UMAX = E > 8 || (W && CACHE) ? 8 : 16;
  constexpr int U = K < UMAX ? K : UMAX;  // a round's keys in batches of U
  // A probe of the cache's tags costs far more than the moves of its result: the
  // lanes of a wide group probe a key each, and the rows' results are spread
  // over the group 16 at a time.  256 bags of ~1,000 keys, every row of the group
  // probing the same 16 keys and this, all hits: 512-byte rows 15.1 and 13.9 us,
  // 1,024-byte fp32 rows 22.9 and 19.2, 2,400-byte rows 62.3 and 51.0; 4,096 bags of
  // ~40 keys, 512-byte fp32 rows 11.8 and 10.5 us.
  constexpr int R = CACHE ? G : K;  // keys of a round
  extern __shared__ float lds[];

  const int tid = threadIdx.x;
  const int gl = tid & (G - 1);
  const int chunk = tid / G;
  const int gpb_shift = a.gpb_shift;
  const int gpb = 1 << gpb_shift;
  const int64_t bag = blockIdx.x;

  int64_t s, e;
  if (a.offsets != nullptr) {
    s = load_key(a.offsets, a.key_bytes, bag);
    e = load_key(a.offsets, a.key_bytes, bag + 1);
    s = s < 0 ? 0 : (s > a.num_keys ? a.num_keys : s);
    e = e < s ? s : (e > a.num_keys ? a.num_keys : e);
  } else {
    s = bag * a.hotness;
    e = s + a.hotness;
  }
  int64_t cs = s, ce = e;
  if (e > s) {
    const int64_t per = (e - s + gpb - 1) >> gpb_shift;
    cs = s + chunk * per;
    if (cs > e) cs = e;
    ce = cs + per < e ? cs + per : e;
  }

  const uint64_t table = (uint64_t)a.table;
  const uint64_t num_rows = a.num_rows;
  const uint32_t rb32 = (uint32_t)a.row_bytes;  // launcher: row_bytes < 2^32
  const uint32_t value_bytes = (uint32_t)a.count * ES;
  const Slice sl = lane_slice<VB, G>(value_bytes, gl, blockIdx.y);

  float acc[E];
#pragma unroll
  for (int c = 0; c < E; ++c) acc[c] = 0.0f;
  float wsum = 0.0f;

  uint32_t misses = 0;
  const int kl = gl & (R - 1);
  // one key per lane and round of R keys, loaded a round ahead
  int64_t ahead = cs + kl < ce ? load_key(a.keys, a.key_bytes, cs + kl) : -1;
  for (int64_t k0 = cs; k0 < ce; k0 += R) {
    const int64_t kk = k0 + kl;
    const int64_t key = ahead;
    if (kk + R < ce) ahead = load_key(a.keys, a.key_bytes, kk + R);
    LaneKey lk{(uint64_t)g_zero_row, 0.0f, 0.0f, Meta{0.0f, 0.0f}};
    if (kk < ce) {
      bool real;
      if constexpr (CACHE) {
        bool miss;
        const uint64_t row = cache_row(a, key, &miss);
        misses += miss ? 1u : 0u;
        real = row != 0;
        if (real) lk.addr = row;
      } else {
        real = (uint64_t)key < num_rows;  // keys outside the table read nothing
        if (real) {
          lk.addr = table + (uint64_t)(uint32_t)key * rb32;
          if constexpr (Fmt<SDT>::meta != 0) lk.m = load_meta_any<SDT>(lk.addr + value_bytes);
        }
      }
      if constexpr (W) {
        lk.ws = load_weight(a.weights, a.weight_dtype, kk);
        lk.w = real ? lk.ws : 0.0f;
      }
    }
    const int n = (int)((ce - k0) < R ? (ce - k0) : R);
    LaneKey part[R / K];
    if constexpr (R > K) spread_keys<R, W>(lk, part);
    else part[0] = lk;
    // batch from key j0 of the round on (compile time, so every lane move has
    // an immediate source lane)
    auto batch = [&](auto jc) {
      constexpr int j0 = decltype(jc)::value;
      if (j0 < n) add_batch<SDT, VB, K, U, W, true, j0 % K>(part[j0 / K], sl.off, value_bytes, acc, wsum);
    };
    for_batches<U, 0, R / U>(batch);
  }

  // butterfly over the wave's groups (the same pairing and additions as pool_kernel)
  butterfly<G>(acc, E, wsum, W);
  if constexpr (CACHE) {
    // one miss-counter atomic per workgroup: thousands on one address
    // serialize; every column of a bag sees the same misses
    if (a.miss_counter != nullptr && blockIdx.y == 0) add_group_misses(a.miss_counter, misses);
  }

  // waves' partial rows, added in wave order
  constexpr int row_elems = G * E;
  const int wave = tid >> 6;
  const int waves = (gpb * G) >> 6;
  float* red = lds;
  float* wred = lds + (blockDim.x >> 6) * row_elems;
  if ((tid & 63) < G) {
#pragma unroll
    for (int c = 0; c < E; ++c) red[wave * row_elems + gl * E + c] = acc[c];
    if (gl == 0) wred[wave] = wsum;
  }
  __syncthreads();
  for (int x = tid; x < row_elems; x += (int)blockDim.x) {
    const Slice xs = lane_slice<VB, G>(value_bytes, x / E, blockIdx.y);
    if (!xs.in_row) break;  // and so is every later element
    float part[16];
    float wp[16];
#pragma unroll
    for (int w = 0; w < 16; ++w) {
      part[w] = w < waves ? red[w * row_elems + x] : 0.0f;
      wp[w] = (W && w < waves) ? wred[w] : 0.0f;
    }
    float v = part[0];
    float ws = wp[0];
#pragma unroll
    for (int w = 1; w < 16; ++w) {
      if (w < waves) {
        v += part[w];
        ws += wp[w];
      }
    }
    if (a.mean) {
      const float d = W ? ws : (float)(e - s);
      v = (d == 0.0f) ? 0.0f : v / d;
    }
    const uint64_t o = (uint64_t)a.out + (uint64_t)(bag * a.out_stride);
    const uint32_t elem = xs.off / ES + (uint32_t)(x % E);
    if (a.out_dtype == kF16)
      *reinterpret_cast<gptr_w<uint16_t>>(o + (uint64_t)elem * 2) = f2h(v);
    else
      *reinterpret_cast<gptr_w<float>>(o + (uint64_t)elem * 4) = v;
  }
}

template <int SDT, int VB, int G>
hipError_t launch_split_g(const PoolLaunch& a, const PoolSlices& g, hipStream_t stream) {
  SplitArgs s{};
  s.keys = a.keys;
  s.offsets = a.offsets;
  s.weights = a.weights;
  s.table = a.src.table;
  s.out = a.out;
  s.num_keys = a.num_keys;
  s.hotness = a.hotness;
  s.row_bytes = a.src.row_bytes;
  s.num_rows = a.src.num_rows;
  s.count = a.count;
  s.out_stride = a.out_stride;
  s.key_bytes = a.key_bytes;
  s.weight_dtype = a.weight_dtype;
  s.mean = a.mean;
  s.out_dtype = a.out_dtype;
  s.gpb_shift = 0;
  while ((1 << s.gpb_shift) < g.gpb) ++s.gpb_shift;
  const int threads = g.gpb * G;
  const dim3 grid((unsigned)a.num_bags, (unsigned)g.columns), block((unsigned)threads);
  // one partial row and weight sum per wave
  const unsigned lds = (unsigned)(threads / 64) * (unsigned)(G * (VB / Fmt<SDT>::esize) * 4 + 4);
  if (a.src.cache_data != nullptr) {
    if constexpr (Fmt<SDT>::meta == 0) {
      SplitCacheArgs c{};
      static_cast<SplitArgs&>(c) = s;
      c.cache_data = a.src.cache_data;
      c.cache_tags = a.src.cache_tags;
      c.num_sets = a.src.num_sets;
      c.miss_counter = a.miss_counter;
      if (a.weighted)
        hipLaunchKernelGGL((pool_split_kernel<SDT, VB, G, true, true>), grid, block, lds, stream, c);
      else
        hipLaunchKernelGGL((pool_split_kernel<SDT, VB, G, false, true>), grid, block, lds, stream, c);
      return hipGetLastError();
    } else {
      return hipErrorInvalidValue;
    }
  }
  if (a.weighted)
    hipLaunchKernelGGL((pool_split_kernel<SDT, VB, G, true>), grid, block, lds, stream, s);
  else
    hipLaunchKernelGGL((pool_split_kernel<SDT, VB, G, false>), grid, block, lds, stream, s);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// short bags: one G-lane group per bag, 256 / G bags per workgroup, the bag's
// keys in key order (the same additions as pool_kernel's one-group-per-bag
// path, so the same bits).  MT: several tables in one launch, table blockIdx.z
// (its bag b writes row b * out_stride + table * out_table_stride): the table is
// the same for a whole workgroup, where a division of the bag's index took a
// fifth of the kernel's instructions.
// ---------------------------------------------------------------------------
struct ShortArgs {
  const void* keys;
  const void* offsets;  // null: fixed hotness
  const void* weights;
  void* out;
  const uint8_t* table;  // one table (MT = false)
  int64_t num_keys;
  int64_t num_bags;  // of one table
  int64_t hotness;
  uint64_t row_bytes;
  uint64_t num_rows;
  int64_t count;
  int64_t out_stride;
  int64_t out_table_stride;
  int key_bytes;
  int weight_dtype;
  int mean;
  int out_dtype;
  int staged;  // output rows go through LDS: whole slices, 16-byte aligned rows
};
struct ShortArgsMT : ShortArgs {
  const uint8_t* tables[kMaxPoolTables];
  uint32_t table_rows[kMaxPoolTables];
};

template <int SDT, int VB, int G, bool W, bool MT, int U, bool EARLY>
__global__ __launch_bounds__(256) void pool_short_kernel(std::conditional_t<MT, ShortArgsMT, ShortArgs> a) {
  constexpr int ES = Fmt<SDT>::esize;
  constexpr int E = VB / ES;
  constexpr int K = kRound<G>;

  const int tid = threadIdx.x;
  const int gl = tid & (G - 1);
  const int64_t first_bag = MT ? (int64_t)blockIdx.z * a.num_bags : 0;
  const int64_t in_table = (int64_t)blockIdx.x * (256 / G) + tid / G;
  const int64_t bag = first_bag + in_table;
  const bool live = in_table < a.num_bags;  // uniform over the group

  int64_t s = 0, e = 0;
  if (live) {
    if (a.offsets != nullptr) {
      s = load_key(a.offsets, a.key_bytes, bag);
      e = load_key(a.offsets, a.key_bytes, bag + 1);
      s = s < 0 ? 0 : (s > a.num_keys ? a.num_keys : s);
      e = e < s ? s : (e > a.num_keys ? a.num_keys : e);
    } else {
      s = bag * a.hotness;
      e = s + a.hotness;
    }
  }
  uint64_t table = (uint64_t)a.table;
  uint64_t num_rows = a.num_rows;
  uint64_t out_row = (uint64_t)a.out;
  if constexpr (MT) {
    table = (uint64_t)a.tables[blockIdx.z];
    num_rows = a.table_rows[blockIdx.z];
    out_row += (uint64_t)(blockIdx.z * a.out_table_stride);
  }
  out_row += (uint64_t)(in_table * a.out_stride);
  const uint32_t rb32 = (uint32_t)a.row_bytes;  // launcher: row_bytes < 2^32
  const uint32_t value_bytes = (uint32_t)a.count * ES;
  const Slice sl = lane_slice<VB, G>(value_bytes, gl, blockIdx.y);

  float acc[E];
#pragma unroll
  for (int c = 0; c < E; ++c) acc[c] = 0.0f;
  float wsum = 0.0f;

  // One key (and weight) per lane and round of K keys, loaded a round ahead:
  // the bag's chain is offsets -> keys -> rows -> rows -> ..., without a wait
  // for keys between the rounds.
  struct Raw {
    int64_t key;
    float w;
  };
  const auto load_raw = [&](int64_t kk) {
    Raw r{-1, 0.0f};  // outside every table
    if (kk < e) {
      r.key = load_key(a.keys, a.key_bytes, kk);
      if (W) r.w = load_weight(a.weights, a.weight_dtype, kk);
    }
    return r;
  };
  const auto resolve = [&](const Raw& r) {
    LaneKey lk{(uint64_t)g_zero_row, 0.0f, r.w, Meta{0.0f, 0.0f}};
    if ((uint64_t)r.key < num_rows) {  // keys outside the table read nothing
      lk.addr = table + (uint64_t)(uint32_t)r.key * rb32;
      lk.w = r.w;
      if constexpr (Fmt<SDT>::meta != 0 && EARLY) lk.m = load_meta_any<SDT>(lk.addr + value_bytes);
    }
    return lk;
  };
  const int kl = gl & (K - 1);
  const Raw first = load_raw(s + kl);
  Raw ahead = load_raw(s + K + kl);
  LaneKey lk = resolve(first);
  for (int64_t k0 = s; k0 < e; k0 += K) {
    const LaneKey next = resolve(ahead);
    ahead = load_raw(k0 + 2 * K + kl);
    const int n = (int)((e - k0) < K ? (e - k0) : K);
    auto batch = [&](auto jc) {
      constexpr int j0 = decltype(jc)::value;
      if (j0 < n) add_batch<SDT, VB, K, U, W, EARLY, j0>(lk, sl.off, value_bytes, acc, wsum);
    };
    for_batches<U, 0, K / U>(batch);
    lk = next;
  }

  if (a.mean) {
    const float d = W ? wsum : (float)(e - s);
#pragma unroll
    for (int c = 0; c < E; ++c) acc[c] = (d == 0.0f) ? 0.0f : acc[c] / d;
  }
  const bool out_f16 = a.out_dtype == kF16;
  if constexpr (E >= 8) {
    if (a.staged && E * (out_f16 ? 2 : 4) > 16) {  // uniform over the launch
      // A lane's values are 32 or 64 output bytes: stored from its registers,
      // each instruction writes 16 bytes of each.  Through LDS every store
      // instruction writes G * 16 contiguous bytes.
      __shared__ __align__(16) uint32_t stage[256 * E];
      uint32_t* mine = stage + (tid - gl) * E;  // the group's row
      const int words = out_f16 ? E / 2 : E;    // per lane
      if (out_f16) {
#pragma unroll
        for (int i = 0; i < E / 2; ++i)
          mine[gl * (E / 2) + i] = (uint32_t)f2h(acc[2 * i]) | ((uint32_t)f2h(acc[2 * i + 1]) << 16);
      } else {
#pragma unroll
        for (int i = 0; i < E; ++i) mine[gl * E + i] = __float_as_uint(acc[i]);
      }
      // read by other lanes of the wave, whose LDS accesses stay in order; the
      // fences keep the compiler from moving them
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      const uint32_t es = out_f16 ? 2 : 4;
      const uint32_t first = blockIdx.y * (uint32_t)(G * E) * es;  // the column's place in the output row
      const uint32_t bytes = (uint32_t)a.count * es;
#pragma unroll
      for (int j = 0; j < E / 4; ++j) {
        const uint32_t chunk = (uint32_t)(j * G + gl) * 16;
        if (4 * j < words && live && first + chunk < bytes) {
          const u32x4 x = *reinterpret_cast<const u32x4*>(mine + chunk / 4);
          __builtin_nontemporal_store(x, reinterpret_cast<gptr_w<u32x4>>(out_row + first + chunk));
        }
      }
      return;
    }
  }
  if (live && sl.in_row)
    store_slice<E>(out_row + (uint64_t)(sl.off / ES) * (out_f16 ? 2 : 4), acc, out_f16);
}

template <int SDT, int VB, int G, bool MT>
hipError_t launch_short_g(const PoolLaunch& a, const PoolSlices& g, hipStream_t stream) {
  std::conditional_t<MT, ShortArgsMT, ShortArgs> s{};
  s.keys = a.keys;
  s.offsets = a.offsets;
  s.weights = a.weights;
  s.out = a.out;
  s.table = a.src.table;
  s.num_keys = a.num_keys;
  s.num_bags = MT ? a.bags_per_table : a.num_bags;
  s.hotness = a.hotness;
  s.row_bytes = a.src.row_bytes;
  s.num_rows = a.src.num_rows;
  s.count = a.count;
  s.out_stride = a.out_stride;
  s.out_table_stride = a.out_table_stride;
  s.key_bytes = a.key_bytes;
  s.weight_dtype = a.weight_dtype;
  s.mean = a.mean;
  s.out_dtype = a.out_dtype;
  s.staged = a.count * Fmt<SDT>::esize % VB == 0 && ((uint64_t)a.out | (uint64_t)a.out_stride |
                                                     (uint64_t)(MT ? a.out_table_stride : 0)) % 16 == 0;
  if constexpr (MT) {
    for (int t = 0; t < a.num_tables; ++t) {
      s.tables[t] = a.tables[t];
      s.table_rows[t] = (uint32_t)a.table_rows[t];
    }
  }
  const int64_t per_wg = 256 / G;
  const dim3 grid((unsigned)((s.num_bags + per_wg - 1) / per_wg), (unsigned)g.columns,
                  MT ? (unsigned)a.num_tables : 1u);
  const dim3 block(256);
  // 4 rows in flight per lane where more waves wait than the chip holds: the
  // registers of 8 or 16 rows would keep waves out (26 tables of 8,192 bags of
  // ~20 keys: 4 -> 104 us, 8 -> 111 us), and for bags of up to 4 keys, whose other
  // rows would be zero rows (16,384 bags of 2 256-byte rows: 4 -> 2.96 us, 8 -> 3.31).
  // Other launches of at most 4 waves per SIMD lose none to 8 rows (16,384 bags of ~30
  // 200-byte rows: 13.9 -> 13.6 us), and bags past 48 keys keep 16 (8 where a lane
  // decodes 16 values or a round has 8 keys).
  // A row's metadata is loaded with the row, by every lane.  Loaded a round ahead by
  // the lane that resolves the key it takes a lane move instead, which saves 3 to 5 %
  // while the rows' lines stay in the caches (1,024 bags of ~20 132-byte rows 5.5 and
  // 5.3 us, 16,384 bags of 8 6.5 and 5.7), but the last one has to come twice where they
  // do not (uniform keys over 1 M rows, 8,192 bags of ~30 14.4 and 16.2 us, 32,768 bags
  // 43.3 and 58.6; 36-byte rows, 32,768 bags of ~20 17.6 and 25.3).
  const int64_t avg = a.keys_per_bag > 0 ? a.keys_per_bag
                                         : a.num_keys / (a.num_bags > 0 ? a.num_bags : 1);
  const bool few = (int64_t)grid.x * grid.y * grid.z <= 4 * 256;  // workgroups of a wave per SIMD
  constexpr bool kMeta = Fmt<SDT>::meta != 0;
  const bool early = kMeta && (uint64_t)a.num_keys <= (48u << 20) / (a.src.row_bytes + 127);  // by lines touched
  constexpr int kWide = VB / Fmt<SDT>::esize > 8 || kRound<G> < 16 ? 8 : 16;
#define NVE_LAUNCH_SHORT(W, U, EARLY) \
  hipLaunchKernelGGL((pool_short_kernel<SDT, VB, G, W, MT, U, EARLY>), grid, block, 0, stream, s)
  if (avg > 48) {
    if (a.weighted) NVE_LAUNCH_SHORT(true, kWide, false); else NVE_LAUNCH_SHORT(false, kWide, false);
  } else if (few && avg > 4 && early) {
    if (a.weighted) NVE_LAUNCH_SHORT(true, 8, kMeta); else NVE_LAUNCH_SHORT(false, 8, kMeta);
  } else if (few && avg > 4) {
    if (a.weighted) NVE_LAUNCH_SHORT(true, 8, false); else NVE_LAUNCH_SHORT(false, 8, false);
  } else {
    if (a.weighted) NVE_LAUNCH_SHORT(true, 4, false); else NVE_LAUNCH_SHORT(false, 4, false);
  }
#undef NVE_LAUNCH_SHORT
  return hipGetLastError();
}

// MT launches take f16 / f32 rows only.
template <int SDT, int VB, int G, bool SHORT = true, bool SPLIT = true>
hipError_t launch_slices_g(const PoolLaunch& a, const PoolSlices& g, hipStream_t stream) {
  if constexpr (SPLIT) {
    if (g.gpb > 1) return launch_split_g<SDT, VB, G>(a, g, stream);
  }
  if constexpr (SHORT) {
    if constexpr (Fmt<SDT>::meta == 0) {
      if (a.num_tables > 0) return launch_short_g<SDT, VB, G, true>(a, g, stream);
    }
    if (g.gpb == 1) return launch_short_g<SDT, VB, G, false>(a, g, stream);
  }
  return hipErrorInvalidValue;
}

// The slices that pool_slices chooses: 16 bytes for wide f16 / f32 rows, for wide
// byte rows 8 bytes up to 128 of them and, where a group has a bag to itself, up to
// 512, else 16.
template <int SDT>
hipError_t launch_slices_sdt(const PoolLaunch& a, const PoolSlices& g, hipStream_t stream) {
  switch (g.vb * 100 + g.g) {
    case 408: return launch_slices_g<SDT, 4, 8>(a, g, stream);
    case 808: return launch_slices_g<SDT, 8, 8>(a, g, stream);
    case 1664: return launch_slices_g<SDT, 16, 64>(a, g, stream);
  }
  if constexpr (Fmt<SDT>::esize == 1) {
    switch (g.vb * 100 + g.g) {
      case 816: return launch_slices_g<SDT, 8, 16>(a, g, stream);
      case 832: return launch_slices_g<SDT, 8, 32, true, false>(a, g, stream);
      case 864: return launch_slices_g<SDT, 8, 64, true, false>(a, g, stream);
      case 1616: return launch_slices_g<SDT, 16, 16, false, true>(a, g, stream);
      case 1632: return launch_slices_g<SDT, 16, 32, false, true>(a, g, stream);
    }
  } else {
    switch (g.vb * 100 + g.g) {
      case 1608: return launch_slices_g<SDT, 16, 8>(a, g, stream);
      case 1616: return launch_slices_g<SDT, 16, 16>(a, g, stream);
      case 1632: return launch_slices_g<SDT, 16, 32>(a, g, stream);
    }
  }
  return hipErrorInvalidValue;
}

}  // namespace

}  // namespace nve_amd
