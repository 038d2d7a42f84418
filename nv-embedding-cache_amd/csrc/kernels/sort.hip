// sort.hip -- stable LSD radix sort of (uint64 key, uint32 value) pairs, an
// exclusive scan and a key-span reduction: the sorting primitives behind the
// cache insert (histogram and set grouping) and dedup.
//
// The reference uses CUB (cub::DeviceRadixSort::SortPairs[Descending],
// DeviceRunLengthEncode::Encode, DeviceScan::ExclusiveSum; deduper.cuh:157-200,
// gather_keys_data_ptrs.cuh:154-183, ec_set_associative_modify.cuh:472-497).
// Only the mathematical results matter (a stable sort; descending sorts are
// expressed by the caller as ascending sorts of a complemented key).
//
// One launch counts every digit of every pass (the digit counts of a pass do
// not depend on the order of the keys), then one launch per pass moves the
// keys.  Digits have 8 bits, or 9 when that takes fewer passes (the last digit
// keeps only the bits below end_bit).
//   count    at most kCountGroups workgroups, each the digit counts of its
//            tiles for every pass; it also clears the passes' state;
//   sweep    a 1024-thread workgroup per tile of 2,048 or 4,096 keys.  A wave ranks
//            its keys with one ballot per digit bit and a running count per digit
//            in LDS; the tile's counts are published, the tile is staged in LDS
//            in digit order, and each digit's place is found from the tiles
//            before: their published counts are added, walking back until one
//            that already knows its own place.  Consecutive threads then store
//            consecutive positions of a digit's run.
// A tile is numbered by a counter that its workgroup increments when it starts,
// so the tiles it waits for have started before it, and every wait ends.  A
// published word holds count and state together (one 64-bit store), so no other
// memory has to be ordered against it.
//
// Bound: latency.  A pass moves 24 bytes a key (6 MB at 262,144 keys), and each of its
// tiles also reads the digit counts of up to 64 counting workgroups (128 KB from L2:
// 8 MB for the 64 tiles of 262,144 keys).  Three launches per pass (tile counts, a
// scan of each digit's row, the scatter) took nine launches for the three passes of
// a table's keys; the four of this sort and the one launch of the dedup's runs take
// the dedup of 8,192 keys from 70 to 45 us, of 32,768 keys from 71 to 51, of 131,072
// keys from 70 to 61, of 262,144 keys from 74 to 71 and of 1,000,000 keys from 123 to
// 107.  Keys that differ in all 64 bits take eight passes over 450,000 to 600,000 keys
// 2 to 4 % longer than the three launches each did (304 and 316 us for 600,000), one
// key repeated 4,000,000 times 5 % (267 and 281); of 1,000,000 such keys 407 and 353 us.
// Tiles are large so that each has few predecessors: with 1024-key tiles every one of
// 256 tiles walks back through most of them.  Nor do more words per step of the walk
// help (1,000,000 keys: kLookAhead 4 and 8 take 107.5 and 109.7 us): the walk is bound
// by the words it reads.
//
// The exclusive scan of an array (run heads in the insert) is
// reduce-then-scan over 4096-element blocks: block sums, a scan of the sums
// (recursively, in the caller's temporary storage), then each block rescans
// its elements from its offset.
#include <algorithm>
#include <type_traits>

#include "device_common.cuh"
#include "lane_moves.cuh"
#include "position_grad.cuh"
#include "sort_launch.hpp"
#include "tile_rank.cuh"

namespace nve_amd {

constexpr int kTileThreads = 1024;
constexpr int kTileWaves = kTileThreads / 64;
constexpr int kCountTile = 2 * kTileThreads;  // keys a counting workgroup has at least
constexpr int kMaxPasses = 8;     // 64 bits in digits of 8, or of 9
constexpr int kCountGroups = 64;  // workgroups whose digit counts every tile adds up

// The digits of a sort: pass p takes (key >> shift[p]) & mask[p].
struct RadixDigits {
  int passes;
  int shift[kMaxPasses];
  uint32_t mask[kMaxPasses];
};

// The sort key of position i: keys[i], or with a raw source the caller's key
// converted on the fly (sign bit flipped when src.flip).
template <bool RAW>
__device__ __forceinline__ uint64_t sort_key(const uint64_t* keys, const RadixSource& src, int64_t i) {
  if constexpr (RAW) {
    const int64_t k = load_key(src.keys, src.key_bytes, i);
    return src.flip ? flip_key(k, src.key_bytes) : (uint64_t)k;
  } else {
    return keys[i];
  }
}

// parts[workgroup][pass][kMaxBins] = digit counts of the workgroup's tiles;
// state[0 .. state_words) and clear[0 .. clear_words) = 0.  With pg.by_key, the
// gradient row of every key position.  With src.span_part, span_part[workgroup] = the
// OR of key ^ key[0] over its keys (the bits where they differ from the first).
template <bool RAW, int ITEMS>
__global__ __launch_bounds__(kTileThreads) void radix_count_kernel(const uint64_t* keys, RadixSource src,
                                                                   int64_t n, RadixDigits dg, uint32_t* parts,
                                                                   uint64_t* state, int64_t state_words,
                                                                   uint64_t* clear, int64_t clear_words,
                                                                   PositionGrad pg) {
  constexpr int kTile = kTileThreads * ITEMS;
  __shared__ uint32_t h[kMaxPasses * kMaxBins];
  __shared__ uint32_t rows[kTile];
  const int tid = threadIdx.x;
  for (int64_t w = (int64_t)blockIdx.x * kTileThreads + tid; w < state_words; w += (int64_t)gridDim.x * kTileThreads)
    state[w] = 0;
  for (int64_t w = (int64_t)blockIdx.x * kTileThreads + tid; w < clear_words; w += (int64_t)gridDim.x * kTileThreads)
    clear[w] = 0;
  for (int d = tid; d < dg.passes * kMaxBins; d += kTileThreads) h[d] = 0;
  __syncthreads();
  uint64_t diff = 0;
  const uint64_t k0 = sort_key<RAW>(keys, src, 0);
  for (int64_t base = (int64_t)blockIdx.x * kTile; base < n; base += (int64_t)gridDim.x * kTile) {
    uint64_t k[ITEMS];
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
      const int64_t i = base + r * kTileThreads + tid;
      k[r] = sort_key<RAW>(keys, src, i < n ? i : 0);
    }
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
      const bool valid = base + r * kTileThreads + tid < n;
      diff |= k[r] ^ k0;  // a lane past the end holds key 0
      for (int p = 0; p < dg.passes; ++p) {
        // the digit of the wave's first lane is added once for all lanes that
        // share it: a hot key's (or a high digit's) lanes would queue on its word
        const uint32_t d = (uint32_t)(k[r] >> dg.shift[p]) & dg.mask[p];
        const uint32_t lead = (uint32_t)__builtin_amdgcn_readfirstlane((int)d);
        const uint64_t same = __ballot(valid && d == lead);
        if (valid && d != lead) atomicAdd(&h[p * kMaxBins + d], 1u);
        if ((tid & 63) == 0 && same) atomicAdd(&h[p * kMaxBins + lead], (uint32_t)__popcll(same));
      }
    }
  }
  if (pg.by_key != nullptr) {  // uniform
    for (int64_t base = (int64_t)blockIdx.x * kTile; base < n; base += (int64_t)gridDim.x * kTile) {
      tile_rows<kTileThreads, kTile>(pg, base, rows);
      for (int x = tid; x < kTile && base + x < n; x += kTileThreads) pg.by_key[base + x] = rows[x];
      __syncthreads();
    }
  }
  if (src.span_part != nullptr) {  // uniform
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) diff |= __shfl_xor(diff, o);
    __shared__ uint64_t red[kTileWaves];
    if ((tid & 63) == 0) red[tid >> 6] = diff;
    __syncthreads();
    if (tid == 0) {
      uint64_t x = 0;
#pragma unroll
      for (int w = 0; w < kTileWaves; ++w) x |= red[w];
      src.span_part[blockIdx.x] = x;
    }
  }
  __syncthreads();
  uint32_t* out = parts + (int64_t)blockIdx.x * dg.passes * kMaxBins;
  for (int d = tid; d < dg.passes * kMaxBins; d += kTileThreads) out[d] = h[d];
}

// parts[0] = the sum of parts[0 .. nparts): with many tiles, each adding up
// nparts counts would cost more than this launch.
__global__ __launch_bounds__(256) void radix_total_kernel(uint32_t* parts, int nparts, int stride) {
  const int d = (int)(blockIdx.x * 256 + threadIdx.x);
  if (d >= stride) return;
  uint32_t t = 0;
#pragma unroll 16
  for (int w = 0; w < nparts; ++w) t += parts[(int64_t)w * stride + d];
  parts[d] = t;
}

// Inclusive scan across the 64 lanes of a wave.
__device__ __forceinline__ uint32_t wave_inclusive_scan(uint32_t v) {
  const int lane = lane_id();
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t t = shfl32(v, lane >= o ? lane - o : lane);
    if (lane >= o) v += t;
  }
  return v;
}

// Exclusive scan of one value per thread over a workgroup of NT threads
// (NT a multiple of 64, at most 4096); `total` receives the sum.  `lds` holds
// NT / 64 + 1 words; every thread of the workgroup must call it.
template <int NT>
__device__ __forceinline__ uint32_t block_exclusive_scan(uint32_t v, uint32_t* lds,
                                                         uint32_t* total) {
  constexpr int kWaves = NT / 64;
  const int lane = lane_id();
  const int wave = (int)threadIdx.x >> 6;
  const uint32_t inc = wave_inclusive_scan(v);
  if (lane == 63) lds[wave] = inc;
  __syncthreads();
  if (threadIdx.x < 64) {
    const uint32_t w = (int)threadIdx.x < kWaves ? lds[threadIdx.x] : 0u;
    const uint32_t wi = wave_inclusive_scan(w);
    if ((int)threadIdx.x < kWaves) lds[threadIdx.x] = wi - w;
    if ((int)threadIdx.x == kWaves - 1) lds[kWaves] = wi;
  }
  __syncthreads();
  const uint32_t res = inc - v + lds[wave];
  *total = lds[kWaves];
  __syncthreads();
  return res;
}

constexpr int kScanThreads = 256;
constexpr int kScanItems = 16;
constexpr int kScanBlock = kScanThreads * kScanItems;

// Sum of each 4096-element block.
__global__ __launch_bounds__(256) void scan_reduce_kernel(const uint32_t* data, int64_t m,
                                                          uint32_t* sums) {
  __shared__ uint32_t lds[kScanThreads / 64 + 1];
  const int64_t base = (int64_t)blockIdx.x * kScanBlock + (int64_t)threadIdx.x * kScanItems;
  uint32_t s = 0;
#pragma unroll
  for (int j = 0; j < kScanItems; ++j)
    if (base + j < m) s += data[base + j];
  uint32_t total;
  (void)block_exclusive_scan<kScanThreads>(s, lds, &total);
  if (threadIdx.x == 0) sums[blockIdx.x] = total;
}

// Exclusive scan of each block from its offset (sums[block], or 0 with a
// single block); the last block writes the grand total.
__global__ __launch_bounds__(256) void scan_down_kernel(uint32_t* data, int64_t m,
                                                        const uint32_t* offsets, uint32_t* total) {
  __shared__ uint32_t lds[kScanThreads / 64 + 1];
  const int64_t base = (int64_t)blockIdx.x * kScanBlock + (int64_t)threadIdx.x * kScanItems;
  uint32_t v[kScanItems];
  uint32_t s = 0;
#pragma unroll
  for (int j = 0; j < kScanItems; ++j) {
    v[j] = base + j < m ? data[base + j] : 0u;
    s += v[j];
  }
  uint32_t block_total;
  uint32_t run = block_exclusive_scan<kScanThreads>(s, lds, &block_total);
  const uint32_t off = offsets ? offsets[blockIdx.x] : 0u;
  run += off;
#pragma unroll
  for (int j = 0; j < kScanItems; ++j) {
    if (base + j < m) data[base + j] = run;
    run += v[j];
  }
  if (total != nullptr && blockIdx.x == gridDim.x - 1 && threadIdx.x == 0)
    *total = off + block_total;
}

constexpr int kLookAhead = 4;  // words read at a time while walking back

// Keys of the tiles before `tile`, from word[tile * stride]: adds published
// counts from tile - 1 down until one that includes all before it.
__device__ __forceinline__ uint64_t keys_before(const uint64_t* word, int64_t tile, int64_t stride) {
  uint64_t sum = 0;
  for (int64_t j = tile - 1; j >= 0;) {
    uint64_t w[kLookAhead];
#pragma unroll
    for (int u = 0; u < kLookAhead; ++u)
      w[u] = j - u >= 0 ? load_state(word + (j - u) * stride) : kStateBefore;  // nothing before the first tile
    bool open = true;  // every word so far was published, none of them the last to add
    int used = 0;
#pragma unroll
    for (int u = 0; u < kLookAhead; ++u) {
      if (open && w[u] >= kStateOwn) {
        sum += w[u] & kStateCount;
        ++used;
        if (w[u] >= kStateBefore) return sum;
      } else {
        open = false;
      }
    }
    j -= used;
    if (used == 0) __builtin_amdgcn_s_sleep(1);
  }
  return sum;
}

struct SweepArgs {
  const uint64_t* keys;
  const uint32_t* vals;
  RadixSource src;  // RAW: the first pass reads the caller's keys (vals null: values = positions)
  uint64_t* ko;
  uint32_t* vo;
  int64_t n;
  int shift;
  uint32_t mask;
  const uint32_t* parts;  // the pass's digit counts, nparts of them part_stride apart
  int nparts;
  int part_stride;
  uint64_t* state;  // the pass's words: tile counter, then kMaxBins per tile
};

template <int RB, bool RAW, int ITEMS>
__global__ __launch_bounds__(kTileThreads) void radix_sweep_kernel(SweepArgs a) {
  constexpr int kBins = 1 << RB;
  constexpr int kTile = kTileThreads * ITEMS;
  static_assert(kBins <= kTileThreads && kBins <= kMaxBins, "one thread per digit");
  __shared__ uint64_t sk[kTile];
  __shared__ uint32_t sv[kTile];
  __shared__ uint32_t cnt[kTileWaves][kBins];  // keys of digit d per wave, then of the waves before
  __shared__ uint32_t lstart[kBins];           // first position of digit d in the staged tile
  __shared__ uint32_t gbase[kBins];            // output position of staged position 0, were it digit d's
  __shared__ uint64_t scan[kTileWaves + 1];
  __shared__ uint32_t s_tile;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  if (tid == 0) s_tile = take_tile(a.state);
  // the keys of tile blockIdx.x, which mostly is the tile: loaded while the
  // counter's answer is on its way
  const int li0 = wave * (64 * ITEMS) + lane;  // key r of the lane: li0 + 64 * r
  uint64_t k[ITEMS];
  uint32_t v[ITEMS];
  int tile_n;
  const auto load = [&](int64_t t) {
    const int64_t base = t * kTile;
    tile_n = (int)(a.n - base < kTile ? a.n - base : kTile);
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
      const int li = li0 + 64 * r;
      k[r] = li < tile_n ? sort_key<RAW>(a.keys, a.src, base + li) : 0ull;
      if constexpr (RAW)
        v[r] = a.vals == nullptr ? (uint32_t)(base + li) : li < tile_n ? a.vals[base + li] : 0u;
      else
        v[r] = li < tile_n ? a.vals[base + li] : 0u;
    }
  };
  load(blockIdx.x);
  // the pass's total of digit tid % kBins, from every kAdders-th part
  constexpr int kAdders = kTileThreads / kBins;
  constexpr int kLoads = kCountGroups / kAdders;
  uint32_t total = 0;
  {
    uint32_t c[kLoads];
#pragma unroll
    for (int u = 0; u < kLoads; ++u) {
      const int w = u * kAdders + tid / kBins;
      c[u] = w < a.nparts ? a.parts[(int64_t)w * a.part_stride + (tid & (kBins - 1))] : 0u;
    }
#pragma unroll
    for (int u = 0; u < kLoads; ++u) total += c[u];
  }
  for (int d = tid; d < kTileWaves * kBins; d += kTileThreads) (&cnt[0][0])[d] = 0;
  sv[tid] = total;
  __syncthreads();
  if (tid < kBins) {
#pragma unroll
    for (int q = 1; q < kAdders; ++q) total += sv[q * kBins + tid];
  } else {
    total = 0;
  }
  const int64_t tile = s_tile;
  if (tile != blockIdx.x) load(tile);  // uniform
  // rank among the wave's keys of the same digit: earlier rounds, then lower lanes
  uint32_t rank[ITEMS];
#pragma unroll
  for (int r = 0; r < ITEMS; ++r)
    rank[r] = wave_digit_rank<RB>((uint32_t)(k[r] >> a.shift) & a.mask, li0 + 64 * r < tile_n, cnt[wave]);
  __syncthreads();
  uint64_t* const word = a.state + 1 + (tid < kBins ? tid : 0);
  uint32_t own = 0;
  if (tid < kBins) {
#pragma unroll
    for (int w = 0; w < kTileWaves; ++w) {
      const uint32_t c = cnt[w][tid];
      cnt[w][tid] = own;
      own += c;
    }
    store_state(word + tile * kMaxBins, (tile == 0 ? kStateBefore : kStateOwn) | own);
  }
  // exclusive sums over the digits: the tile's counts and the totals
  const uint32_t inc_own = wave_sum_scan(own), inc_total = wave_sum_scan(total);
  if (lane == 63) scan[wave] = ((uint64_t)inc_total << 32) | inc_own;
  __syncthreads();
  uint64_t ex = ((uint64_t)(inc_total - total) << 32) | (inc_own - own);
#pragma unroll
  for (int w = 0; w < kBins / 64; ++w)
    if (w < wave) ex += scan[w];
  if (tid < kBins) lstart[tid] = (uint32_t)ex;
  __syncthreads();
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    if (li0 + 64 * r < tile_n) {
      const uint32_t d = (uint32_t)(k[r] >> a.shift) & a.mask;
      const uint32_t pos = lstart[d] + cnt[wave][d] + rank[r];
      sk[pos] = k[r];
      sv[pos] = v[r];
    }
  }
  if (tid < kBins) {
    const uint64_t before = keys_before(word, tile, kMaxBins);
    if (tile > 0) store_state(word + tile * kMaxBins, kStateBefore | (before + own));
    gbase[tid] = (uint32_t)(ex >> 32) + (uint32_t)before - (uint32_t)ex;
  }
  __syncthreads();
  // the tile in digit order: runs of one digit go to consecutive positions
  for (int j = tid; j < tile_n; j += kTileThreads) {
    const uint64_t kk = sk[j];
    const uint32_t pos = gbase[(uint32_t)(kk >> a.shift) & a.mask] + (uint32_t)j;
    a.ko[pos] = kk;
    a.vo[pos] = sv[j];
  }
}

// OR over i of keys[i] ^ keys[0]: the bits where keys differ.  One atomic per
// workgroup at most, and none when the workgroup adds no new bit: thousands
// of atomics on one address serialize in one L2 channel.
__global__ __launch_bounds__(256) void key_span_kernel(const uint64_t* keys, int64_t n,
                                                       unsigned long long* out) {
  __shared__ uint64_t red[4];
  const uint64_t k0 = keys[0];
  uint64_t acc = 0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    acc |= keys[i] ^ k0;
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) acc |= __shfl_xor(acc, o);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    const uint64_t a = red[0] | red[1] | red[2] | red[3];
    const uint64_t seen = __hip_atomic_load(out, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (a & ~seen) atomicOr(out, (unsigned long long)a);
  }
}

// ---------------------------------------------------------------------------
size_t scan_temp_bytes(int64_t m) {
  // block sums of every level of the recursion, each level 256-byte aligned
  size_t bytes = 0;
  for (int64_t nb = (m + kScanBlock - 1) / kScanBlock; nb > 1; nb = (nb + kScanBlock - 1) / kScanBlock)
    bytes += ((size_t)nb * sizeof(uint32_t) + 255) / 256 * 256;
  return bytes;
}

namespace {
// Rounds of 64 keys per wave, and so the tile of a sweep (1,024 keys per round).
// Two rounds halve a tile's chain of ranking rounds and double the workgroups
// where 4,096-key tiles leave most CUs idle, but a tile walks back over twice as many
// others, and every tile adds up the counting workgroups' parts.  Dedup with two and
// with four rounds: 8,192 keys 45.1 and 51.0 us, 32,768 keys 51.0 and 56.8, 131,072
// keys 61.2 and 64.9, 200,000 keys 67.4 and 68.2, 262,144 keys 71.4 and 71.2 (a backprop
// of them 121.7 and 119.2), 300,000 keys 78.6 and 77.1, 400,000 keys 84.5 and 81.8,
// 1,000,000 keys 126.4 and 107.5: the line lies between 200,000 and 262,144, at 112
// tiles.  (One round up to 16,384 keys: within 0.3 us of two at 8,192 and 16,384 keys,
// 1.4 us less at 5,000.)
constexpr int64_t kTwoRoundKeys = 112 * 2048;
int tile_items(int64_t n) { return n <= kTwoRoundKeys ? 2 : 4; }
int64_t tiles_of(int64_t n) {
  const int64_t tile = kTileThreads * tile_items(n);
  return n > 0 ? (n + tile - 1) / tile : 1;
}
// The most tiles of any batch of at most n keys: storage sized for n serves them all.
int64_t most_tiles(int64_t n) { return std::max(tiles_of(n), tiles_of(std::min(n, kTwoRoundKeys))); }
int64_t pass_words(int64_t tiles) { return 1 + tiles * kMaxBins; }
// Past this many tiles (more than run at once, one on each CU) one launch adds the
// counts up.  With it and without: backprop of 600,000 keys (147 tiles) 149.9 and 146.2
// us, dedup of 700,000 keys 97.8 and 96.6, of 1,100,000 keys (269 tiles) 133.4 and
// 136.3, of 4,000,000 keys 292 and 300.
constexpr int64_t kMaxAddingTiles = 256;
}  // namespace

int64_t radix_span_parts(int64_t n) {
  const int64_t groups = n > 0 ? (n + kCountTile - 1) / kCountTile : 1;
  return groups < kCountGroups ? groups : kCountGroups;
}

size_t radix_sort_temp_bytes(int64_t n) {
  const size_t sort = (size_t)kMaxPasses * (size_t)pass_words(most_tiles(n)) * 8 +
                      (size_t)radix_span_parts(n) * kMaxPasses * kMaxBins * 4;
  const size_t scan = scan_temp_bytes(n);
  return sort > scan ? sort : scan;
}

hipError_t radix_sort_pairs(uint64_t* keys, uint32_t* vals, uint64_t* keys_alt, uint32_t* vals_alt,
                            int64_t n, int begin_bit, int end_bit, void* temp, int* result_in_alt,
                            hipStream_t stream, const RadixSource* src, uint64_t* clear, int64_t clear_words,
                            const PositionGrad* pg) {
  *result_in_alt = 0;
  if (n <= 1 || end_bit <= begin_bit) return src != nullptr ? hipErrorInvalidValue : hipSuccess;
  if (n > 0xffffffffLL || end_bit > 64) return hipErrorInvalidValue;  // values and counts of 32 bits
  const int64_t tiles = tiles_of(n);
  // 9-bit digits when they take fewer passes than 8-bit ones (26-bit keys: 3
  // passes instead of 4); the last digit keeps only the bits below end_bit
  const int width = end_bit - begin_bit;
  const int rb = (width + 8) / 9 < (width + 7) / 8 ? 9 : 8;
  RadixDigits dg{};
  for (int shift = begin_bit; shift < end_bit; shift += rb) {
    const int bits = end_bit - shift < rb ? end_bit - shift : rb;
    dg.shift[dg.passes] = shift;
    dg.mask[dg.passes] = (1u << bits) - 1u;
    ++dg.passes;
  }
  uint64_t* state = static_cast<uint64_t*>(temp);
  const int64_t words = pass_words(tiles);
  uint32_t* parts = reinterpret_cast<uint32_t*>(state + (int64_t)dg.passes * words);
  int nparts = (int)radix_span_parts(n);
  const int stride = dg.passes * kMaxBins;
  const RadixSource none{};
  const PositionGrad pooled = pg != nullptr && pg->mode != kBackpropConcat ? *pg : PositionGrad{};
  const int items = tile_items(n);
#define NVE_LAUNCH_COUNT(RAW, ITEMS, SRC)                                                                         \
  hipLaunchKernelGGL((radix_count_kernel<RAW, ITEMS>), dim3(nparts), dim3(kTileThreads), 0, stream, keys, SRC, n, \
                     dg, parts, state, dg.passes * words, clear, clear_words, pooled)
  if (src != nullptr) {
    if (items == 2) NVE_LAUNCH_COUNT(true, 2, *src); else NVE_LAUNCH_COUNT(true, 4, *src);
  } else {
    if (items == 2) NVE_LAUNCH_COUNT(false, 2, none); else NVE_LAUNCH_COUNT(false, 4, none);
  }
#undef NVE_LAUNCH_COUNT
  if (tiles > kMaxAddingTiles) {
    hipLaunchKernelGGL(radix_total_kernel, dim3((stride + 255) / 256), dim3(256), 0, stream, parts, nparts, stride);
    nparts = 1;
  }
  SweepArgs a{};
  a.keys = keys;
  a.vals = vals;
  a.ko = keys_alt;
  a.vo = vals_alt;
  a.n = n;
  a.nparts = nparts;
  a.part_stride = stride;
  for (int p = 0; p < dg.passes; ++p) {
    a.shift = dg.shift[p];
    a.mask = dg.mask[p];
    a.parts = parts + p * kMaxBins;
    a.state = state + p * words;
    const bool raw = src != nullptr && p == 0;
    a.src = raw ? *src : none;
    if (raw) a.vals = pooled.by_key != nullptr && weight_from_row(pooled.mode) ? pooled.by_key : nullptr;
    const dim3 grid((unsigned)tiles), block(kTileThreads);
    const auto sweep = [&](auto IT) {
      constexpr int kItems = decltype(IT)::value;
      if (rb == 9 && raw)
        hipLaunchKernelGGL((radix_sweep_kernel<9, true, kItems>), grid, block, 0, stream, a);
      else if (rb == 9)
        hipLaunchKernelGGL((radix_sweep_kernel<9, false, kItems>), grid, block, 0, stream, a);
      else if (raw)
        hipLaunchKernelGGL((radix_sweep_kernel<8, true, kItems>), grid, block, 0, stream, a);
      else
        hipLaunchKernelGGL((radix_sweep_kernel<8, false, kItems>), grid, block, 0, stream, a);
    };
    if (items == 2) sweep(std::integral_constant<int, 2>{});
    else sweep(std::integral_constant<int, 4>{});
    a.keys = p & 1 ? keys : keys_alt;
    a.vals = p & 1 ? vals : vals_alt;
    a.ko = p & 1 ? keys_alt : keys;
    a.vo = p & 1 ? vals_alt : vals;
    *result_in_alt ^= 1;
  }
  return hipGetLastError();
}

hipError_t exclusive_scan_u32(uint32_t* data, int64_t m, uint32_t* total, void* temp,
                              hipStream_t stream) {
  if (m <= 0) return hipSuccess;
  const int64_t nb = (m + kScanBlock - 1) / kScanBlock;
  if (nb > 0x7fffffff) return hipErrorInvalidValue;
  if (nb == 1) {
    hipLaunchKernelGGL(scan_down_kernel, dim3(1), dim3(kScanThreads), 0, stream, data, m,
                       (const uint32_t*)nullptr, total);
    return hipGetLastError();
  }
  uint32_t* sums = static_cast<uint32_t*>(temp);
  void* rest = static_cast<uint8_t*>(temp) + ((size_t)nb * sizeof(uint32_t) + 255) / 256 * 256;
  hipLaunchKernelGGL(scan_reduce_kernel, dim3(nb), dim3(kScanThreads), 0, stream, data, m, sums);
  hipError_t e = exclusive_scan_u32(sums, nb, nullptr, rest, stream);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(scan_down_kernel, dim3(nb), dim3(kScanThreads), 0, stream, data, m, sums,
                     total);
  return hipGetLastError();
}

hipError_t key_span(const uint64_t* keys, int64_t n, unsigned long long* out, hipStream_t stream) {
  if (n <= 0) return hipSuccess;
  int64_t grid = (n + 1023) / 1024;  // four keys per thread
  if (grid > 512) grid = 512;
  hipLaunchKernelGGL(key_span_kernel, dim3(grid), dim3(256), 0, stream, keys, n, out);
  return hipGetLastError();
}

}  // namespace nve_amd
