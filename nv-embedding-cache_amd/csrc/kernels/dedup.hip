// dedup.hip -- key deduplication on the GPU (Deduper::dedup, deduper.cuh:136-221)
// and the dedup-then-gather.
//
// dedup: stable radix sort of (key, position) -> runs of equal keys -> per
// run: unique key, start offset, count; per position: inverse = original
// position in key order.  The runs take one launch; a batch of at most
// kSmallDedupKeys keys is sorted and written by one workgroup in one launch.
// Outputs match the reference's: unique keys ascending (signed order), counts,
// the stable inverse map and exclusive offsets.
//
// dedup-then-gather needs no order, so it dedups by hashing instead of
// sorting (three launches): every distinct key of a workgroup claims a slot of
// an open-addressed table (linear probing, at most half full) with one
// compare-and-swap, the winner becoming the key's owner and its workgroup
// copying the key's table row to the owner's output row at once (each distinct
// row read once); with 32-bit keys a slot holds key and owner, so every claimant
// learns the owner at once; then every other position copies its owner's output
// row (UnpackDedup, cuda_utils.cuh:24-79).
#include "device_common.cuh"
#include "dedup_launch.hpp"
#include "lane_moves.cuh"
#include "position_grad.cuh"
#include "sort_launch.hpp"
#include "tile_rank.cuh"

namespace nve_amd {

// OR of x over the NT threads of the workgroup, in every thread (all threads call it)
template <int NT>
__device__ __forceinline__ uint64_t block_or(uint64_t x) {
  __shared__ uint64_t red[NT / 64];
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) x |= __shfl_xor(x, o);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = x;
  __syncthreads();
  uint64_t all = 0;
#pragma unroll
  for (int w = 0; w < NT / 64; ++w) all |= red[w];
  return all;
}

__global__ __launch_bounds__(256) void dedup_prep_kernel(const void* keys, int key_bytes, int64_t n,
                                                         int flip, uint64_t* k64, uint32_t* v) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    const int64_t k = load_key(keys, key_bytes, i);
    k64[i] = flip ? flip_key(k, key_bytes) : (uint64_t)k;
    v[i] = (uint32_t)i;
  }
}

// ---------------------------------------------------------------------------
// runs of the sorted keys, every output of the dedup in one launch: per position
// its inverse entry and unique index, per run its key and offset at the head
// and its count at the tail.  A 1024-thread workgroup per 4096 positions counts
// its run heads, publishes the count and its last head, and takes those of the
// tiles before by walking back over them, while the other waves already write
// their positions' gradient rows.  Bound: the latency of that chain, and the
// tile counter (one address: with 1024-key tiles 256 increments queued, 12.5 us
// for 262,144 keys, 9.7 with 4096).  Counting heads in a launch of its own and
// finding each position's bag here took 17.9 us.
// ---------------------------------------------------------------------------
constexpr int kRunThreads = 1024;
constexpr int kRunItems = 4;
constexpr int kRunBlock = kRunThreads * kRunItems;

// The runs of a workgroup's NT * ITEMS positions, position base + j * NT + tid
// in round j of thread tid, so that every load and store is of consecutive
// positions.  A wave's 64 positions of a round are a segment: its run heads
// are a ballot, its place the scan of the segments' head counts.
template <int NT, int ITEMS>
struct RunTile {
  static constexpr int kWaves = NT / 64;
  static constexpr int kSegs = ITEMS * kWaves;
  static_assert(kSegs <= 64, "one wave scans the segments");
  uint32_t seg_c[kSegs];  // heads of the tile before the segment
  int seg_l[kSegs];       // last head of the tile before it (-1: none)
  uint32_t sum;           // heads of the tile
  int max;                // its last head (-1: none)
};

// heads[j] = the wave's run heads of round j; t: filled for the whole
// workgroup (every thread calls it; key_at(i) is read for i in [0, n)).
template <int NT, int ITEMS, typename K>
__device__ __forceinline__ void find_runs(RunTile<NT, ITEMS>& t, const K& key_at, int64_t base, int64_t n,
                                          uint64_t (&heads)[ITEMS]) {
  constexpr int kSegs = RunTile<NT, ITEMS>::kSegs;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) {
    const int64_t i = base + j * NT + tid;
    heads[j] = __ballot(i < n && (i == 0 || key_at(i) != key_at(i - 1)));
    const int seg = j * (NT / 64) + wave;
    if (lane == 0) {
      t.seg_c[seg] = (uint32_t)__popcll(heads[j]);
      t.seg_l[seg] = heads[j] ? j * NT + wave * 64 + 63 - __builtin_clzll(heads[j]) : -1;
    }
  }
  __syncthreads();
  if (tid < 64) {
    const uint32_t c = tid < kSegs ? t.seg_c[tid] : 0u;
    int l = tid < kSegs ? t.seg_l[tid] : -1;
    const uint32_t inc = wave_sum_scan(c);
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int p = __shfl_up(l, o);
      if (lane >= o) l = p > l ? p : l;
    }
    const int before = __shfl_up(l, 1);
    if (tid < kSegs) {
      t.seg_c[tid] = inc - c;
      t.seg_l[tid] = lane > 0 ? before : -1;
    }
    if (tid == 63) {
      t.sum = inc;
      t.max = l;
    }
  }
  __syncthreads();
}

// The outputs of the tile: u0 heads before it, h0 the last of them.
template <int NT, int ITEMS, typename K>
__device__ __forceinline__ void emit_runs(const RunTile<NT, ITEMS>& t, const K& key_at, const DedupOut& o,
                                          const uint64_t (&heads)[ITEMS], const uint32_t (&pos)[ITEMS], int64_t base,
                                          int64_t n, uint32_t u0, int64_t h0) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint64_t upto = ~0ull >> (63 - lane);
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) {
    const int64_t i = base + j * NT + tid;
    if (i >= n) continue;
    const int seg = j * (NT / 64) + wave;
    const uint64_t m = heads[j] & upto;
    const uint32_t u = u0 + t.seg_c[seg] + (uint32_t)__popcll(m) - 1u;
    const uint64_t key = key_at(i);
    if ((heads[j] >> lane) & 1u) {
      store_key(o.unique, o.key_bytes, u, unflip_key(key, o.key_bytes));
      store_key(o.offsets, o.key_bytes, u, i);
    }
    if (o.inverse != nullptr) store_key(o.inverse, o.key_bytes, i, (int64_t)pos[j]);
    if (o.pos_key != nullptr) o.pos_key[i] = u;
    if (i == n - 1 || key != key_at(i + 1)) {  // the run ends here
      const int64_t start = m ? base + j * NT + wave * 64 + 63 - __builtin_clzll(m)
                              : (t.seg_l[seg] >= 0 ? base + t.seg_l[seg] : h0);
      store_key(o.counts, o.key_bytes, u, i + 1 - start);
    }
  }
}

// The unique count and the keys' span to the head in device memory and, where
// given, to its copy in pinned host memory.
__device__ __forceinline__ void write_total(const DedupOut& o, uint32_t total) {
  o.head->total = total;
  if (o.host_head != nullptr) o.host_head->total = total;
}
__device__ __forceinline__ void write_span(const DedupOut& o, unsigned long long span) {
  o.head->span = span;
  if (o.host_head != nullptr) o.host_head->span = span;
}

struct RunArgs {
  const uint64_t* ks;
  const uint32_t* vs;
  int64_t n;
  const uint64_t* span_part;  // null: no span to check
  int64_t nparts;
  uint64_t* state;  // tile counter, then per tile its head count and its last head + 1
  bool carried;     // vs holds gradient rows
  DedupOut out;
};

__global__ __launch_bounds__(kRunThreads) void run_outputs_kernel(RunArgs a) {
  __shared__ uint32_t s_tile, s_u0;
  __shared__ int64_t s_h0;
  const int tid = threadIdx.x;
  if (tid == 0) s_tile = take_tile(a.state);
  __syncthreads();
  const int64_t tile = s_tile;
  if (tile == 0) {  // uniform over the workgroup
    uint64_t x = 0;
    if (a.span_part != nullptr)
      for (int64_t j = tid; j < a.nparts; j += kRunThreads) x |= a.span_part[j];
    x = block_or<kRunThreads>(x);
    if (tid == 0) write_span(a.out, x);
  }
  const int64_t base = tile * kRunBlock;
  const auto key_at = [&](int64_t i) { return a.ks[i]; };
  uint32_t pos[kRunItems];
#pragma unroll
  for (int j = 0; j < kRunItems; ++j) {
    const int64_t i = base + j * kRunThreads + tid;
    pos[j] = i < a.n ? a.vs[i] : 0;
  }
  __shared__ RunTile<kRunThreads, kRunItems> runs;
  uint64_t run_heads[kRunItems];
  find_runs<kRunThreads, kRunItems>(runs, key_at, base, a.n, run_heads);
  const uint32_t sum = runs.sum;
  const uint64_t max1 = runs.max >= 0 ? (uint64_t)(base + runs.max + 1) : 0;  // last head + 1, 0: none
  if (tid < 64) {
    // publish, then the tiles before: the sum of their head counts and the
    // nearest one's last head, 64 of them at a time.  Every one of them has
    // started and publishes without waiting for another, so each wait ends.
    uint64_t* const word = a.state + 1 + 2 * tile;
    if (tid < 2) store_state(word + tid, (tile == 0 ? kStateBefore : kStateOwn) | (tid == 0 ? sum : max1));
    uint64_t heads = 0, last = 0;  // last head + 1, 0: none
    bool open_c = tile > 0, open_l = tile > 0;  // uniform over the wave
    for (int64_t top = tile - 1; top >= 0 && (open_c || open_l); top -= 64) {
      const int64_t t = top - tid;
      uint64_t wc = kStateBefore, wl = kStateBefore;  // before the first tile: nothing
      if (t >= 0) {
        do {
          wc = load_state(a.state + 1 + 2 * t);
          wl = load_state(a.state + 2 + 2 * t);
        } while (wc < kStateOwn || wl < kStateOwn);
      }
      if (open_c) {
        const uint64_t closed = __ballot(wc >= kStateBefore);
        const int end = closed ? __builtin_ctzll(closed) : 63;  // the last lane to add
        uint32_t v = tid <= end ? (uint32_t)(wc & kStateCount) : 0u;  // heads fit 32 bits
        v = wave_sum_scan(v);
        heads += (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
        open_c = closed == 0;
      }
      if (open_l) {
        const uint64_t known = __ballot(wl >= kStateBefore || (wl & kStateCount) != 0);
        if (known) {
          last = __shfl(wl, __builtin_ctzll(known)) & kStateCount;
          open_l = false;
        }
      }
    }
    if (tid == 0) {
      s_u0 = (uint32_t)heads;
      s_h0 = (int64_t)last - 1;
      if (tile > 0) {
        store_state(word, kStateBefore | (heads + sum));
        store_state(word + 1, kStateBefore | (max1 ? max1 : last));
      }
      if (tile == gridDim.x - 1) write_total(a.out, (uint32_t)heads + sum);
    }
  }
  if (a.out.pg.rows != nullptr) {
    const auto row_at = [&](uint32_t p) { return a.out.pg.by_key[p]; };
    position_grads<kRunItems>(a.out.pg, a.carried, row_at, base + tid, kRunThreads, a.n, pos);
  }
  __syncthreads();
  emit_runs<kRunThreads, kRunItems>(runs, key_at, a.out, run_heads, pos, base, a.n, s_u0, s_h0);
}

// ---------------------------------------------------------------------------
// The whole dedup of a small batch (at most 1024 * ITEMS keys) in one workgroup
// and one launch: the keys stay in LDS between the passes, and the passes cover
// exactly the bits in which the keys differ, so nothing is assumed about them.
// Bound: the latency of one workgroup's passes; the sort and the runs took six
// launches (dedup of 500 keys 58.8 -> 19.0 us, 2,000 keys 58.2 -> 25.7, 4,096 keys 59.3 ->
// 28.3; one workgroup of 8,192 keys took as long as the radix sort, 50 us).
// ---------------------------------------------------------------------------
template <int ITEMS>
__global__ __launch_bounds__(1024) void dedup_small_kernel(const void* keys, int n, DedupOut o) {
  constexpr int RB = 9;  // as the radix sort: three passes for the keys of tables of up to 2^27 rows
  constexpr int kBins = 1 << RB;
  constexpr int kWaves = 16;
  __shared__ uint64_t sk[1024 * ITEMS];
  __shared__ uint32_t sv[1024 * ITEMS];
  __shared__ uint32_t rows[1024 * ITEMS];
  __shared__ uint32_t cnt[kWaves][kBins];
  __shared__ uint32_t lstart[kBins];
  __shared__ uint32_t wsum[kBins / 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int li0 = wave * (64 * ITEMS) + lane;  // key r of the lane: li0 + 64 * r
  uint64_t k[ITEMS];
  uint32_t v[ITEMS];
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const int li = li0 + 64 * r;
    k[r] = flip_key(load_key(keys, o.key_bytes, li < n ? li : 0), o.key_bytes);
    v[r] = (uint32_t)li;
  }
  // pooled gradients: the row of every key position; values: rows where they do
  const bool pooled = o.pg.rows != nullptr && o.pg.mode != kBackpropConcat;  // uniform
  const bool carried = pooled && weight_from_row(o.pg.mode);
  if (pooled) {
    tile_rows<1024, 1024 * ITEMS>(o.pg, 0, rows);
    if (carried) {
#pragma unroll
      for (int r = 0; r < ITEMS; ++r) v[r] = rows[li0 + 64 * r];
    }
  }
  // the bits in which the keys differ (a lane past the end holds key 0)
  uint64_t diff = 0;
  const uint64_t k0 = flip_key(load_key(keys, o.key_bytes, 0), o.key_bytes);
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) diff |= k[r] ^ k0;
  const uint64_t span = block_or<1024>(diff);
  const int bits = span ? 64 - __builtin_clzll(span) : 0;

  int shift = 0;
  do {  // at least once, which lays the keys out in LDS
    for (int d = tid; d < kWaves * kBins; d += 1024) (&cnt[0][0])[d] = 0;
    __syncthreads();
    uint32_t rank[ITEMS];
#pragma unroll
    for (int r = 0; r < ITEMS; ++r)
      rank[r] = wave_digit_rank<RB>((uint32_t)(k[r] >> shift) & (kBins - 1), li0 + 64 * r < n, cnt[wave]);
    __syncthreads();
    uint32_t own = 0, inc = 0;
    if (tid < kBins) {
#pragma unroll
      for (int w = 0; w < kWaves; ++w) {
        const uint32_t c = cnt[w][tid];
        cnt[w][tid] = own;
        own += c;
      }
      inc = wave_sum_scan(own);
      if (lane == 63) wsum[wave] = inc;
    }
    __syncthreads();
    if (tid < kBins) {
      uint32_t ex = inc - own;
#pragma unroll
      for (int w = 0; w < kBins / 64; ++w)
        if (w < wave) ex += wsum[w];
      lstart[tid] = ex;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
      if (li0 + 64 * r < n) {
        const uint32_t d = (uint32_t)(k[r] >> shift) & (kBins - 1);
        const uint32_t at = lstart[d] + cnt[wave][d] + rank[r];
        sk[at] = k[r];
        sv[at] = v[r];
      }
    }
    __syncthreads();
    shift += RB;
    if (shift < bits) {
#pragma unroll
      for (int r = 0; r < ITEMS; ++r) {
        const int li = li0 + 64 * r;
        if (li < n) {
          k[r] = sk[li];
          v[r] = sv[li];
        }
      }
    }
  } while (shift < bits);

  const auto key_at = [&](int64_t i) { return sk[i]; };
  uint32_t pos[ITEMS];
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) {
    const int i = j * 1024 + tid;
    pos[j] = i < n ? sv[i] : 0;
  }
  __shared__ RunTile<1024, ITEMS> runs;
  uint64_t run_heads[ITEMS];
  find_runs<1024, ITEMS>(runs, key_at, 0, n, run_heads);
  if (tid == 0) {
    write_total(o, runs.sum);
    write_span(o, 0);
  }
  if (o.pg.rows != nullptr) {
    const auto row_at = [&](uint32_t p) { return rows[p]; };
    position_grads<ITEMS>(o.pg, carried, row_at, tid, 1024, n, pos);
  }
  emit_runs<1024, ITEMS>(runs, key_at, o, run_heads, pos, 0, n, 0u, -1);
}

// ---------------------------------------------------------------------------
// hash dedup for the gather
// ---------------------------------------------------------------------------
constexpr uint32_t kNoSlot = 0xffffffffu;

// Table keys are 32-bit when every row index fits (num_rows < 2^32), else
// 64-bit; all ones marks an empty slot (no row index has that value).
template <typename KT>
constexpr KT empty_slot() {
  return (KT)~(KT)0;
}

// the table's keys to empty
template <typename KT>
__global__ __launch_bounds__(256) void hash_clear_kernel(KT* tab, int64_t slots) {
  constexpr int64_t per = 16 / sizeof(KT);  // slots per 16-byte store
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if ((i + 1) * per <= slots) {
    u32x4 e{0xffffffffu, 0xffffffffu, 0xffffffffu, 0xffffffffu};
    reinterpret_cast<u32x4*>(tab)[i] = e;
  } else {
    for (int64_t j = i * per; j < slots; ++j) tab[j] = empty_slot<KT>();
  }
}

// Multiplicative (Fibonacci) hash to `bits` bits.
__device__ __forceinline__ uint32_t slot_hash(uint64_t k, int bits) {
  return (uint32_t)((k * 0x9E3779B97F4A7C15ull) >> (64 - bits));
}

__device__ __forceinline__ uint32_t cas(uint32_t* p, uint32_t expect, uint32_t v) {
  return atomicCAS(p, expect, v);
}
__device__ __forceinline__ uint64_t cas(uint64_t* p, uint64_t expect, uint64_t v) {
  return (uint64_t)atomicCAS(reinterpret_cast<unsigned long long*>(p), (unsigned long long)expect,
                             (unsigned long long)v);
}

// Claim key k's slot of a table of 2^bits slots (linear probing; the caller
// guarantees a free slot).  Returns the slot; *won: this call put k there.
// A slot only changes from empty to a key, so the compare-and-swap's answer
// is final.
template <typename KT>
__device__ __forceinline__ uint32_t claim(KT* tab, KT k, int bits, bool* won) {
  const uint32_t mask = (1u << bits) - 1u;
  uint32_t h = slot_hash(k, bits);
  for (;;) {
    const KT cur = cas(tab + h, empty_slot<KT>(), k);
    if (cur == empty_slot<KT>() || cur == k) {
      *won = cur == empty_slot<KT>();
      return h;
    }
    h = (h + 1) & mask;
  }
}

struct HashClaim {
  const void* keys;
  int key_bytes;
  int64_t n;
  uint64_t num_rows;
  void* tab;
  int bits;
  uint32_t* owner;    // owner[slot]: position that owns the slot's key
  uint32_t* slot_of;  // slot_of[i]: slot of position i's key (kNoSlot: out of range)
  const uint8_t* table;
  uint64_t row_bytes;
  uint8_t* out;
  int64_t out_stride;
  int g_shift;  // 2^g_shift lanes move one row
  int passes;   // row pieces of 2^g_shift * VB bytes
};

// Claim 32-bit key k for position pos in a table of 2^bits 64-bit slots
// holding key << 32 | owner position (all ones: empty), so that a loser of
// the compare-and-swap learns the owner from its answer.  Returns the owner;
// *won: pos became it.
__device__ __forceinline__ uint32_t claim_owner(uint64_t* tab, uint32_t k, uint32_t pos, int bits,
                                                bool* won) {
  const uint32_t mask = (1u << bits) - 1u;
  const uint64_t mine = ((uint64_t)k << 32) | pos;
  uint32_t h = slot_hash(k, bits);
  for (;;) {
    const uint64_t cur = cas(tab + h, ~0ull, mine);
    if (cur == ~0ull) {
      *won = true;
      return pos;
    }
    if ((uint32_t)(cur >> 32) == k) {
      *won = false;
      return (uint32_t)cur;
    }
    h = (h + 1) & mask;
  }
}

constexpr int kClaimThreads = 1024;  // one key per thread
constexpr int kLocalBits = 11;       // 2048 LDS slots per workgroup, at most half full

// The claims and the owners' copies in one launch.  Each workgroup first
// dedups its 1024 keys in an LDS table, so a key claims its global slot once
// per workgroup rather than once per occurrence (device-scope
// compare-and-swaps on one hot key's slot serialize at the memory side).  The
// global winner of a slot owns the key: it records itself in owner[slot], and
// its workgroup then copies the key's table row to the owner's output row --
// each distinct row is read once.  Rows move as in the plain gather:
// 2^g_shift lanes per row, U rows in flight per lane group, every load of a
// round issued before any store.  Measured on 262,144 Zipf(1.05) keys, this
// launch and the repeats' take 39 us where separate claim, owner-list and
// owner-copy launches took 48; chunks of 512 or 2048 keys per workgroup were
// slower (41 and 42 us), and so was reading a slot before its
// compare-and-swap (43 us: the workgroups reach the hot keys' slots together).
// Packing key and owner into one slot (32-bit keys) then let the repeats read
// each position's owner directly (39.6 -> 37.5 us), and copying each wave's
// wins without waiting for the other waves' claims gave 36.1 us.
// PACKED (32-bit keys): the table holds key and owner together and slot_of
// receives each position's owner; otherwise the table holds keys, owner[]
// the owner of each slot and slot_of each position's slot.
template <typename KT, int VB, int U, bool PACKED>
__global__ __launch_bounds__(kClaimThreads) void hash_claim_copy_kernel(HashClaim a) {
  static_assert(!PACKED || sizeof(KT) == 4, "packed slots hold 32-bit keys");
  __shared__ KT lkey[1 << kLocalBits];
  __shared__ uint32_t lslot[1 << kLocalBits];  // global slot (PACKED: owner) of the local entry
  __shared__ uint64_t win_row[kClaimThreads];  // each wave's wins (64 entries a wave): table row
  __shared__ uint32_t win_pos[kClaimThreads];  // ... and output row
  const int tid = threadIdx.x;
  // the key load is issued before the LDS table is cleared
  const int64_t i = (int64_t)blockIdx.x * kClaimThreads + tid;
  bool in = false;
  KT k = 0;
  if (i < a.n) {
    const uint64_t k64 = (uint64_t)load_key(a.keys, a.key_bytes, i);
    in = k64 < a.num_rows;  // keys outside the table get no slot and no output row
    k = (KT)k64;
  }
  for (int j = tid; j < (1 << kLocalBits); j += kClaimThreads) lkey[j] = empty_slot<KT>();
  __syncthreads();
  uint32_t ls = 0;
  bool first = false;
  if (in) ls = claim<KT>(lkey, k, kLocalBits, &first);
  __syncthreads();
  bool won = false;
  if (first) {
    if constexpr (PACKED) {
      lslot[ls] = claim_owner(static_cast<uint64_t*>(a.tab), (uint32_t)k, (uint32_t)i, a.bits, &won);
    } else {
      const uint32_t gs = claim<KT>(static_cast<KT*>(a.tab), k, a.bits, &won);
      lslot[ls] = gs;
      if (won) a.owner[gs] = (uint32_t)i;
    }
  }
  // each wave lists the keys it won in its own LDS region and copies their
  // rows at once, without waiting for the other waves' claims
  const uint64_t ballot = __ballot(won);
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const uint32_t below = (uint32_t)__popcll(ballot & (lane == 0 ? 0ull : (~0ull >> (64 - lane))));
  const int nw = (int)__popcll(ballot);
  uint64_t* wrow = win_row + wave * 64;
  uint32_t* wpos = win_pos + wave * 64;
  if (won) {
    wrow[below] = (uint64_t)k;
    wpos[below] = (uint32_t)i;
  }
  // lanes read what other lanes of the wave wrote: LDS keeps a wave's
  // accesses in order; the fences keep the compiler from moving them
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  const int G = 1 << a.g_shift;
  const int gl = lane & (G - 1);
  const int grp = lane >> a.g_shift;
  const int groups = 64 >> a.g_shift;
  const uint64_t zero_row = (uint64_t)g_zero_row;
  for (int p = 0; p < a.passes; ++p) {
    const int64_t off = ((int64_t)p * G + gl) * VB;
    const bool in_row = off < (int64_t)a.row_bytes;
    for (int q0 = 0; q0 < nw; q0 += groups * U) {
      uint64_t src[U];
      uint32_t dst[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int q = q0 + u * groups + grp;
        const bool real = q < nw && in_row;
        src[u] = real ? (uint64_t)a.table + wrow[q] * a.row_bytes + off : zero_row + (off & kZeroRowMask);
        dst[u] = real ? wpos[q] : kNoSlot;
      }
      Vec<VB> v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) v[u] = load_vec<VB>(src[u]);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (dst[u] == kNoSlot) continue;
        store_vec<VB, false>(a.out + (int64_t)dst[u] * a.out_stride + off, v[u]);
      }
    }
  }
  __syncthreads();  // every local entry's owner (or slot) is in LDS
  if (i < a.n) a.slot_of[i] = in ? lslot[ls] : kNoSlot;
}

// Every position that does not own its key copies its owner's output row
// (written by the claims' launch).  A wave resolves T positions (one per
// lane), then groups of G lanes move one row each, U rows in flight, VB
// bytes per lane and load.
struct HashRepeat {
  int64_t n;
  uint64_t row_bytes;
  const uint32_t* slot_of;
  const uint32_t* owner;
  uint8_t* out;
  int64_t out_stride;
};

template <int VB, int U, bool PACKED>
__global__ __launch_bounds__(256) void hash_repeat_kernel(HashRepeat a, int g_shift, int t_shift, int passes) {
  const int T = 1 << t_shift;
  const int lane = threadIdx.x & 63;
  const int64_t tile = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const int64_t base = tile << t_shift;
  if (base >= a.n) return;  // whole wave past the end
  const int64_t j = base + lane;
  uint64_t src = 0;  // row to copy from, 0: nothing to do for this lane's position
  if (lane < T && j < a.n) {
    const uint32_t sl = a.slot_of[j];
    if (sl != kNoSlot) {
      const uint32_t own = PACKED ? sl : a.owner[sl];
      if (own != (uint32_t)j) src = (uint64_t)a.out + (uint64_t)own * (uint64_t)a.out_stride;
    }
  }
  const uint32_t dst = (uint32_t)j;
  const int G = 1 << g_shift;
  const int gl = lane & (G - 1);
  const int grp = lane >> g_shift;
  const int groups = 64 >> g_shift;
  const int per_group = T >> (6 - g_shift) > 0 ? T >> (6 - g_shift) : 1;
  const uint64_t zero_row = (uint64_t)g_zero_row;
  for (int p = 0; p < passes; ++p) {
    const int64_t off = ((int64_t)p * G + gl) * VB;
    const bool in_row = off < (int64_t)a.row_bytes;
    for (int q0 = 0; q0 < per_group; q0 += U) {
      uint64_t ra[U];
      uint32_t rd[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int q = q0 + u;
        const int from = grp + (q < per_group ? q : 0) * groups;
        ra[u] = shfl64(src, from);
        rd[u] = shfl32(dst, from);
        if (q >= per_group) ra[u] = 0;
      }
      Vec<VB> v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const bool real = ra[u] != 0;
        v[u] = load_vec<VB>((real ? ra[u] : zero_row) + ((real && in_row) ? off : (off & kZeroRowMask)));
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (ra[u] == 0 || !in_row) continue;
        store_vec<VB>(a.out + (int64_t)rd[u] * a.out_stride + off, v[u]);
      }
    }
  }
}

size_t hash_dedup_slots(int64_t n) {
  size_t s = 1024;
  while (s < 2 * (size_t)n) s <<= 1;
  return s;
}

size_t hash_dedup_key_bytes(int64_t num_rows) { return (uint64_t)num_rows <= 0xffffffffull ? 4 : 8; }

hipError_t launch_hash_dedup_gather(const void* keys, int key_bytes, int64_t n, const uint8_t* table,
                                    int64_t num_rows, int64_t row_bytes, void* out, int64_t out_stride,
                                    void* tab, uint32_t* owner, uint32_t* slot_of, hipStream_t stream) {
  if (n <= 0) return hipSuccess;
  const int64_t slots = (int64_t)hash_dedup_slots(n);
  int bits = 0;
  while ((1ll << bits) < slots) ++bits;
  const bool k32 = hash_dedup_key_bytes(num_rows) == 4;
  // widest vector every row, output row and base is aligned to
  int vb = 16;
  while (vb > 1 && (row_bytes % vb || out_stride % vb || (uintptr_t)table % vb || (uintptr_t)out % vb))
    vb >>= 1;
  const int64_t nv = row_bytes / vb;
  int g = 1;
  while (g < nv && g < 64) g <<= 1;
  const int passes = (int)((nv + g - 1) / g);
  int gs = 0;
  while ((1 << gs) < g) ++gs;
  constexpr int U = 8;
  const int tkeys = (64 / g) * U < 64 ? (64 / g) * U : 64;
  int ts = 0;
  while ((1 << ts) < tkeys) ++ts;
  const int64_t waves = (n + tkeys - 1) / tkeys;
  const int64_t grid = (waves * 64 + 255) / 256;
  if (grid > 0x7fffffffLL) return hipErrorInvalidValue;
  const dim3 claim_grid((unsigned)((n + kClaimThreads - 1) / kClaimThreads));
  HashClaim c{keys, key_bytes, n, (uint64_t)num_rows, tab, bits, owner, slot_of, table, (uint64_t)row_bytes,
              static_cast<uint8_t*>(out), out_stride, gs, passes};
  HashRepeat r{n, (uint64_t)row_bytes, slot_of, owner, static_cast<uint8_t*>(out), out_stride};
  // 64-bit slots either way: 32-bit keys packed with their owner, or 64-bit keys
  hipLaunchKernelGGL(hash_clear_kernel<uint64_t>, dim3((slots / 2 + 255) / 256), dim3(256), 0, stream,
                     static_cast<uint64_t*>(tab), slots);
#define HC(V)                                                                                           \
  do {                                                                                                  \
    if (k32) {                                                                                          \
      hipLaunchKernelGGL((hash_claim_copy_kernel<uint32_t, V, U, true>), claim_grid,                    \
                         dim3(kClaimThreads), 0, stream, c);                                            \
      hipLaunchKernelGGL((hash_repeat_kernel<V, U, true>), dim3(grid), dim3(256), 0, stream, r, gs, ts, \
                         passes);                                                                       \
    } else {                                                                                            \
      hipLaunchKernelGGL((hash_claim_copy_kernel<uint64_t, V, U, false>), claim_grid,                   \
                         dim3(kClaimThreads), 0, stream, c);                                            \
      hipLaunchKernelGGL((hash_repeat_kernel<V, U, false>), dim3(grid), dim3(256), 0, stream, r, gs,    \
                         ts, passes);                                                                   \
    }                                                                                                   \
  } while (0)
  switch (vb) {
    case 16: HC(16); break;
    case 8: HC(8); break;
    case 4: HC(4); break;
    case 2: HC(2); break;
    default: HC(1); break;
  }
#undef HC
  return hipGetLastError();
}

int64_t dedup_span_parts(int64_t n) { return radix_span_parts(n); }

bool carries_rows(int mode) { return mode != kBackpropConcat && weight_from_row(mode); }

hipError_t launch_dedup_prep(const void* keys, int key_bytes, int64_t n, int flip, uint64_t* k64,
                             uint32_t* v, hipStream_t stream) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(dedup_prep_kernel, dim3((n + 255) / 256), dim3(256), 0, stream, keys, key_bytes,
                     n, flip, k64, v);
  return hipGetLastError();
}

int64_t run_state_words(int64_t n) { return 1 + 2 * ((n + kRunBlock - 1) / kRunBlock); }

hipError_t launch_dedup_runs(const uint64_t* ks, const uint32_t* vs, int64_t n, const uint64_t* span_part,
                             uint64_t* state, bool carried, const DedupOut& out, hipStream_t stream) {
  if (n <= 0) return hipSuccess;
  const RunArgs a{ks, vs, n, span_part, dedup_span_parts(n), state, carried, out};
  hipLaunchKernelGGL(run_outputs_kernel, dim3((unsigned)((n + kRunBlock - 1) / kRunBlock)), dim3(kRunThreads), 0,
                     stream, a);
  return hipGetLastError();
}

hipError_t launch_dedup_small(const void* keys, int64_t n, const DedupOut& out, hipStream_t stream) {
  if (n <= 0) return hipSuccess;
  if (n > kSmallDedupKeys) return hipErrorInvalidValue;
  if (n <= 1024)
    hipLaunchKernelGGL(dedup_small_kernel<1>, dim3(1), dim3(1024), 0, stream, keys, (int)n, out);
  else
    hipLaunchKernelGGL(dedup_small_kernel<4>, dim3(1), dim3(1024), 0, stream, keys, (int)n, out);
  return hipGetLastError();
}

}  // namespace nve_amd
