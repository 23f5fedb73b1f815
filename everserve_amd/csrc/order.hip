// A restore's (slot, staged row) pairs in slot order, on the device: the ordering that lets the
// pair scatter (evs_scatter_pairs in rows.hip) write each layer's cache front to back, for a
// caller whose slot list is already in HBM. The pairs are sorted on the low key_bits bits of the
// slot ids (the cache's slot count fixes how many matter: 18 for 262,144 slots). The sort is
// stable, so equal slots keep their listed order. Everything it needs beyond its inputs and
// outputs lives in a workspace the caller allocates.
//
// Up to 2^20 pairs it is the radix sort below. What bounds it there is not the data (6 MB at
// 262,144 pairs, 1 us) but the chain of dependent launches and memory round trips, so a pass sorts
// 9 bits (18-bit slot ids take two) and is two launches: each workgroup counts its tile's digits,
// then each ranks its own tile and adds up the other tiles' counts by itself, with no scan kernel
// between. Counts are 16 bits, so that one wave reads a tile's 512 of them in one instruction. The
// launches are those of key_bits; how many passes the ids really need is found on the device (the
// first count also ORs the ids), and the launches past that return at once. 8,192 pairs and fewer
// are one launch of one workgroup. Microseconds a call, against rocPRIM's radix sort, which took
// every size before (a merge sort of many launches below about 2^20 pairs), 18 key bits: 1,500
// pairs 12.0 and 23.4 (a call that sorts one pair: 12.0 and 15.5), 16,384 21.2 and 28.6, 65,536
// 22.4 and 44.4, 262,144 29.8 and 106.4 (32 bits: 37.0 and 107.9); 21 bits, 1,048,576 pairs: 75
// and 191.
// Above 2^20 pairs rocPRIM's radix sort is used (2,097,152 pairs of 21 bits: 120 us, 197 here):
// every workgroup adds up every tile's counts, work that grows with the square of the tiles. So it
// is for a few sizes below (see kMergedFirst). Left slower here than there: ids that need all four
// passes of a 32-bit key, up to 36,000 pairs (32,768 pairs 43.4 and 40.9 us), and more passes, up
// to 200,000 (64 bits 103 and 80); padding ids need every pass of their key. rocPRIM clears its
// counters in the workspace with hipMemsetAsync, so this call is not one to capture in a HIP graph.
//
// evs_order_pairs_static is the same call for callers that cannot allocate (no workspace
// argument): its scratch is a file-scope device array of a fixed size.

#include <mutex>

#include <rocprim/device/device_radix_sort.hpp>

#include "common.hpp"

namespace evs {
namespace {

constexpr int kIotaThreads = 256;
constexpr int64_t kAlign = 256;

// The radix sort of up to kMaxSorted pairs.
constexpr int kDigitBits = 9;
constexpr int kBins = 1 << kDigitBits;
constexpr int kSortThreads = 512;  // one a bin
constexpr int kWaves = kSortThreads / 64;
constexpr int kMaxTiles = 256;  // tiles a sort has at most: one thread a tile ORs their ids
static_assert(kSortThreads == kBins && kMaxTiles <= kSortThreads, "one thread a bin, one a tile");
constexpr int64_t kMaxSorted = int64_t{1} << 20;

// A tile: kSortThreads x R pairs, wave w's the R runs of 64 from w * R * 64 on. R is 4 up to 2^19
// pairs and 8 above, so that a sort has at most kMaxTiles tiles: 1,048,576 pairs of 21 bits took
// 75 us in 256 tiles and 84 in 128, 262,144 30 us in 128 tiles and 35 in 64.
constexpr int64_t tile_pairs(int r) { return int64_t{kSortThreads} * r; }
int rounds_of(int64_t n) { return n <= kMaxTiles * tile_pairs(4) ? 4 : 8; }
static_assert(kMaxTiles * tile_pairs(8) >= kMaxSorted && tile_pairs(8) < 65536,
              "a tile's counts are 16 bits");
// Up to this many pairs one workgroup sorts them all in one launch: 5,000 in 16.5 us, 19.1 in four
// launches (18 bits). kHalfTile and fewer take half its rounds (2,049 pairs of 18 bits 10.6 and 15.0
// us, 4,000 of 20 bits 14.9 and 20.6), kQuarterTile and fewer half the waves too.
constexpr int64_t kOneTile = 8192;
constexpr int64_t kHalfTile = 4096;
constexpr int64_t kQuarterTile = 2048;
// From kOneTile to this many pairs, keys of three passes and more take rocPRIM's sort, which merges
// once less often than above: 8,193 and 16,384 pairs of 20 bits 27.4 and 29.1 us (31.0 and 31.8
// here), of 32 bits 29.5 and 30.1, here 28.1 and 28.9 for ids of 18 bits and 41.5 and 42.7 with
// padding among them; 20,000 pairs of 20 bits 38.3 (32.0).
constexpr int64_t kMergedFirst = 16384;
// A workspace that holds that sort's, for every larger call of such keys too.
constexpr int64_t kMergedBytes = int64_t{512} << 10;

struct SortArgs {
  const int64_t* slots;  // the ids as given
  int64_t* out_keys;
  int64_t* out_rows;
  int64_t* tmp_keys;     // the workspace's pairs
  int64_t* tmp_rows;
  uint16_t* counts;      // [tiles][kBins]: how many of a tile's pairs have each digit
  uint64_t* ors;         // [tiles]: a tile's ids ORed together
  uint64_t key_mask;
  int64_t n;
  int tiles;
  int even;              // an output overlaps the ids: the first pass must not write there
};

// The passes the ids need: one at least, and an even number where the first pass may only write
// the workspace. `bits`: every id ORed together.
__device__ __forceinline__ int passes_of(uint64_t bits, int even) {
  const int significant = bits == 0 ? 0 : 64 - __builtin_clzll(bits);
  int p = (significant + kDigitBits - 1) / kDigitBits;
  p = p < 1 ? 1 : p;
  return even ? (p + 1) / 2 * 2 : p;
}

// Every tile's ids ORed together, the same in every thread. All threads call it.
__device__ __forceinline__ uint64_t or_of_all(const uint64_t* ors, int tiles) {
  __shared__ uint64_t s_or[kWaves];
  uint64_t v = static_cast<int>(threadIdx.x) < tiles ? ors[threadIdx.x] : 0;
  for (int m = 32; m >= 1; m >>= 1) v |= __shfl_xor(v, m);
  if ((threadIdx.x & 63) == 0) s_or[threadIdx.x >> 6] = v;
  __syncthreads();
  v = 0;
  for (int w = 0; w < kWaves; w++) v |= s_or[w];
  __syncthreads();
  return v;
}

__device__ __forceinline__ uint32_t digit_of(const SortArgs& a, int64_t key, int pass) {
  return static_cast<uint32_t>((static_cast<uint64_t>(key) & a.key_mask) >> (pass * kDigitBits)) &
         (kBins - 1);
}

// Whether pass `pass` of `passes` writes the outputs: the last one does, those before take turns
// with the workspace. Pass 0 reads the ids as given, whose rows are their numbers.
__device__ __forceinline__ bool writes_out(int pass, int passes) {
  return ((passes - 1 - pass) & 1) == 0;
}

// Between a wave's accesses to LDS that its lanes make for each other: the compiler keeps them in
// order across this (the hardware does by itself).
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Count each digit of one tile, and in pass 0 OR its ids.
template <int R>
__global__ __launch_bounds__(kSortThreads) void count_digits(SortArgs a, int pass) {
  __shared__ uint32_t s_count[kBins];
  const int tid = threadIdx.x;
  const int64_t* keys = a.slots;
  if (pass > 0) {
    const int passes = passes_of(or_of_all(a.ors, a.tiles), a.even);
    if (pass >= passes) return;
    keys = writes_out(pass - 1, passes) ? a.out_keys : a.tmp_keys;
  }
  s_count[tid] = 0;
  __syncthreads();
  const int64_t first = static_cast<int64_t>(blockIdx.x) * tile_pairs(R) + tid;
  int64_t key[R];
#pragma unroll
  for (int r = 0; r < R; r++) {
    const int64_t i = first + r * kSortThreads;
    key[r] = keys[i < a.n ? i : a.n - 1];  // past the end: the last one again, not counted
  }
  uint64_t any = 0;
#pragma unroll
  for (int r = 0; r < R; r++) {
    if (first + r * kSortThreads < a.n) atomicAdd(&s_count[digit_of(a, key[r], pass)], 1u);
    any |= static_cast<uint64_t>(key[r]) & a.key_mask;
  }
  if (pass == 0) {
    __shared__ uint64_t s_any[kWaves];
    for (int m = 32; m >= 1; m >>= 1) any |= __shfl_xor(any, m);
    if ((tid & 63) == 0) s_any[tid >> 6] = any;
    __syncthreads();
    if (tid == 0) {
      for (int w = 1; w < kWaves; w++) any |= s_any[w];
      a.ors[blockIdx.x] = any;
    }
  }
  __syncthreads();
  a.counts[static_cast<int64_t>(blockIdx.x) * kBins + tid] = static_cast<uint16_t>(s_count[tid]);
}

// Rank a tile's pairs by digit: rank[r] is the number of pairs of this thread's wave with its
// pair r's digit that come before it, and s_count[w][d] the pairs of wave w with digit d. Each wave
// finds the lanes that share a digit by one ballot a bit, and one of them counts for all: no
// atomics, and the listed order is kept. s_count is this wave's row, zeroed by the wave.
template <int R>
__device__ __forceinline__ void rank_digits(const uint32_t (&digit)[R], int64_t first, int64_t n,
                                            uint32_t (&s_count)[kBins], uint32_t (&rank)[R]) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int r = 0; r < R; r++) {
    const bool live = first + r * 64 + lane < n;
    const uint32_t earlier = s_count[digit[r]];
    const uint64_t live_lanes = __ballot(live);
    uint32_t lo = static_cast<uint32_t>(live_lanes), hi = static_cast<uint32_t>(live_lanes >> 32);
#pragma unroll
    for (int b = 0; b < kDigitBits; b++) {
      const uint32_t set = static_cast<uint32_t>(static_cast<int32_t>(digit[r] << (31 - b)) >> 31);
      const uint64_t with = __ballot(set != 0);
      lo &= ~(static_cast<uint32_t>(with) ^ set);  // the lanes whose bit b is this lane's
      hi &= ~(static_cast<uint32_t>(with >> 32) ^ set);
    }
    const uint32_t mine =  // of them, the lanes before this one
        __builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, 0));
    rank[r] = earlier + mine;
    wave_sync();  // every lane has read its count before one lane adds to it
    if (live && mine == 0) s_count[digit[r]] = earlier + __popc(lo) + __popc(hi);
    wave_sync();
  }
}

// The exclusive sum over the workgroup's threads (one a bin). s_wave: kWaves words.
__device__ __forceinline__ uint32_t scan_bins(uint32_t v, uint32_t* s_wave) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t sum = v;
  for (int m = 1; m < 64; m <<= 1) {
    const uint32_t below = __shfl_up(sum, m);
    if (lane >= m) sum += below;
  }
  if (lane == 63) s_wave[wave] = sum;
  __syncthreads();
  for (int w = 0; w < wave; w++) sum += s_wave[w];
  return sum - v;
}

// The tile of workgroup b: XCD b % 8 takes one contiguous part of them.
__device__ __forceinline__ int xcd_part(int b, int tiles) {
  constexpr int kXcds = 8;
  const int x = b % kXcds, q = tiles / kXcds, r = tiles % kXcds;
  return x * q + (x < r ? x : r) + b / kXcds;
}

// Put one tile's pairs where the whole sort's counts say.
template <int R>
__global__ __launch_bounds__(kSortThreads) void place_pairs(SortArgs a, int pass) {
  __shared__ uint32_t s_count[kWaves][kBins];  // a wave's counts, then where its first pair goes
  __shared__ uint32_t s_all[kWaves][kBins];    // every tile's counts, summed by wave
  __shared__ uint32_t s_earlier[kWaves][kBins];  // those of the tiles before this one
  __shared__ uint32_t s_wave[kWaves];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // Workgroups are dealt to the XCDs round-robin: each XCD takes neighbouring tiles, whose pairs of
  // one digit go to neighbouring places, so that few lines are written by two XCDs.
  const int tile = xcd_part(blockIdx.x, a.tiles);
  const int passes = passes_of(or_of_all(a.ors, a.tiles), a.even);
  if (pass >= passes) return;
  const bool out = writes_out(pass, passes);
  const int64_t* keys = pass == 0 ? a.slots : out ? a.tmp_keys : a.out_keys;
  const int64_t* rows = out ? a.tmp_rows : a.out_rows;  // not read in pass 0

  const int64_t first = static_cast<int64_t>(tile) * tile_pairs(R) + wave * (R * 64);
  int64_t key[R];
  uint32_t row[R], digit[R], rank[R];
#pragma unroll
  for (int r = 0; r < R; r++) {
    const int64_t i = first + r * 64 + lane;
    key[r] = keys[i < a.n ? i : a.n - 1];
    row[r] = static_cast<uint32_t>(i);
  }
  if (pass > 0) {
#pragma unroll
    for (int r = 0; r < R; r++) {
      const int64_t i = first + r * 64 + lane;
      row[r] = static_cast<uint32_t>(rows[i < a.n ? i : a.n - 1]);
    }
  }
  // the counts of every tile: wave w sums tiles w, w + kWaves, ...; a lane holds 8 bins
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
  const u32x4* counts = reinterpret_cast<const u32x4*>(a.counts) + lane;
  constexpr int kRowWords = kBins * 2 / 16;
  uint32_t all[8] = {}, earlier[8] = {};
  constexpr int kAhead = 8;
  for (int t0 = wave; t0 < a.tiles; t0 += kWaves * kAhead) {
    u32x4 c[kAhead];
#pragma unroll
    for (int j = 0; j < kAhead; j++) {
      const int t = t0 + j * kWaves;
      c[j] = counts[static_cast<int64_t>(t < a.tiles ? t : a.tiles - 1) * kRowWords];
    }
#pragma unroll
    for (int j = 0; j < kAhead; j++) {
      const int t = t0 + j * kWaves;
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const uint32_t lo = t < a.tiles ? c[j][q] & 0xffffu : 0u;
        const uint32_t hi = t < a.tiles ? c[j][q] >> 16 : 0u;
        all[2 * q] += lo;
        all[2 * q + 1] += hi;
        if (t < tile) {
          earlier[2 * q] += lo;
          earlier[2 * q + 1] += hi;
        }
      }
    }
  }
#pragma unroll
  for (int q = 0; q < 8; q++) {
    s_all[wave][lane * 8 + q] = all[q];
    s_earlier[wave][lane * 8 + q] = earlier[q];
    s_count[wave][lane * 8 + q] = 0;
  }
  wave_sync();
#pragma unroll
  for (int r = 0; r < R; r++) digit[r] = digit_of(a, key[r], pass);
  rank_digits<R>(digit, first, a.n, s_count[wave], rank);
  __syncthreads();
  uint32_t total = 0, start = 0;
  for (int w = 0; w < kWaves; w++) {
    total += s_all[w][tid];
    start += s_earlier[w][tid];
  }
  start += scan_bins(total, s_wave);
  for (int w = 0; w < kWaves; w++) {
    const uint32_t mine = s_count[w][tid];
    s_count[w][tid] = start;
    start += mine;
  }
  __syncthreads();
  int64_t* to_keys = out ? a.out_keys : a.tmp_keys;
  int64_t* to_rows = out ? a.out_rows : a.tmp_rows;
#pragma unroll
  for (int r = 0; r < R; r++) {
    if (first + r * 64 + lane >= a.n) continue;
    const uint32_t at = s_count[wave][digit_of(a, key[r], pass)] + rank[r];
    to_keys[at] = key[r];
    to_rows[at] = row[r];
  }
}

// A sort of at most kThreads * R pairs: every pass in one launch of one workgroup, the pairs in LDS
// between them.
template <int kThreads, int R>
__global__ __launch_bounds__(kThreads) void sort_tile(SortArgs a) {
  constexpr int kTileWaves = kThreads / 64;
  __shared__ uint32_t s_count[kTileWaves][kBins];
  __shared__ int64_t s_key[kThreads * R];
  __shared__ uint32_t s_row[kThreads * R];
  __shared__ uint32_t s_wave[kTileWaves];
  __shared__ uint64_t s_any[kTileWaves];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t first = wave * (R * 64);
  int64_t key[R];
  uint32_t row[R], digit[R], rank[R];
  uint64_t any = 0;
#pragma unroll
  for (int r = 0; r < R; r++) {
    const int64_t i = first + r * 64 + lane;
    key[r] = a.slots[i < a.n ? i : a.n - 1];
    row[r] = static_cast<uint32_t>(i);
    any |= static_cast<uint64_t>(key[r]) & a.key_mask;
  }
  for (int m = 32; m >= 1; m >>= 1) any |= __shfl_xor(any, m);
  if (lane == 0) s_any[wave] = any;
  __syncthreads();
  any = 0;
  for (int w = 0; w < kTileWaves; w++) any |= s_any[w];
  const int passes = passes_of(any, 0);
  for (int pass = 0;; pass++) {
#pragma unroll
    for (int q = 0; q < 8; q++) s_count[wave][lane * 8 + q] = 0;
    wave_sync();
#pragma unroll
    for (int r = 0; r < R; r++) digit[r] = digit_of(a, key[r], pass);
    rank_digits<R>(digit, first, a.n, s_count[wave], rank);
    __syncthreads();
    uint32_t total = 0;
    if (tid < kBins)
      for (int w = 0; w < kTileWaves; w++) total += s_count[w][tid];
    uint32_t start = scan_bins(total, s_wave);
    if (tid < kBins) {
      for (int w = 0; w < kTileWaves; w++) {
        const uint32_t mine = s_count[w][tid];
        s_count[w][tid] = start;
        start += mine;
      }
    }
    __syncthreads();
    const bool last = pass == passes - 1;
#pragma unroll
    for (int r = 0; r < R; r++) {
      if (first + r * 64 + lane >= a.n) continue;
      const uint32_t at = s_count[wave][digit[r]] + rank[r];
      if (last) {
        a.out_keys[at] = key[r];
        a.out_rows[at] = row[r];
      } else {
        s_key[at] = key[r];
        s_row[at] = row[r];
      }
    }
    if (last) return;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < R; r++) {
      const int64_t i = first + r * 64 + lane;
      if (i >= a.n) continue;
      key[r] = s_key[i];
      row[r] = s_row[i];
    }
  }
}

__global__ __launch_bounds__(kIotaThreads) void iota(int64_t* rows, int64_t n) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kIotaThreads + threadIdx.x;
  if (i < n) rows[i] = i;
}

int64_t round_up(int64_t v) { return (v + kAlign - 1) / kAlign * kAlign; }

bool overlap(const void* p, int64_t p_bytes, const void* q, int64_t q_bytes) {
  const uintptr_t x = reinterpret_cast<uintptr_t>(p), y = reinterpret_cast<uintptr_t>(q);
  return x < y + static_cast<uintptr_t>(q_bytes) && y < x + static_cast<uintptr_t>(p_bytes);
}

// Whether an output overlaps the ids.
bool writes_ids(const int64_t* slots, int64_t n, const int64_t* slots_out,
                const int64_t* rows_out) {
  return overlap(slots, n * 8, slots_out, n * 8) || overlap(slots, n * 8, rows_out, n * 8);
}

int tiles_of(int64_t n) {
  const int64_t tile = tile_pairs(rounds_of(n));
  return static_cast<int>((n + tile - 1) / tile);
}

// The radix sort's workspace: the pairs between passes, the counts and the ORs. Sized for the
// smaller tile at every size, though a sort past 2^19 pairs has half as many, so that it grows with
// the pairs: a workspace for a caller's largest call holds its smaller ones.
int64_t sorted_bytes(int64_t n) {
  const int64_t tiles = (n + tile_pairs(4) - 1) / tile_pairs(4);
  return 2 * round_up(n * 8) + round_up(tiles * kBins * 2) + round_up(tiles * 8);
}

// Whether the radix sort takes these pairs (where an output overlaps the ids it takes every call of
// up to kMaxSorted).
bool sorted_here(int64_t n, int bits) {
  const bool merged = n > kOneTile && n <= kMergedFirst && bits > 2 * kDigitBits;
  return n <= kMaxSorted && !merged;
}

int sort_pairs(const int64_t* slots, int64_t n, int bits, int64_t* slots_out, int64_t* rows_out,
               void* workspace, hipStream_t s) {
  char* w = static_cast<char*>(workspace);
  SortArgs a{};
  a.n = n;
  a.tiles = tiles_of(n);
  a.slots = slots;
  a.out_keys = slots_out;
  a.out_rows = rows_out;
  a.tmp_keys = reinterpret_cast<int64_t*>(w);
  w += round_up(n * 8);
  a.tmp_rows = reinterpret_cast<int64_t*>(w);
  w += round_up(n * 8);
  a.counts = reinterpret_cast<uint16_t*>(w);
  w += round_up(int64_t{a.tiles} * kBins * 2);
  a.ors = reinterpret_cast<uint64_t*>(w);
  a.key_mask = bits == 64 ? ~uint64_t{0} : (uint64_t{1} << bits) - 1;
  a.even = writes_ids(slots, n, slots_out, rows_out);
  const dim3 threads(kSortThreads);
  // one workgroup reads every id before it writes: an overlap is no matter
  if (n <= kOneTile) {
    if (n <= kQuarterTile)
      hipLaunchKernelGGL((sort_tile<512, 4>), dim3(1), dim3(512), 0, s, a);
    else if (n <= kHalfTile)
      hipLaunchKernelGGL((sort_tile<1024, 4>), dim3(1), dim3(1024), 0, s, a);
    else
      hipLaunchKernelGGL((sort_tile<1024, 8>), dim3(1), dim3(1024), 0, s, a);
    EVS_LAUNCHED("evs_order_pairs");
    return EVS_OK;
  }
  int passes = (bits + kDigitBits - 1) / kDigitBits;
  if (a.even) passes = (passes + 1) / 2 * 2;
  const dim3 grid(static_cast<uint32_t>(a.tiles));
  for (int p = 0; p < passes; p++) {
    if (rounds_of(n) == 4) {
      hipLaunchKernelGGL(count_digits<4>, grid, threads, 0, s, a, p);
      hipLaunchKernelGGL(place_pairs<4>, grid, threads, 0, s, a, p);
    } else {
      hipLaunchKernelGGL(count_digits<8>, grid, threads, 0, s, a, p);
      hipLaunchKernelGGL(place_pairs<8>, grid, threads, 0, s, a, p);
    }
    EVS_LAUNCHED("evs_order_pairs");
  }
  return EVS_OK;
}

// rocPRIM's temporary storage for n pairs of 64-bit keys and values over `bits` key bits.
int sort_storage(int64_t n, int bits, size_t* bytes) {
  *bytes = 0;
  EVS_HIP(rocprim::radix_sort_pairs(nullptr, *bytes, static_cast<const uint64_t*>(nullptr),
                                    static_cast<uint64_t*>(nullptr),
                                    static_cast<const int64_t*>(nullptr),
                                    static_cast<int64_t*>(nullptr), static_cast<uint32_t>(n), 0u,
                                    static_cast<unsigned>(bits), hipStream_t{nullptr}));
  return EVS_OK;
}

// The allocation-free variant's scratch: the workspace of a call of up to
// EVS_ORDER_STATIC_MAX_PAIRS pairs, in a file-scope device array. Every GPU the
// library runs on holds its own copy until the process ends. Host code never passes the array's
// name to a kernel (in host code it is a stand-in, not a device address): the address comes from
// hipGetSymbolAddress, once per device, with that device current.
static __device__ __align__(256) unsigned char scratch[EVS_ORDER_STATIC_SCRATCH_BYTES];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_lock;
void* g_scratch[kMaxDevices];  // the array's address on each device, once looked up

// The current device's copy of the scratch array.
int scratch_here(void** out) {
  int dev = -1;
  EVS_HIP(hipGetDevice(&dev));
  EVS_REQUIRE(dev >= 0 && dev < kMaxDevices, "evs_order_pairs_static: device %d past the %d "
              "devices it keeps a scratch address for", dev, kMaxDevices);
  std::lock_guard<std::mutex> hold(g_scratch_lock);
  if (g_scratch[dev] == nullptr) {
    void* p = nullptr;
    EVS_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    EVS_REQUIRE(p != nullptr, "evs_order_pairs_static: no device address for the scratch");
    g_scratch[dev] = p;
  }
  *out = g_scratch[dev];
  return EVS_OK;
}

}  // namespace
}  // namespace evs

extern "C" int evs_order_pairs_workspace(int64_t num_pairs, int key_bits, int64_t* bytes) {
  evs::clear_error();
  EVS_REQUIRE(bytes != nullptr, "evs_order_pairs_workspace: null output");
  EVS_REQUIRE(num_pairs >= 0 && num_pairs < (int64_t{1} << 31),
              "evs_order_pairs_workspace: 0 <= num_pairs < 2^31, got %lld",
              static_cast<long long>(num_pairs));
  EVS_REQUIRE(key_bits >= 1 && key_bits <= 64, "evs_order_pairs_workspace: key_bits in 1..64");
  if (num_pairs <= evs::kMaxSorted) {
    *bytes = evs::sorted_bytes(num_pairs);
    const bool merged = num_pairs > evs::kOneTile && key_bits > 2 * evs::kDigitBits;
    if (merged && *bytes < evs::kMergedBytes) *bytes = evs::kMergedBytes;
    return EVS_OK;
  }
  size_t sort_bytes = 0;
  const int rc = evs::sort_storage(num_pairs, key_bits, &sort_bytes);
  if (rc != EVS_OK) return rc;
  *bytes = evs::round_up(num_pairs * 8) + evs::round_up(static_cast<int64_t>(sort_bytes));
  return EVS_OK;
}

extern "C" int evs_order_pairs(const int64_t* slots, int64_t num_pairs, int key_bits,
                               int64_t* slots_out, int64_t* rows_out, void* workspace,
                               int64_t workspace_bytes, void* stream) {
  evs::clear_error();
  int64_t need = 0;
  int rc = evs_order_pairs_workspace(num_pairs, key_bits, &need);
  if (rc != EVS_OK) return rc;
  if (num_pairs == 0) return EVS_OK;
  EVS_REQUIRE(slots != nullptr && slots_out != nullptr && rows_out != nullptr &&
                  workspace != nullptr,
              "evs_order_pairs: null pointer");
  EVS_REQUIRE(workspace_bytes >= need,
              "evs_order_pairs: the workspace holds %lld bytes, %lld needed",
              static_cast<long long>(workspace_bytes), static_cast<long long>(need));
  EVS_REQUIRE((reinterpret_cast<uintptr_t>(workspace) & (evs::kAlign - 1)) == 0,
              "evs_order_pairs: the workspace must be %lld-byte aligned",
              static_cast<long long>(evs::kAlign));
  hipStream_t s = evs::as_stream(stream);
  const bool in_place = num_pairs <= evs::kMaxSorted &&
                        evs::writes_ids(slots, num_pairs, slots_out, rows_out);
  if (evs::sorted_here(num_pairs, key_bits) || in_place)
    return evs::sort_pairs(slots, num_pairs, key_bits, slots_out, rows_out, workspace, s);
  int64_t* rows = static_cast<int64_t*>(workspace);
  char* sort_tmp = static_cast<char*>(workspace) + evs::round_up(num_pairs * 8);
  size_t sort_bytes = 0;
  rc = evs::sort_storage(num_pairs, key_bits, &sort_bytes);
  if (rc != EVS_OK) return rc;
  EVS_REQUIRE(evs::round_up(num_pairs * 8) + static_cast<int64_t>(sort_bytes) <= need,
              "evs_order_pairs: rocPRIM needs %lld bytes for %lld pairs",
              static_cast<long long>(sort_bytes), static_cast<long long>(num_pairs));
  const int64_t grid = (num_pairs + evs::kIotaThreads - 1) / evs::kIotaThreads;
  hipLaunchKernelGGL(evs::iota, dim3(static_cast<uint32_t>(grid)), dim3(evs::kIotaThreads), 0, s,
                     rows, num_pairs);
  EVS_LAUNCHED("evs_order_pairs");
  // the slot ids are compared as unsigned on their low key_bits bits: a padding id (negative)
  // lands wherever those bits put it, and the pair scatter skips it
  EVS_HIP(rocprim::radix_sort_pairs(sort_tmp, sort_bytes,
                                    reinterpret_cast<const uint64_t*>(slots),
                                    reinterpret_cast<uint64_t*>(slots_out),
                                    static_cast<const int64_t*>(rows), rows_out,
                                    static_cast<uint32_t>(num_pairs), 0u,
                                    static_cast<unsigned>(key_bits), s));
  return EVS_OK;
}

extern "C" int evs_order_pairs_static(const int64_t* slots, int64_t num_pairs, int key_bits,
                                      int64_t* slots_out, int64_t* rows_out, void* stream) {
  evs::clear_error();
  EVS_REQUIRE(num_pairs >= 0 && num_pairs <= EVS_ORDER_STATIC_MAX_PAIRS,
              "evs_order_pairs_static: %lld pairs, at most %d fit its scratch; give "
              "evs_order_pairs a workspace for more",
              static_cast<long long>(num_pairs), EVS_ORDER_STATIC_MAX_PAIRS);
  int64_t need = 0;
  int rc = evs_order_pairs_workspace(num_pairs, key_bits, &need);
  if (rc != EVS_OK) return rc;
  EVS_REQUIRE(need <= EVS_ORDER_STATIC_SCRATCH_BYTES,
              "evs_order_pairs_static: %lld pairs of %d key bits need %lld bytes of scratch, "
              "it holds %d", static_cast<long long>(num_pairs), key_bits,
              static_cast<long long>(need), EVS_ORDER_STATIC_SCRATCH_BYTES);
  if (num_pairs == 0) return EVS_OK;
  void* ptr = nullptr;  // this device's copy of the scratch array
  rc = evs::scratch_here(&ptr);
  if (rc != EVS_OK) return rc;
  // everything in it is written by the call before it is read, so nothing from the previous
  // call's contents is
  return evs_order_pairs(slots, num_pairs, key_bits, slots_out, rows_out, ptr,
                         EVS_ORDER_STATIC_SCRATCH_BYTES, stream);
}
