// The step's KV rows between the paged cache and a staging buffer, on gfx950.
//
// Gather (the snapshot) reads each (layer, head slot, slot) K and V half-row out of a paged cache
// and writes it into a buffer laid out [layers, heads, capacity, 2, head_dim]; scatter (the
// restore) is its inverse. A cache layout is five strides (block, offset in block, head slot,
// K-or-V, element), so the three paged layouts and strided views share one kernel
// (core/everserve/state/kvcopy.py:105-116; the reference kernels are core/csrc/gather.cu:29-71).
//
// Work is cut into small tiles of (one layer, HG consecutive held heads, TS consecutive slots).
// One workgroup owns a tile: its first TS threads turn the tile's slot ids (or block ids) into
// byte offsets inside a layer, the first HG threads the head slots, both into LDS, so each moved
// word costs two LDS reads and no 64-bit division. Each thread then moves VPT words at a time,
// every load in flight before the first store. A word is the widest of 16, 8, 4, 2 and 1 bytes
// that every half-row, contiguous and aligned on both sides, is whole words of (bf16 d=128: 16
// words of 16 bytes a half-row, fp8 d=120: 15 of 8), at least one element. Within a tile the words
// run along the staging buffer (K then V of one row, row after row), so a wave stores whole rows:
// 1 KiB contiguous for bf16 d=128. For the gather
// the tile numbers run through a slot range's head groups first, so the workgroups reading the
// heads of one cache block (adjacent in every paged layout) are neighbours, dealt round-robin to
// the XCDs; the slot and pair scatters' XCD remap (xcd_tile) keeps runs of 64 neighbouring tiles
// on one XCD, and the range scatter's gives each XCD one contiguous part of the grid. Tiles are
// kept small (a few KiB) and numerous: on MI355X many short independent workgroups keep more
// bytes in flight than fewer long ones. Measured and rejected:
// a persistent grid with prefetched indices, and an LDS-staged transpose that reads a tile in
// cache order and writes it in staging order (both slower on every config); for the scatter,
// words in cache order and issuing a tile's loads before its slot ids are read (both slower);
// fewer workgroups per CU (unused LDS as a cap), which speeds a plain copy up by 8 % at 8 KiB per
// workgroup but slows these kernels, whose index prologue needs every resident workgroup to hide
// its latency; each wave reading its own rows' ids with scalar loads, no LDS and no barrier
// (2 % slower: the per-lane choice among the wave's rows costs more than the barrier).

#include <numeric>

#include "common.hpp"

namespace evs {
namespace {

// Tuning, chosen by measurement on MI355X (the defaults); the macros let a sweep build variants
// side by side.
#ifndef EVS_GATHER_THREADS
#define EVS_GATHER_THREADS 256
#endif
#ifndef EVS_SCATTER_THREADS
#define EVS_SCATTER_THREADS 128
#endif
// Words per thread per pass, per direction: all of a pass's loads are issued before its stores.
#ifndef EVS_GATHER_VPT
#define EVS_GATHER_VPT 2
#endif
#ifndef EVS_SCATTER_VPT
#define EVS_SCATTER_VPT 2
#endif
// Per direction, bit 0: nontemporal loads, bit 1: nontemporal stores. Every byte here is touched
// once, so no line is worth keeping in L2 or the Infinity Cache. For the scatter in staged order
// the nontemporal row loads also keep the slot ids in L2: each of a slot range's 8 head tiles
// reads them, far apart in time, and with plain row loads streaming through L2 every read missed
// (HBM traffic 1.0078x the algorithmic bytes at C4; 1.00002x with the loads nontemporal, and
// 5,646-5,657 against 5,627-5,653 GB/s, interleaved rounds on one box). The range scatter reads
// no ids, and its nontemporal loads ran at 5,900 against 5,852 GB/s (C4, one box).
#ifndef EVS_GATHER_NT
#define EVS_GATHER_NT 3
#endif
#ifndef EVS_SCATTER_NT
#define EVS_SCATTER_NT 3
#endif
#ifndef EVS_RANGES_NT
#define EVS_RANGES_NT EVS_SCATTER_NT
#endif
// The gather's 16-byte stores also carry sc1, device scope: written through this XCD's L2, which
// then holds no dirty lines of the staging buffer to write back later. Measured on MI355X (9
// interleaved rounds, the bytes equal): C2 6,087 against 6,003 GB/s on random blocks and 6,168
// against 6,084 on sorted ones, C3 6,147 against 6,045. The scatter's stores were unchanged by it
// (5,619 either way), and keep the plain nontemporal bit. 0: the plain bit for the gather too.
#ifndef EVS_GATHER_STORE_SC1
#define EVS_GATHER_STORE_SC1 1
#endif
// The scatter's word order in a tile. 0: along the cache in the common layouts (a wave covers
// consecutive heads of one slot, K then V); 1: along the staging buffer (whole staged rows).
#ifndef EVS_SCATTER_ORDER
#define EVS_SCATTER_ORDER 1
#endif
// Workgroups are dealt to the XCDs round-robin by id, so consecutive tiles (the tiles of one cache
// block) would each run on another XCD. The chunk per direction remaps tile numbers: 0 leaves
// them; G > 0 gives each XCD G consecutive tiles of every run of kXcds * G; -1 gives each XCD one
// contiguous range of the whole grid.
// The gather leaves the round-robin dealing: against runs of 64 it measured 1.3 % faster on C2's
// random blocks, 3.1 % on sorted ones, 1.2-1.7 % on C3 and 4 % at decode size (5 interleaved
// rounds, three boxes).
#ifndef EVS_GATHER_XCD_CHUNK
#define EVS_GATHER_XCD_CHUNK 0
#endif
// A gather whose tiles cover every held head (one head group, as on a rank holding one KV head)
// numbers its tiles along the slots alone, and there runs of 16 tiles per XCD (128 KiB of staged
// rows each) beat round-robin. 7 interleaved rounds on each of two boxes: one bf16 head, 80
// layers, 65,536 slots 6,184 / 6,218 against 5,946 / 5,978 GB/s (runs of 4 / 8 on the first:
// 5,771 / 5,902); C3's fp8 head 6,138 / 6,216 against 6,030 / 6,131. With several head groups
// the round-robin default stays (C2 6,078 against 6,074 under this switch's build).
#ifndef EVS_GATHER_XCD_CHUNK_ONE_GROUP
#define EVS_GATHER_XCD_CHUNK_ONE_GROUP 16
#endif
#ifndef EVS_SCATTER_XCD_CHUNK
#define EVS_SCATTER_XCD_CHUNK 64
#endif
// The scatter of written ranges (staged rows to the slots of (start, count) ranges, which ascend
// in a restore) gives each XCD one contiguous part of the grid, so that the XCDs write the cache
// in 8 streams that each run front to back. On ascending slots that measured faster than runs of
// 64 on every box tried: a restore's chunk (1 layer, 8 heads, 65,536 slots) 6,339 against 5,735
// GB/s for an isolated launch; 16 layers of C4's cache 5,801-6,144 against 5,447-5,537. For the
// slot scatter's permuted slots it depended on the box (16 layers: 4.8 % faster on two runs, 2.4 %
// slower on another; C4's 32 layers 2 % slower), so that one keeps runs of 64.
#ifndef EVS_RANGES_XCD_CHUNK
#define EVS_RANGES_XCD_CHUNK -1
#endif
constexpr uint32_t kXcds = 8;
constexpr int64_t kCUs = 256;
// The pair scatter (a staged row per listed slot, listed in the order the caller wants written):
// its tiles span all heads (2 slots x 8 heads at bf16 d=128, 8 KiB) and its words run along the
// cache, so that a caller listing its slots in increasing order writes each layer's cache front
// to back. A tile is one pass (256 threads x 2 words) and its reads, which are random, are
// nontemporal, as the gather's are. On C4's permuted block table with the pairs in slot order it
// measured 5,994 GB/s, against 5,660 for the scatter in staged order on the same box.
#ifndef EVS_PAIRS_TILE_WORDS
#define EVS_PAIRS_TILE_WORDS 512
#endif
#ifndef EVS_PAIRS_HEADS_PER_TILE
#define EVS_PAIRS_HEADS_PER_TILE 0
#endif
#ifndef EVS_PAIRS_ORDER
#define EVS_PAIRS_ORDER 0
#endif
#ifndef EVS_PAIRS_XCD_CHUNK
#define EVS_PAIRS_XCD_CHUNK 64
#endif
#ifndef EVS_PAIRS_THREADS
#define EVS_PAIRS_THREADS 256
#endif
#ifndef EVS_PAIRS_NT
#define EVS_PAIRS_NT 3  // its reads are random, as the gather's are: nontemporal both ways
#endif
#ifndef EVS_PAIRS_VPT
#define EVS_PAIRS_VPT 2
#endif
// Tile shape per direction: words a tile aims at, heads it covers (0: all), head groups fastest.
#ifndef EVS_GATHER_TILE_WORDS
#define EVS_GATHER_TILE_WORDS 512
#endif
#ifndef EVS_GATHER_HEADS_PER_TILE
#define EVS_GATHER_HEADS_PER_TILE 2
#endif
#ifndef EVS_GATHER_GROUP_FASTEST
#define EVS_GATHER_GROUP_FASTEST 1
#endif
#ifndef EVS_SCATTER_TILE_WORDS
#define EVS_SCATTER_TILE_WORDS 256
#endif
#ifndef EVS_SCATTER_HEADS_PER_TILE
#define EVS_SCATTER_HEADS_PER_TILE 1
#endif
#ifndef EVS_SCATTER_GROUP_FASTEST
#define EVS_SCATTER_GROUP_FASTEST 0
#endif
#ifndef EVS_RANGES_GROUP_FASTEST
#define EVS_RANGES_GROUP_FASTEST EVS_SCATTER_GROUP_FASTEST
#endif

// s_waitcnt's operand for vmcnt(0) alone: the other counters at their largest
constexpr int kVmcntZero = 0x0f70;
constexpr int kMaxTileSlots = 64;
constexpr int kMaxHeads = 256;      // LDS table of head offsets

enum Dir : int { kGather = 0, kScatter = 1 };
// kBySlots: row t of a layer's staging goes to (or comes from) slot slots[t]; kByBlocks: row t is
// offset t % bs of the (t / bs)-th listed block; kByPairs (scatter): staged row rows_of[i] goes
// to slot slots[i]; kByRanges (scatter): row t goes to slot starts[k] + t - first_rows[k] of the
// range k with first_rows[k] <= t < first_rows[k + 1].
enum Index : int { kBySlots = 0, kByBlocks = 1, kByPairs = 2, kByRanges = 3 };

// A kernel's form. kSpanning (slot and range scatters): the tile spans heads, see launch_typed.
// kSmall (the gather of 16-byte words): half the threads and half the tile.
enum Form : int { kPlain = 0, kSpanning = 1, kSmall = 2 };

constexpr int threads_of(int d, int i, int form = kPlain) {
  return i == kByPairs        ? EVS_PAIRS_THREADS
         : form == kSmall     ? EVS_GATHER_THREADS / 2
         : d == kGather       ? EVS_GATHER_THREADS
         : form == kSpanning  ? 256
                              : EVS_SCATTER_THREADS;
}
// A narrower word's tiles hold more of them where the call is large enough (see tile_words): up to
// 2x at 8 bytes (the same bytes a tile), 4x below, where the work is the address arithmetic a word
// takes. 400 MB gathered from one head, 4x and 2x against 1x: 8-byte words (bf16 100) 5,507 and
// 5,467 against 3,670 GB/s, 2-byte words (fp8 126) 3,433 and 2,428 against 1,546; (bf16 124,
// 8-byte) 4,286 and 5,516 against 4,560.
constexpr int narrow_of(size_t word) { return word == 16 ? 1 : word == 8 ? 2 : 4; }
constexpr int base_vpt(int d, int i) {
  return i == kByPairs ? EVS_PAIRS_VPT : d == kGather ? EVS_GATHER_VPT : EVS_SCATTER_VPT;
}
// Words a thread and pass: the gather's as many times more, and the slot and range scatters' of
// 4-byte words; the other scatters' passes, and the pair scatter's tiles, at most twice as many.
// Microseconds for 8 layers of 4,096 slots of 8 heads, four times, twice, and by elements in a
// 16-byte word's tiles: pairs, bf16 121 215, 137 and 140, fp8 126 116, 79 and 125; slots, bf16 121
// 181, 140 and 197; ranges 216, 163 and 277; but slots of 4-byte words (bf16 126) 80 and 86. Four
// times as many words a pair tile ran 39.5 against 43.7 (fp8 100, kv_first), but 59.5 against 46.5
// in the combined layout.
constexpr int vpt_of(int d, int i, size_t word) {
  const bool most = d == kGather || (i != kByPairs && word == 4);
  return base_vpt(d, i) * (most ? narrow_of(word) : word == 16 ? 1 : 2);
}
constexpr int nt_of(int d, int i) {
  return i == kByPairs    ? EVS_PAIRS_NT
         : i == kByRanges  ? EVS_RANGES_NT
         : d == kGather    ? EVS_GATHER_NT
                           : EVS_SCATTER_NT;
}
// the gather's words run along the staging buffer, so that its tile's words are all live ones
constexpr int word_order(int d, int i, int form) {
  return i == kByPairs       ? EVS_PAIRS_ORDER
         : d == kGather      ? 1
         : form == kSpanning ? 2
                             : EVS_SCATTER_ORDER;
}
static_assert(threads_of(kGather, kBySlots) >= kMaxTileSlots &&
                  threads_of(kScatter, kBySlots) >= kMaxTileSlots &&
                  threads_of(kScatter, kByPairs) >= kMaxTileSlots,
              "the first TS threads fill a tile's slot offsets: a workgroup needs kMaxTileSlots");

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

struct RowsArgs {
  const int64_t* layer_ptrs;  // device: each layer's cache base address
  const int64_t* slots;       // kBySlots: device slot ids
  const int32_t* blocks;      // kByBlocks: device block ids
  const int64_t* heads;       // device head slots
  char* rows;                 // the staging buffer, [L, H, cap, 2, d]
  int64_t* slots_out;         // kByBlocks: the expanded slot ids, or null
  const int64_t* rows_of;     // kByPairs: the staged row of each listed slot
  const int64_t* starts;      // kByRanges: device, each range's first slot
  const int64_t* first_rows;  // kByRanges: device, each range's first row, then n
  int64_t nranges;            // kByRanges
  int64_t n;                  // slots moved per layer
  int64_t cap;                // staging capacity (rows per (layer, head))
  int64_t half_bytes;         // d * elem
  int64_t sb, so, sh, skv;    // cache strides in bytes: block, offset, head, K-or-V
  int64_t sj;                 // cache bytes between consecutive words of a half-row
  int64_t bs;                 // slots per block
  int bs_shift;               // log2(bs) when bs is a power of two, else -1
  int H;
  int HG;                     // heads per tile (a tile's heads are HG consecutive of `heads`)
  int TS;                     // slots per tile
  int group_fastest;          // tile numbers run through head groups first
  int xcd_chunk;              // tiles per XCD per run (see xcd_tile)
  uint32_t W;                 // words per half-row
  FastDiv div_w;              // words per half-row
  FastDiv div_h;              // heads per tile
  FastDiv div_ts;             // slots per tile
  FastDiv div_ts_last;        // slots of a layer's last tile
  FastDiv div_tiles;          // slot tiles per (layer, head group)
  FastDiv div_groups;         // head groups
};

// Every address these kernels touch is global memory (device, or host memory mapped for the
// device), but the cache's come out of a table of integers, so the compiler would emit flat
// accesses; the casts to address space 1 make them global ones.
template <typename T>
using global_ptr = __attribute__((address_space(1))) T*;

// The two sides of a word. The host has checked every stride and the staging buffer for it, but
// the layers' bases are in device memory: a word of 16 bytes has its bases' alignment from the
// caller, and a narrower one may start at any byte of the cache, as a global access may (the
// instructions are the aligned ones). Microseconds a call where the bases lie one element off the
// word, moved by elements, by words cut into bytes and so: the gather of 8,192 slots of one
// bf16 head of 100, 32 layers, 177, 114 and 46; of one 32-bit head of 126 197, 310 and 95; of 8
// slots of 8 bf16 heads of 100, one layer, 2.8, 9.6 and 3.1.
enum Side : int { kStaged, kCache };
template <typename T, Side S>
struct WordOn {
  typedef T type __attribute__((aligned(S == kStaged || sizeof(T) == 16 ? sizeof(T) : 1)));
};

template <typename T, Side S, bool kNt>
__device__ __forceinline__ T load_word(const char* p) {
  typedef typename WordOn<T, S>::type Word;
  const global_ptr<const Word> g = (global_ptr<const Word>)(p);
  if (kNt) return __builtin_nontemporal_load(g);
  return *g;
}

template <typename T, Side S, bool kNt, bool kSc1 = false>
__device__ __forceinline__ void store_word(char* p, T v) {
  typedef typename WordOn<T, S>::type Word;
  const global_ptr<Word> g = (global_ptr<Word>)(p);
  if constexpr (kNt && kSc1 && sizeof(T) == 16)
    // No builtin sets the scope bits on a plain store; the word and the address are the asm's
    // inputs, so the compiler waits for the loaded word before it, as for any store. A store of
    // more than 64 bits reads its data registers after it issues, so a VALU write to them needs
    // one wait state after it; the compiler's hazard check does not see inside the asm, so the
    // s_nop gives that wait state whatever is scheduled next.
    asm volatile("global_store_dwordx4 %0, %1, off sc1 nt\n\ts_nop 0" : : "v"(g), "v"(v)
                 : "memory");
  else if constexpr (kNt && kSc1 && sizeof(T) == 8)
    asm volatile("global_store_dwordx2 %0, %1, off sc1 nt" : : "v"(g), "v"(v) : "memory");
  else if (kNt)
    __builtin_nontemporal_store(v, g);
  else
    *g = v;
}

__device__ __forceinline__ int64_t block_of(int64_t s, const RowsArgs& a) {
  return a.bs_shift >= 0 ? (s >> a.bs_shift) : s / a.bs;
}

__device__ __forceinline__ int64_t offset_in_block(int64_t s, const RowsArgs& a) {
  return a.bs_shift >= 0 ? (s & (a.bs - 1)) : s % a.bs;
}

// Which (layer, head group, slot tile) a tile number names.
struct TileId {
  uint32_t layer, group, tile;
};

// The tile workgroup id b runs, ids being dealt to kXcds XCDs round-robin (x = b % kXcds).
//   chunk > 0: in each run of kXcds * chunk ids, XCD x takes tiles [x chunk, (x + 1) chunk) of the
//              run; a last partial run keeps its ids;
//   chunk < 0: XCD x takes the contiguous tiles [x (q + 1), ...) when x < r, after them q each,
//              for grid = kXcds q + r.
// Both are bijections of [0, grid).
__device__ __forceinline__ uint32_t xcd_tile(uint32_t b, uint32_t grid, int chunk) {
  if (chunk == 0) return b;
  const uint32_t x = b % kXcds, local = b / kXcds;
  if (chunk > 0) {
    const uint32_t run = kXcds * static_cast<uint32_t>(chunk);
    if (b >= grid / run * run) return b;
    const uint32_t g = static_cast<uint32_t>(chunk);
    return (b / run) * run + x * g + local % g;
  }
  const uint32_t q = grid / kXcds, r = grid % kXcds;
  return x < r ? x * (q + 1) + local : r * (q + 1) + (x - r) * q + local;
}

__device__ __forceinline__ TileId tile_id(const RowsArgs& a, uint32_t b) {
  TileId id;
  uint32_t q;
  if (a.group_fastest) {
    // head groups fastest: the tiles that read one slot range's heads run side by side
    a.div_groups.divmod(b, q, id.group);
    a.div_tiles.divmod(q, id.layer, id.tile);
  } else {
    a.div_tiles.divmod(b, q, id.tile);
    a.div_groups.divmod(q, id.layer, id.group);
  }
  return id;
}

// The slot of staged row t (0 <= t < n) in the written ranges: the last range k whose first row
// is at most t (first_rows ascending, first_rows[0] = 0, the last entry n), so an empty range is
// passed over. Ranges that break these rules give slots the caller did not mean, as wrong slot ids
// would; a negative one moves nothing. Found for a tile's rows by the tile's first wave together:
// every lane of wave 0 calls it, lane i with row t = t0 + i (rows past the tile's repeat its last;
// t0 <= t < n). The range
// of t0 is found by a 64-way search, each level one read a lane and a ballot (two levels up to
// 4,096 ranges, where bisection takes a dependent read for each of 12 halvings); then the 64
// ranges from there are read at once, first rows and starts, and each lane picks its own among
// them with shuffles. A lane whose row lies past those 64 ranges (only when many ranges are
// empty) bisects the rest. Every read stays inside first_rows[0 .. nranges] and
// starts[0 .. nranges - 1] whatever the arrays hold.
__device__ __forceinline__ int64_t wave_slot_in_ranges(const RowsArgs& a, int64_t t0, int64_t t) {
  const int64_t nr = a.nranges;
  if (nr == 1) return a.starts[0] + (t - a.first_rows[0]);
  const int lane = static_cast<int>(threadIdx.x & 63);
  int64_t lo = 0, hi = nr;  // the range of t0 is in [lo, hi)
  while (hi - lo > 1) {
    const int64_t step = (hi - lo + 63) >> 6;
    const int64_t p = lo + lane * step;
    const uint64_t le = __ballot(p < hi && a.first_rows[p] <= t0);
    lo += le != 0 ? static_cast<int64_t>(63 - __builtin_clzll(le)) * step : 0;
    hi = lo + step < hi ? lo + step : hi;
  }
  const int64_t k = lo + lane;
  const int64_t fr = a.first_rows[k < nr ? k : nr];  // first_rows[nr] = n: past every row
  const int64_t st = a.starts[k < nr ? k : nr - 1];
  // c: the last of the 64 whose first row is at most t
  int c = 0;
  for (int b = 32; b >= 1; b >>= 1) {
    const int64_t v = __shfl(fr, c + b);
    if (v <= t) c += b;
  }
  int64_t slot = __shfl(st, c) + (t - __shfl(fr, c));
  if (c == 63 && lo + 63 < nr - 1) {
    int64_t l2 = lo + 63, h2 = nr;
    while (h2 - l2 > 1) {
      const int64_t mid = (l2 + h2) >> 1;
      if (a.first_rows[mid] <= t)
        l2 = mid;
      else
        h2 = mid;
    }
    slot = a.starts[l2] + (t - a.first_rows[l2]);
  }
  return slot;
}

// The index entry row t of a layer needs: its slot id, or in the block-table path its block's id.
// It is read at a clamped position (n >= 1 here), so that the read needs no branch; the caller
// discards what it read for a row past n.
template <int I>
__device__ __forceinline__ int64_t index_entry(const RowsArgs& a, int64_t t) {
  const int64_t tc = t < a.n ? t : a.n - 1;
  if (I == kByBlocks) return a.blocks[block_of(tc, a)];
  return a.slots[tc];
}

// Byte offset of slot t's row inside a layer, or -1 when nothing moves for it: t past the end,
// or padding in the scatter. Padding (a negative id) makes the gather read slot 0, as the torch
// path does (core/everserve/state/mirror.py:579). A block-table gather also writes the slot id.
template <int D, int I>
__device__ __forceinline__ int64_t slot_offset(const RowsArgs& a, uint32_t layer, int64_t t,
                                               int64_t entry) {
  if (t >= a.n) return -1;
  if (I == kByBlocks) {
    // row t is offset t % bs of the (t / bs)-th listed block: no slot id to split again
    const int64_t q = block_of(t, a);
    const int64_t r = t - q * a.bs;
    const int64_t blk = entry;
    if (a.slots_out != nullptr && layer == 0) a.slots_out[t] = blk * a.bs + r;
    if (blk < 0) return D == kGather ? 0 : -1;  // as a negative slot id
    return blk * a.sb + r * a.so;
  }
  int64_t s = entry;
  if (s < 0) s = (D == kGather) ? 0 : -1;
  return s >= 0 ? block_of(s, a) * a.sb + offset_in_block(s, a) * a.so : -1;
}

// Where word v of a tile lies: head index h within the tile's group, slot tl within the tile,
// K or V (k) and word j of the half-row. div_ts divides by the slots the words run over.
struct WordAt {
  uint32_t h, tl, k, j;
};

template <int kOrder>
__device__ __forceinline__ WordAt word_at(const RowsArgs& a, const FastDiv& div_ts, uint32_t v) {
  WordAt w;
  uint32_t q, q2;
  a.div_w.divmod(v, q, w.j);
  if (kOrder == 0) {
    // v = ((k * TS + tl) * HG + h) * W + j
    a.div_h.divmod(q, q2, w.h);
    div_ts.divmod(q2, w.k, w.tl);
  } else if (kOrder == 2) {
    // v = ((tl * HG + h) * 2 + k) * W + j: the heads' rows of one slot, slot after slot
    w.k = q & 1u;
    a.div_h.divmod(q >> 1, w.tl, w.h);
  } else {
    // v = ((h * TS + tl) * 2 + k) * W + j: K then V of one staged row, row after row
    w.k = q & 1u;
    div_ts.divmod(q >> 1, w.h, w.tl);
  }
  return w;
}

// Byte offset of a word of staged row `row` in the layer's part of the staging buffer.
__device__ __forceinline__ int64_t staged_offset(const RowsArgs& a, uint32_t h0, int64_t row,
                                                 const WordAt& w, int64_t word_bytes) {
  return (static_cast<int64_t>(h0 + w.h) * a.cap + row) * (2 * a.half_bytes) +
         w.k * a.half_bytes + static_cast<int64_t>(w.j) * word_bytes;
}

// Move kWords words a thread of a gather's tile, kThreads words apart from word v0 + its number
// on, every load in flight before the first store. The last of the wave's kWords runs of 64 may
// end past the tile's words.
template <int kWords, typename T, int kThreads, int kNt, typename Locate>
__device__ __forceinline__ void gather_words(uint32_t v0, uint32_t words, const Locate& locate) {
  T w[kWords];
  char* src[kWords];
  char* dst[kWords];
#pragma unroll
  for (int i = 0; i < kWords; i++) {
    const uint32_t at = v0 + i * kThreads + threadIdx.x;
    locate(i == kWords - 1 && at >= words ? words - 1 : at, src[i], dst[i]);
  }
  // Each load stays where it is issued (the scheduler otherwise issued the second word's
  // load first, after the first's address work, so the first store waited for both loads):
  // now the first word's store waits for its own load only. 9-11 interleaved rounds on two
  // boxes: C2 6,110-6,113 against 6,096-6,098 GB/s, C3 6,159 against 6,124, one bf16 head
  // 6,266 against 6,197, the combined layout 6,090 against 6,057, blocks_first unchanged.
#pragma unroll
  for (int i = 0; i < kWords; i++) {
    w[i] = load_word<T, kCache, (kNt & 1) != 0>(src[i]);
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int i = 0; i < kWords; i++)
    store_word<T, kStaged, (kNt & 2) != 0, EVS_GATHER_STORE_SC1 != 0>(dst[i], w[i]);
}

// A wave's words of the tile from v0 on (`wave`: its first thread's number): kWords a thread for as
// long as the tile has them, then by halves.
template <int kWords, typename T, int kThreads, int kNt, typename Locate>
__device__ __forceinline__ void gather_by_halves(uint32_t v0, uint32_t wave, uint32_t words,
                                                 const Locate& locate) {
  for (; v0 + wave + (kWords - 1) * kThreads < words; v0 += kWords * kThreads)
    gather_words<kWords, T, kThreads, kNt>(v0, words, locate);
  if constexpr (kWords > 1)
    gather_by_halves<kWords / 2, T, kThreads, kNt>(v0, wave, words, locate);
}

// Move a scatter's tile of `words` words, kWords a thread and pass; those locate() has no place for
// move nothing.
template <int kWords, typename T, int D, int I, int F, typename Locate>
__device__ __forceinline__ void scatter_words(uint32_t words, const Locate& locate) {
  constexpr int kThreads = threads_of(D, I, F);
  for (uint32_t v0 = 0; v0 < words; v0 += kThreads * kWords) {
    // The slot scatter waits for each load before the next: its stores land in a random order,
    // and fewer accesses in flight ran faster (65,536 permuted slots x 4 layers x 8 bf16 heads
    // of 128: 5,764 GB/s, 5,620 with a thread's loads in flight together, 5,746 with the last
    // load not waited for). The range and pair scatters, whose stores run along the cache, ran
    // slower so (5,207 against 5,602 and 5,790 against 5,837), and keep their loads together, as
    // does the slot scatter that spans heads (bf16 112, 8 heads: 5,235 against 4,908).
    T w[kWords];
    char* src[kWords];
    char* dst[kWords];
    bool live[kWords];
#pragma unroll
    for (int i = 0; i < kWords; i++)
      live[i] = locate(v0 + i * kThreads + threadIdx.x, dst[i], src[i]);
#pragma unroll
    for (int i = 0; i < kWords; i++) {
      if (live[i]) w[i] = load_word<T, kStaged, (nt_of(D, I) & 1) != 0>(src[i]);
      if (I == kBySlots && F == kPlain) __builtin_amdgcn_s_waitcnt(kVmcntZero);
    }
#pragma unroll
    for (int i = 0; i < kWords; i++)
      if (live[i]) store_word<T, kCache, (nt_of(D, I) & 2) != 0>(dst[i], w[i]);
  }
}

// The same in passes no wider than such a tile needs: a small call's holds one pass of a 16-byte
// word's.
template <int kWords, typename T, int D, int I, int F, typename Locate>
__device__ __forceinline__ void scatter_passes(uint32_t words, const Locate& locate) {
  if constexpr (kWords > base_vpt(D, I)) {
    if (words <= threads_of(D, I, F) * kWords / 2) {
      scatter_passes<kWords / 2, T, D, I, F>(words, locate);
      return;
    }
  }
  scatter_words<kWords, T, D, I, F>(words, locate);
}

// Move one tile's words: the slots' offsets and the heads' are in LDS, and for the pair scatter
// the staged rows'. A wave past the tile's last word leaves; in the wave that holds the last word
// the gather's lanes past it move that word again, which costs nothing (the same lines in the
// same instruction) and keeps every access free of a branch: with a branch around each, the
// compiler waits for every memory operation in flight before each store, which serialises a
// thread's stores (1 % slower on a full tile). Before, lanes without a word moved a cell of a
// device array of their own instead: where the head dim leaves a tile's passes partly empty, those
// write-through stores of every workgroup met on the same few lines and held the gather to
// 1.5-1.8 TB/s. 400 MB of one or eight heads, head dims 80, 96, 112, 120 and 192 in bf16 and fp8:
// 1,461-1,813 GB/s before, 5,076-6,105 now (bf16 120, eight heads kv_first 1,483 and 5,078; 112
// combined 1,650 and 5,678); head dim 128 unchanged (5,642 and 5,613; one head 6,103 and 6,105).
// The scatter keeps a branch around each access, and a word past its tile moves nothing.
template <typename T, int D, int I, int F>
__device__ __forceinline__ void move_tile(const RowsArgs& a, const int64_t* s_slot,
                                          const int64_t* s_head, const int64_t* s_src,
                                          int64_t layer_base, uint32_t layer, uint32_t group,
                                          int64_t t0) {
  constexpr int kThreads = threads_of(D, I, F);
  constexpr int kVpt = vpt_of(D, I, sizeof(T));
  const uint32_t h0 = group * a.HG;
  const uint32_t tid = threadIdx.x;
  char* cache_w = reinterpret_cast<char*>(layer_base);
  char* rows_l = a.rows + static_cast<int64_t>(layer) * a.H * a.cap * (2 * a.half_bytes);

  // The gather's words are its tile's live ones alone, [0, words); the scatter's run over the whole
  // tile, and those of a slot past n or a head past H move nothing.
  const bool short_tile = D == kGather && t0 + a.TS > a.n;
  const uint32_t slots = short_tile ? static_cast<uint32_t>(a.n - t0) : a.TS;
  const FastDiv div_ts = short_tile ? a.div_ts_last : a.div_ts;
  const bool few_heads = D == kGather && h0 + a.HG > static_cast<uint32_t>(a.H);
  const uint32_t words = (few_heads ? a.H - h0 : a.HG) * slots * 2 * a.W;

  // where word v lies on both sides, and whether it moves
  const auto locate = [&](uint32_t v, char*& cache, char*& staged) {
    const WordAt at = word_at<word_order(D, I, F)>(a, div_ts, v);
    const bool in_tile =
        D == kGather || (v < words && h0 + at.h < static_cast<uint32_t>(a.H));
    const int64_t slot_off = in_tile ? s_slot[at.tl] : -1;
    const int64_t row = I == kByPairs ? s_src[at.tl] : t0 + at.tl;
    cache = cache_w + slot_off + s_head[in_tile ? at.h : 0] + at.k * a.skv + at.j * a.sj;
    staged = rows_l + staged_offset(a, h0, row, at, sizeof(T));
    return slot_off >= 0;
  };

  if constexpr (D == kGather) {
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid & ~63u);
    if constexpr (kVpt > 2) {
      gather_by_halves<kVpt, T, kThreads, nt_of(D, I)>(0, wave, words, locate);
    } else {
      // the same for two words a thread, written out: this form ran 0.3-0.8 % faster for them
      for (uint32_t v0 = 0; v0 < words; v0 += kThreads * kVpt) {
        if (v0 + wave >= words) break;  // this wave's later passes lie further on still
        if (v0 + wave + (kVpt - 1) * kThreads < words) {
          gather_words<kVpt, T, kThreads, nt_of(D, I)>(v0, words, locate);
        } else {
          for (uint32_t v1 = v0; v1 + wave < words; v1 += kThreads)
            gather_words<1, T, kThreads, nt_of(D, I)>(v1, words, locate);
        }
      }
    }
    return;
  }
  scatter_passes<kVpt, T, D, I, F>(words, locate);
}

// Fill a tile's slot and head offsets into LDS. The first wave reads both index entries before it
// uses either, so that the two reads are in flight together; its lanes past the tile's slots and
// heads read the tile's last entry again, so that the reads touch only the tile's own lines.
template <int D, int I, int F>
__device__ __forceinline__ void tile_offsets(const RowsArgs& a, const TileId& id, int64_t t0,
                                             int64_t* s_slot, int64_t* s_head, int64_t* s_src) {
  const int tid = threadIdx.x;
  const int h0 = static_cast<int>(id.group) * a.HG;
  static_assert(kMaxTileSlots == 64, "the first wave fills a tile's slots: one lane a slot");
  if (tid < kMaxTileSlots) {
    const int64_t t = t0 + (tid < a.TS ? tid : a.TS - 1);
    // a slot, or a block; the range path reads as a wave, the others a lane at a time
    int64_t entry;
    if constexpr (I == kByRanges)
      entry = wave_slot_in_ranges(a, t0, t < a.n ? t : a.n - 1);
    else
      entry = index_entry<I == kByPairs ? kBySlots : I>(a, t);
    const int64_t src = I == kByPairs ? a.rows_of[t < a.n ? t : a.n - 1] : 0;
    const int hc = h0 + (tid < a.HG ? tid : a.HG - 1);
    const int64_t head = a.heads[hc < a.H ? hc : a.H - 1];
    if (tid < a.TS) {
      int64_t off = slot_offset<D, I == kByBlocks ? kByBlocks : kBySlots>(a, id.layer, t0 + tid,
                                                                          entry);
      if (I == kByPairs) {
        if (src < 0 || src >= a.cap) off = -1;  // a staged row outside the buffer moves nothing
        s_src[tid] = src;
      }
      s_slot[tid] = off;
    }
    if (tid < a.HG && h0 + tid < a.H) s_head[tid] = head * a.sh;
  }
  for (int h = kMaxTileSlots + tid; h < a.HG && h0 + h < a.H; h += threads_of(D, I, F))
    s_head[h] = a.heads[h0 + h] * a.sh;
}

// One tile per workgroup.
template <typename T, int D, int I, int F>
__global__ __launch_bounds__(threads_of(D, I, F)) void move_rows(RowsArgs a) {
  __shared__ int64_t s_slot[kMaxTileSlots];  // byte offset of a slot's row in a layer, -1: none
  __shared__ int64_t s_head[kMaxHeads];      // byte offset of a head slot in a row group
  __shared__ int64_t s_src[I == kByPairs ? kMaxTileSlots : 1];  // kByPairs: staged row of a slot

  const TileId id = tile_id(a, xcd_tile(blockIdx.x, gridDim.x, a.xcd_chunk));
  const int64_t t0 = static_cast<int64_t>(id.tile) * a.TS;
  // Read before the block-table path's slot-tag store below: after a store the compiler cannot
  // keep this uniform read scalar (the store might alias it), and a vector read of it made every
  // pass wait for all memory operations in flight (measured 8 % slower).
  const int64_t layer_base = a.layer_ptrs[id.layer];
  tile_offsets<D, I, F>(a, id, t0, s_slot, s_head, s_src);
  __syncthreads();
  move_tile<T, D, I, F>(a, s_slot, s_head, s_src, layer_base, id.layer, id.group, t0);
}

struct RowsCall {
  const int64_t* layer_ptrs;
  int64_t L;
  const int64_t* slots;
  const int32_t* blocks;
  int64_t n_index;  // slots, or blocks
  const int64_t* heads;
  int64_t H;
  char* rows;
  int64_t cap;
  int64_t d;
  int64_t bs;
  const int64_t* strides;
  int64_t elem;
  int64_t* slots_out;
  const int64_t* rows_of;
  hipStream_t stream;
  const int64_t* starts = nullptr;      // kByRanges
  const int64_t* first_rows = nullptr;  // kByRanges
  int64_t nranges = 0;                  // kByRanges
};

// Half-rows that are no whole number of 128-byte memory lines leave lines that two heads' or two
// tiles' words share. Two workgroups that each write a part of a line, or read it, on different
// XCDs may move it twice, so the tile's heads and slots are chosen to cover lines whole. MiB a
// launch of 8,192 slots x 8 fp8 heads of 120, 8 layers (120 each way), before and now: the gather
// fetched 193 and 151 and wrote 140 and 120, the scatter wrote 178 and 139. Of bf16 112 (112 each
// way) the scatter wrote 113 and 117: its parts of a line met in a cache before, and what it gained
// (see launch_typed) is not in the bytes.
constexpr int64_t kLine = 128;

// The fewest runs of `bytes`, one after another, that fill whole lines.
int64_t per_line(int64_t bytes) { return kLine / std::gcd(kLine, bytes); }

// Launch tiles of `hg` heads (0: all) and about `target` words. lines: a gather's tile may be cut
// or grown to whole lines of its rows, and a call past the launch limit is tried in plain tiles.
template <int D, int I, int F, typename T>
int launch_tiles(RowsArgs a, int64_t L, int64_t hg, int64_t target, hipStream_t stream,
                 const char* name, bool lines = true) {
  const uint32_t W = a.W;
  const int64_t threads = threads_of(D, I, F);
  a.HG = static_cast<int>(hg > 0 && hg < a.H ? hg : a.H);
  a.group_fastest = D == kGather      ? EVS_GATHER_GROUP_FASTEST
                    : I == kByRanges ? EVS_RANGES_GROUP_FASTEST
                                     : EVS_SCATTER_GROUP_FASTEST;
  a.xcd_chunk = I == kByPairs ? EVS_PAIRS_XCD_CHUNK
                : I == kByRanges ? EVS_RANGES_XCD_CHUNK
                : D == kGather ? EVS_GATHER_XCD_CHUNK : EVS_SCATTER_XCD_CHUNK;
  const int64_t groups = (a.H + a.HG - 1) / a.HG;
  if (D == kGather && groups == 1) a.xcd_chunk = EVS_GATHER_XCD_CHUNK_ONE_GROUP;
  const int64_t per_slot = static_cast<int64_t>(a.HG) * 2 * W;
  int64_t ts = target / per_slot;
  if (D == kGather && lines) {
    // Whole lines of each head's staged rows, where that leaves no more than an eighth of the
    // tile's words empty or needs no more than two tiles' words (of 8 or 16 bytes). 400 MB of one
    // head: bf16 120 (16 slots a tile for 17) 5,971 against 5,148 GB/s, fp8 80 (48 for 51) 5,967
    // against 5,142; bf16 100 (20 to 16) would run at 5,139 against 5,465, bf16 126 (8 to 16, two
    // heads, 4-byte words) at 4,865 against 5,361.
    const int64_t whole = per_line(2 * a.half_bytes);
    if (ts / whole * whole * 8 >= ts * 7)
      ts = ts / whole * whole;
    else if (sizeof(T) >= 8 && ts < whole && whole * per_slot <= 2 * target)
      ts = whole;
  }
  ts = ts < 1 ? 1 : (ts > kMaxTileSlots ? kMaxTileSlots : ts);
  if (ts > a.n) ts = a.n;
  const int64_t tiles = (a.n + ts - 1) / ts;
  const int64_t grid = tiles * groups * L;
  EVS_REQUIRE(ts * per_slot < (int64_t{1} << 31), "%s: a tile of %lld words is too large", name,
              static_cast<long long>(ts * per_slot));
  // HIP on AMD GPUs takes at most 2^32 - 1 work-items along x (gridDim.x * blockDim.x). A shape
  // chosen for its lines may leave some of a tile's words empty, and so need more workgroups, and
  // the pair scatter's tiles hold no more than twice a 16-byte word's: a call that is too large for
  // them still fits the plain ones.
  if (lines && grid * threads >= (int64_t{1} << 32))
    return launch_tiles<D, I, kPlain, T>(
        a, L,
        I == kByPairs    ? EVS_PAIRS_HEADS_PER_TILE
        : D == kGather ? EVS_GATHER_HEADS_PER_TILE
                       : EVS_SCATTER_HEADS_PER_TILE,
        (I == kByPairs    ? EVS_PAIRS_TILE_WORDS
         : D == kGather ? EVS_GATHER_TILE_WORDS
                        : EVS_SCATTER_TILE_WORDS) * narrow_of(sizeof(T)),
        stream, name, false);
  EVS_REQUIRE(grid * threads < (int64_t{1} << 32),
              "%s: %lld workgroups of %d threads exceed the launch limit of 2^32 - 1 work-items; "
              "split the call by layers", name, static_cast<long long>(grid),
              static_cast<int>(threads));
  a.TS = static_cast<int>(ts);
  a.div_w = FastDiv(W);
  a.div_h = FastDiv(static_cast<uint32_t>(a.HG));
  a.div_ts = FastDiv(static_cast<uint32_t>(ts));
  a.div_ts_last = FastDiv(static_cast<uint32_t>(a.n - (tiles - 1) * ts));
  a.div_tiles = FastDiv(static_cast<uint32_t>(tiles));
  a.div_groups = FastDiv(static_cast<uint32_t>(groups));
  hipLaunchKernelGGL((move_rows<T, D, I, F>), dim3(static_cast<uint32_t>(grid)),
                     dim3(static_cast<uint32_t>(threads)), 0, stream, a);
  EVS_LAUNCHED(name);
  return EVS_OK;
}

// Heads of a gather's tile. Two, or four where the heads of a slot lie side by side in half-rows of
// at most 256 bytes (four slots a tile or more) and the rows of two neighbouring heads in the
// staging buffer are at most 4 MiB apart: a tile writes all its heads at once, and heads 8 MiB
// apart and more meet on the same memory channels. bf16, 8 heads of 128,
// 32 layers, four against two: 8,192 slots (4 MiB) 6,310 against 6,088 GB/s, 5,001 6,303 against
// 6,014, 1,000 6,035 against 5,919; 16,384 slots (8 MiB) 6,111 against 6,160, 65,536 (8 layers)
// 5,915 against 5,980; four heads in all, 8,192 slots 5,956 against 6,213. Where the half-rows are no whole lines: as many heads as fill them, or all,
// if two tiles' words hold whole lines of those heads' staged rows. 400 MB, 8 heads: bf16 80 (4
// heads) 5,541 against 5,124 with two, fp8 112 (8) 5,341 against 4,445, fp8 120 (8) 4,957 against
// 3,517; bf16 100, whose 8 heads do not fit, 5,072 with four against 3,865 with 8.
int64_t gather_heads(const RowsArgs& a, int64_t target) {
  if (a.sh != a.half_bytes) return EVS_GATHER_HEADS_PER_TILE;
  const int64_t whole = per_line(a.half_bytes);
  const int64_t hg = whole < a.H ? whole : a.H;
  if (whole > 2 && whole <= 16 && a.H % hg == 0 &&
      per_line(2 * a.half_bytes) * hg * 2 * a.W <= 2 * target)
    return hg;
  return a.H > 4 && a.H % 4 == 0 && a.half_bytes <= 256 &&
                 a.cap * 2 * a.half_bytes <= (int64_t{4} << 20)
             ? 4
             : EVS_GATHER_HEADS_PER_TILE;
}

// Heads of a spanning scatter's tile: enough to fill whole lines of a slot's heads (or all of
// them), the most of those that leave the fewest of a pass's words without work.
int64_t span_heads(const RowsArgs& a, int64_t target) {
  const int64_t H = a.H, whole = per_line(a.half_bytes), head_words = 2 * a.W;
  int64_t best = whole < H ? whole : H, best_live = 0;
  for (int64_t hg = whole; hg < H + whole; hg += whole) {
    const int64_t h = hg < H ? hg : H;
    const int64_t slots = target / (h * head_words);
    if (slots == 0) break;
    const int64_t groups = (H + h - 1) / h;
    const int64_t live = H * slots * head_words * 256 / (groups * target);  // of 256
    if (live >= best_live) {
      best = h;
      best_live = live;
    }
  }
  return best;
}

// Sizes of a call, in words, at which its tiles change: below them a larger tile leaves a CU so
// few waves that their own round trips are the call's time. From kTwice on the tiles of narrow
// words hold twice a 16-byte word's number, from kFourTimes (words below 8 bytes) four times.
// Below kFewWords a gather's tile has two heads at most. From kHalfTile on the gather of kSmall's
// rule takes half-size tiles. Microseconds with the large tiles at every size, and so: gathers of
// 8 slots of 8 heads of one layer, fp8 120 3.85 and 2.64, bf16 120 3.32 and 2.62; 16 slots x 32
// layers 4.22 and 2.81, 3.60 and 2.85; the scatter's 8 slots of 8 fp8 heads of 120 3.12 and 2.66.
// Calls past each line ran as fast or faster in the larger tiles (0.4 to 3.5 million words of
// every width, each 1x, 2x and 4x).
constexpr int64_t kFewWords = 1024 * kCUs;
constexpr int64_t kTwice = 2048 * kCUs;
constexpr int64_t kFourTimes = 8192 * kCUs;
constexpr int64_t kHalfTile = 65536 * kCUs;

// The words a tile aims at in a call of `words`, with `base` a 16-byte word's.
template <typename T>
int64_t tile_words(int64_t base, int64_t words) {
  const int64_t times = words >= kFourTimes ? 4 : words >= kTwice ? 2 : 1;
  return base * (times < narrow_of(sizeof(T)) ? times : narrow_of(sizeof(T)));
}

template <int D, int I, typename T>
int launch_typed(RowsArgs a, int64_t L, uint32_t W, hipStream_t stream, const char* name) {
  a.W = W;
  const int64_t words = L * a.H * a.n * 2 * W;
  if constexpr (I == kByPairs) {
    const int64_t twice = words < kFourTimes ? words : kTwice;  // at most (see vpt_of)
    return launch_tiles<D, I, kPlain, T>(a, L, EVS_PAIRS_HEADS_PER_TILE,
                                        tile_words<T>(EVS_PAIRS_TILE_WORDS, twice), stream, name);
  } else if constexpr (D == kGather) {
    const int64_t target = tile_words<T>(EVS_GATHER_TILE_WORDS, words);
    const int64_t hg = words < kFewWords ? EVS_GATHER_HEADS_PER_TILE : gather_heads(a, target);
    if constexpr (sizeof(T) == 16) {
      // Two heads a tile of several (their rows far apart, see gather_heads), half-rows of one or
      // two whole lines, in a large call: half the tile. bf16 heads of 128, microseconds a call in
      // half-size and whole tiles: 8 heads, 16,384 slots x 32 layers 706 and 711, 32,768 x 16 760
      // and 770; 4 heads, 32,768 x 16 363 and 370; 16 heads, 32,768 x 16 1,588 and 1,581; d 64 the
      // same within 1 %. Half-rows of 512 bytes lost (8 heads, 32,768 x 16 1,543 and 1,471), and so
      // did smaller calls (4 heads, 1,000 slots x 32 layers 24.5 and 22.9; 8 32-bit heads, 1,500
      // slots of one layer 6.6 and 5.4).
      if (hg == 2 && a.H > 2 && a.sh == a.half_bytes && per_line(a.half_bytes) == 1 &&
          a.half_bytes <= 256 && words >= kHalfTile)
        return launch_tiles<D, I, kSmall, T>(a, L, hg, target / 2, stream, name);
    }
    return launch_tiles<D, I, kPlain, T>(a, L, hg, target, stream, name);
  } else {
    // Where a slot's heads lie side by side in half-rows that are no whole lines, the scatter of
    // one head a tile writes each line in parts from several workgroups: the tile spans heads
    // instead, one slot's heads after another. 400 MB, 8 heads, by slots: fp8 64 4,519 -> 5,630
    // GB/s, 96 2,220 -> 5,290, 120 1,910 -> 4,627, bf16 80 2,950 -> 5,358, 112 3,498 -> 5,235, 120
    // 3,104 -> 5,347; by 1,034 ranges: fp8 64 3,823 -> 5,423, bf16 80 2,834 -> 4,921. Half-rows of
    // whole lines run faster one head a tile (bf16 128: 5,862 against 5,627 spanning). A slot whose
    // heads do not fit one pass spans only where such slots fill the CUs twice: 18 slots x 8 layers
    // of 16 bf16 heads of 121 took 6.6 us spanning and take 4.4, 64 slots 7.2 and 7.0.
    if (a.H > 1 && a.sh == a.half_bytes && per_line(a.half_bytes) > 1) {
      const int64_t target = tile_words<T>(512, words);  // 2 a thread
      const int64_t heads = span_heads(a, target);
      if (heads * 2 * W <= 512 || words / (heads * 2 * W) >= 2 * kCUs)
        return launch_tiles<D, I, kSpanning, T>(a, L, heads, target, stream, name);
    }
    return launch_tiles<D, I, kPlain, T>(a, L, EVS_SCATTER_HEADS_PER_TILE,
                                        tile_words<T>(EVS_SCATTER_TILE_WORDS, words), stream, name);
  }
}

// The checks of a call's arguments. *moves is false when the call has nothing to move (no slot,
// head or layer); its pointers are not checked then.
template <int D, int I>
int check_call(const RowsCall& c, const char* name, bool* moves) {
  *moves = false;
  EVS_REQUIRE(c.strides != nullptr, "%s: a layout is five strides", name);
  EVS_REQUIRE(c.elem == 1 || c.elem == 2 || c.elem == 4, "%s: unsupported element size %lld",
              name, static_cast<long long>(c.elem));
  EVS_REQUIRE(c.L >= 0 && c.n_index >= 0 && c.H >= 0, "%s: negative count", name);
  EVS_REQUIRE(c.d >= 1 && c.bs >= 1, "%s: head_dim and block_size must be positive", name);
  EVS_REQUIRE(c.H <= kMaxHeads, "%s: at most %d head slots per call, got %lld", name, kMaxHeads,
              static_cast<long long>(c.H));
  const int64_t n = I == kByBlocks ? c.n_index * c.bs : c.n_index;
  // a pair names its staged row, so pairs may outnumber the rows (a row written to several slots)
  EVS_REQUIRE(I == kByPairs || n <= c.cap,
              "%s: more slots (%lld) than the staging capacity (%lld)", name,
              static_cast<long long>(n), static_cast<long long>(c.cap));
  EVS_REQUIRE(c.cap >= 0, "%s: negative capacity", name);
  if (n == 0 || c.H == 0 || c.L == 0) return EVS_OK;
  EVS_REQUIRE(c.layer_ptrs != nullptr && c.heads != nullptr && c.rows != nullptr,
              "%s: null pointer", name);
  EVS_REQUIRE(I == kByBlocks ? c.blocks != nullptr
              : I == kByRanges ? c.starts != nullptr && c.first_rows != nullptr
                               : c.slots != nullptr,
              "%s: null index", name);
  EVS_REQUIRE(I != kByPairs || c.rows_of != nullptr, "%s: null row list", name);
  EVS_REQUIRE(I != kByRanges || c.nranges >= 1, "%s: rows to move but no range", name);
  *moves = true;
  return EVS_OK;
}

template <int D, int I>
int move(const RowsCall& c, const char* name) {
  bool moves = false;
  const int rc = check_call<D, I>(c, name, &moves);
  if (rc != EVS_OK || !moves) return rc;
  const int64_t n = I == kByBlocks ? c.n_index * c.bs : c.n_index;
  const int64_t e = c.elem;
  RowsArgs a{};
  a.layer_ptrs = c.layer_ptrs;
  a.slots = c.slots;
  a.blocks = c.blocks;
  a.heads = c.heads;
  a.rows = c.rows;
  a.slots_out = c.slots_out;
  a.rows_of = c.rows_of;
  a.starts = c.starts;
  a.first_rows = c.first_rows;
  a.nranges = c.nranges;
  a.n = n;
  a.cap = c.cap;
  a.half_bytes = c.d * e;
  a.sb = c.strides[0] * e;
  a.so = c.strides[1] * e;
  a.sh = c.strides[2] * e;
  a.skv = c.strides[3] * e;
  a.bs = c.bs;
  a.bs_shift = -1;
  if ((c.bs & (c.bs - 1)) == 0) {
    int s = 0;
    while ((int64_t{1} << s) < c.bs) ++s;
    a.bs_shift = s;
  }
  a.H = static_cast<int>(c.H);

  // The widest word that every half-row is whole words of, on both sides; one element where a
  // half-row's elements are not contiguous in the cache. By 8, 4 and 2 bytes instead of one
  // element, 400 MB gathered from one combined-layout head: fp8 120 771 -> 5,560 GB/s, bf16 100
  // 1,225 -> 5,120, fp8 100 -> 3,130, fp8 126 824 -> 3,490. The scatter: fp8 120 718 -> 5,100,
  // bf16 100 1,134 -> 4,520.
  int64_t word = e;
  if (c.strides[4] == 1)
    for (const int64_t w : {int64_t{16}, int64_t{8}, int64_t{4}, int64_t{2}}) {
      if (w <= word) break;
      if (((c.d * e | reinterpret_cast<int64_t>(c.rows) | a.sb | a.so | a.sh | a.skv) & (w - 1)) == 0) {
        word = w;
        break;
      }
    }
  a.sj = c.strides[4] == 1 ? word : c.strides[4] * e;
  EVS_REQUIRE(word == 16 || c.d < (int64_t{1} << 24), "%s: head_dim too large", name);
  const uint32_t W = static_cast<uint32_t>(c.d * e / word);
  switch (word) {
    case 16:
      return launch_typed<D, I, u32x4>(a, c.L, W, c.stream, name);
    case 8:
      return launch_typed<D, I, u32x2>(a, c.L, W, c.stream, name);
    case 4:
      return launch_typed<D, I, uint32_t>(a, c.L, W, c.stream, name);
    case 2:
      return launch_typed<D, I, uint16_t>(a, c.L, W, c.stream, name);
    default:
      return launch_typed<D, I, uint8_t>(a, c.L, W, c.stream, name);
  }
}

}  // namespace
}  // namespace evs

extern "C" int evs_gather_rows(const int64_t* layer_ptrs, int64_t num_layers,
                               const int64_t* slots, int64_t num_slots, const int64_t* heads,
                               int64_t num_heads, void* out, int64_t capacity, int64_t head_dim,
                               int64_t block_size, const int64_t* strides, int64_t elem_size,
                               void* stream) {
  evs::clear_error();
  evs::RowsCall c{layer_ptrs, num_layers, slots, nullptr, num_slots, heads, num_heads,
                  static_cast<char*>(out), capacity, head_dim, block_size, strides, elem_size,
                  nullptr, nullptr, evs::as_stream(stream)};
  return evs::move<evs::kGather, evs::kBySlots>(c, "evs_gather_rows");
}

extern "C" int evs_gather_blocks(const int64_t* layer_ptrs, int64_t num_layers,
                                 const int32_t* block_ids, int64_t num_blocks,
                                 const int64_t* heads, int64_t num_heads, void* out,
                                 int64_t capacity, int64_t head_dim, int64_t block_size,
                                 const int64_t* strides, int64_t elem_size, int64_t* slots_out,
                                 void* stream) {
  evs::clear_error();
  evs::RowsCall c{layer_ptrs, num_layers, nullptr, block_ids, num_blocks, heads, num_heads,
                  static_cast<char*>(out), capacity, head_dim, block_size, strides, elem_size,
                  slots_out, nullptr, evs::as_stream(stream)};
  return evs::move<evs::kGather, evs::kByBlocks>(c, "evs_gather_blocks");
}

extern "C" int evs_scatter_rows(const int64_t* layer_ptrs, int64_t num_layers,
                                const int64_t* slots, int64_t num_slots, const int64_t* heads,
                                int64_t num_heads, const void* in, int64_t capacity,
                                int64_t head_dim, int64_t block_size, const int64_t* strides,
                                int64_t elem_size, void* stream) {
  evs::clear_error();
  evs::RowsCall c{layer_ptrs, num_layers, slots, nullptr, num_slots, heads, num_heads,
                  const_cast<char*>(static_cast<const char*>(in)), capacity, head_dim,
                  block_size, strides, elem_size, nullptr, nullptr, evs::as_stream(stream)};
  return evs::move<evs::kScatter, evs::kBySlots>(c, "evs_scatter_rows");
}

extern "C" int evs_scatter_pairs(const int64_t* layer_ptrs, int64_t num_layers,
                                 const int64_t* slots, const int64_t* rows_of, int64_t num_pairs,
                                 const int64_t* heads, int64_t num_heads, const void* in,
                                 int64_t capacity, int64_t head_dim, int64_t block_size,
                                 const int64_t* strides, int64_t elem_size, void* stream) {
  evs::clear_error();
  evs::RowsCall c{layer_ptrs, num_layers, slots, nullptr, num_pairs, heads, num_heads,
                  const_cast<char*>(static_cast<const char*>(in)), capacity, head_dim,
                  block_size, strides, elem_size, nullptr, rows_of, evs::as_stream(stream)};
  return evs::move<evs::kScatter, evs::kByPairs>(c, "evs_scatter_pairs");
}

extern "C" int evs_scatter_ranges(const int64_t* layer_ptrs, int64_t num_layers,
                                  const int64_t* starts, const int64_t* first_rows,
                                  int64_t num_ranges, int64_t num_rows, const int64_t* heads,
                                  int64_t num_heads, const void* in, int64_t capacity,
                                  int64_t head_dim, int64_t block_size, const int64_t* strides,
                                  int64_t elem_size, void* stream) {
  evs::clear_error();
  EVS_REQUIRE(num_ranges >= 0, "evs_scatter_ranges: negative range count");
  evs::RowsCall c{layer_ptrs, num_layers, nullptr, nullptr, num_rows, heads, num_heads,
                  const_cast<char*>(static_cast<const char*>(in)), capacity, head_dim,
                  block_size, strides, elem_size, nullptr, nullptr, evs::as_stream(stream),
                  starts, first_rows, num_ranges};
  return evs::move<evs::kScatter, evs::kByRanges>(c, "evs_scatter_ranges");
}
