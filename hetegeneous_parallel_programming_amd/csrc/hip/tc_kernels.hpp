// Device-side layout shared by the kernels (tc_kernels.hip) and the host
// runtime (tc_runtime.cpp, tc_batch.cpp).  Plain structs only: the runtime
// never sees kernel bodies, it calls the launchers declared at the bottom.
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>

#include "tc_host.h"

namespace tck {

constexpr int kBlock = 256;   // threads per workgroup = 4 wave64s
constexpr int kWaves = kBlock / 64;

// Degree bins, in the order tiles are handed out (heaviest first).
enum Bin : int {
  BIN_GLOBAL = 0,  // d+(u) > kCapBlock: whole workgroup, pivot list read from HBM
  BIN_BLOCK = 1,   // whole workgroup, pivot list in LDS
  BIN_WAVE = 2,    // one wave64 per pivot
  BIN_G32 = 3,     // 32-lane groups
  BIN_G16 = 4,     // 16-lane groups
  BIN_G8 = 5,      // 8-lane groups
  kNumBins = 6,
  kNoBin = 0xFF    // pivot cannot close a triangle (d+ < 2 or no wedge)
};

// Largest pivot list (ids + 1) of each bin: the tree of a bin's pivot fits
// kCap words.
constexpr int kCapG8 = 32, kCapG16 = 64, kCapG32 = 256, kCapWave = 1024, kCapBlock = 4096;
// LDS words of one group's pivot-set area per bin (hash tables or tree);
// every bin's areas fill the same 4096-word region of a workgroup.
constexpr int kAreaG8 = 128, kAreaG16 = 256, kAreaG32 = 512, kAreaWave = 1024, kAreaBlock = 4096;

// Partner rows per tile of each bin (rounds = rows per group in light bins).
__host__ __device__ inline int tile_pivots(int bin, int rounds) {
  switch (bin) {
    case BIN_GLOBAL:
    case BIN_BLOCK: return 1;
    case BIN_WAVE: return kBlock / 64;
    case BIN_G32: return (kBlock / 32) * rounds;
    case BIN_G16: return (kBlock / 16) * rounds;
    default: return (kBlock / 8) * rounds;
  }
}

// Rows per group in the tiles of a light bin of `rows` rows on a grid of
// `grid` workgroups: `most`, or fewer where the tiles would then not reach
// every workgroup (a mid-size graph's few thousand light rows would run on a
// few dozen of the 256 CUs).
__host__ __device__ inline int tile_rounds(int bin, int64_t rows, int64_t grid, int most) {
  const int64_t r = rows / (grid * tile_pivots(bin, 1));
  return (int)(r < 1 ? 1 : most > 0 && r > most ? most : most < 1 ? 1 : r);
}

// Counter words of a plan (uint32).  The tile queue heads, one per queue and
// XCD, are a cache line apart: heads that share a line are served one after
// another.
constexpr int kCntBinCount = 0;                   // [kNumBins]
constexpr int kCntFallback = kNumBins;            // hash builds that fell back to the tree
constexpr int kPlanWords = 32;                    // words up to here are read back
constexpr int kCntHeads = 32;                     // queue i, eighth e: word kCntHeads + kHeadStride * (8 i + e)
constexpr int kHeadStride = 32;
constexpr int kNumHeads = kNumBins + 2;           // a bin's; then the bitmap kernels' two
constexpr int kCoreHead = kNumBins;
constexpr int kNumCounters = kCntHeads + 8 * kHeadStride * kNumHeads;

// Partner rows.  Every DAG edge (u, v) is counted from the endpoint whose
// out-list is longer: its "owner" x keeps N+(x) as the LDS set and its
// "partner" p has N+(p) streamed through it, so each edge streams
// min(d+(u), d+(v)) ids instead of d+(v).  Owner of (u, v): u when
// d+(v) <= d+(u) (partner v), else v (partner u).  The partners of one
// owner x are consecutive in the partner-id array; x's list is cut into
// ceil(count / kPartnersPerRow) "partner rows" (vrow[k] = x, partner ids
// pci[vrp[k] .. vrp[k+1])), the unit of work of the count.
constexpr int kPartnersPerRow = TCH_PARTNERS_PER_ROW;

// Streamed ids are loaded kChunk at a time, so a load may begin at the last id
// of a colidx pool: pools are allocated with kCiPad ids past their end (their
// values never count).
constexpr int kChunk = 4;
constexpr int64_t kCiPad = kChunk;

// Rows of a graph with codes: every id of the list has one; none of them
// ranks below the row's own vertex.
constexpr uint8_t kClosed = 1, kOrdered = 2;

// 16-bit codes of vertices for the bitmap kernels.  A code's low 13 bits are
// a byte of the bitmap, its high 3 bits a bit of that byte; a graph of n
// vertices (at most kCoreIds) spreads them over 2^kb bytes, the fewest that
// hold n bits.  Vertex i's code is the bit-reversed low kb + 3 bits of
// i * kCodeMul (a bijection): the product's top bits pick the LDS bank, so
// ids that share low bits, as an R-MAT graph's hubs do, do not share banks.
// kNoCode is no vertex's code.
constexpr int kCoreByteBits = 13;
constexpr int64_t kCoreIds = 65535;
constexpr int kCoreChunk = 8;               // codes per load
constexpr int64_t kCorePad = 4096;          // codes allocated past a pool's end (see kCiPad)
constexpr int64_t kCorePool = (int64_t)1 << 30;  // ids of a pool with codes: byte offsets stay 32-bit
// Where the codes of the list of n ids at ci position p are: twice p, rounded
// up to a multiple of the largest power of two within n (at most a 128-byte
// line of codes).  That leaves every list inside [2p, 2p + 2n), so lists do
// not overlap, and long lists start on a cache line, short ones on the word
// that holds them (RMAT-22: the lines a count reads, 19.6 -> 17 GB).
__host__ __device__ inline uint32_t code_start(int64_t p, uint32_t n) {
  const uint32_t a = n >= 64 ? 64u : n >= 32 ? 32u : n >= 16 ? 16u : n >= 8 ? 8u : 1u;
  return ((uint32_t)p * 2u + a - 1u) & ~(a - 1u);
}
// Where a list of n ids at ci position p is in a pool of lists on lines: twice
// p, or the next 128-byte line where it would straddle one -- less than n ids
// further on, so lists stay inside [2p, 2p + 2n) and do not overlap.
__host__ __device__ inline int64_t line_start(int64_t p, int32_t n) {
  const int64_t s = 2 * p;
  return (s & 31) + n > 32 ? (s + 31) & -32 : s;
}
constexpr uint32_t kCodeMul = 0x9E37u;      // odd, near 2^16 / phi
__host__ __device__ constexpr uint32_t core_code(uint32_t i, int kb) {
  uint32_t r = i * kCodeMul;
  r = (r & 0x5555u) << 1 | (r >> 1 & 0x5555u);
  r = (r & 0x3333u) << 2 | (r >> 2 & 0x3333u);
  r = (r & 0x0F0Fu) << 4 | (r >> 4 & 0x0F0Fu);
  r = (r & 0x00FFu) << 8 | (r >> 8 & 0x00FFu);  // 16 bits reversed
  r >>= kCoreByteBits - kb;                     // kb + 3 bits reversed
  return (r >> kb) << kCoreByteBits | (r & ((1u << kb) - 1u));
}
constexpr uint16_t kNoCode = (uint16_t)core_code(65535, kCoreByteBits);
// The bitmap byte of the code in half `half` of a word: below 2^kb whatever the
// 16 bits are.  A load may hold what no list owns (the room between lists, what
// is past the pool's last), which is looked up like any code and not counted;
// with the 13 bits of the largest bitmap it would read past a smaller one.
__host__ __device__ inline uint32_t code_byte(uint32_t word, int half, int kb) {
  return (word >> (16 * half)) & ((1u << kb) - 1u);
}
// Smallest kb for n vertices (the bitmap is cleared 16 bytes per lane of a wave).
inline int core_bits(int64_t n) {
  int kb = 10;
  while (kb < kCoreByteBits && ((int64_t)8 << kb) < n) ++kb;
  return kb;
}

// One graph of a (possibly single-graph) count.
//   DAG: rowptr at rp_off of the rowptr pool (values relative to ci_off of
//        the colidx pool), n_rows rows; only rows [own_begin, own_end) have
//        their out-edges counted (a partition's owned range), other rows are
//        lists read through them (halo).
//   Partners: the graph's partner list references at pci_off of the
//        partner pool (as many slots as the DAG has ids).  Its partner rows
//        take slots [pr_base, pr_base + nv_max + 1) of the launch's VRow and
//        row-offset arrays; those slots are also the plan indices.
//   Build: the graph's n_rows + 1 slots of a partner build's per-row
//        scratch start at row_base, and its ids' slots of the build's
//        per-id scratch at eb (graphs in order, contiguous).
// List references (set and partners) and row offsets are absolute in their
// pools, so planning and counting never read this descriptor.
struct GraphDesc {
  int64_t rp_off;
  int64_t ci_off;
  int64_t pci_off;
  int64_t row_base;
  int64_t pr_base;
  int32_t n_rows;
  int32_t nv_max;
  int32_t own_begin;
  int32_t own_end;
  int64_t eb;
};

// Partner rows a graph of n rows and m DAG ids may need (it takes this
// many slots plus one).
inline int32_t partner_rows_max(int64_t n, int64_t m) {
  return (int32_t)(n + m / kPartnersPerRow + 1);
}

struct Tune {
  int32_t t_g8, t_g16, t_g32, t_wave, rounds;
  int32_t tree_only;   // 1: pivot sets are always LDS trees; 2: for sub-wave groups
  int32_t hash_kicks;  // evictions per hash insert before falling back to the tree
};

struct PlanBufs {
  uint16_t* bin_of;     // [P] work class << 3 | bin of each pivot (kNoBin: none)
  uint64_t* items;      // [P] (graph << 32 | partner row), ordered by (bin, plan index)
  uint32_t* blk;        // [kNumBins * nblk + 1] per-(bin, planning block) counts -> offsets
  int64_t* part;        // [scan_partials(kNumBins * nblk + 1)] scan partials
  uint32_t* counters;   // [kNumCounters]
  uint64_t* outs;       // [ngraphs] u64 counts, or a single graph's kOutWords words
};

// A single graph's count is summed in kOutSlots words a cache line apart:
// every workgroup ends with an add, and adds to one word are served one per
// ~12 ns (8192 waves: 0.1 ms).
constexpr int kOutSlots = 32, kOutStride = 16, kOutWords = kOutSlots * kOutStride;

// A batch of few graphs has the same trouble: every heavy row ends with an add
// to its graph's word, and the words of 16 graphs share a line (8 graphs R-MAT
// n=30000 of 1.2 M ids: 1.19 ms; so 0.42).  Words per graph: at most kOutSlots, at most
// kBatchWords in all; 1 (no slots) from kBatchGraphs on, whose adds are spread
// by the graphs themselves.
constexpr int kBatchGraphs = 64, kBatchWords = 512;
inline int batch_slots(int64_t graphs) {
  if (graphs >= kBatchGraphs) return 1;
  int s = kOutSlots;
  while (s > 1 && s * graphs > kBatchWords) s /= 2;
  return s;
}

// A list of the DAG as one word: offset in the colidx pool in the high 39
// bits, length in the low 25 (out-degrees are below 2^25 by the upload
// checks).
typedef uint64_t ListRef;
constexpr int kLenBits = 25;
__host__ __device__ inline ListRef list_ref(int64_t start, int64_t len) {
  return ((uint64_t)start << kLenBits) | (uint64_t)len;
}
// A partner's list reference has two more bits on top (offsets stay below
// 2^37): kRefClosed, every id of the list N+(v) of its edge's head v has a
// 16-bit code, so that the edge can be counted over codes; kRefSlot, during a
// build only.
constexpr ListRef kRefSlot = 1ull << 63, kRefClosed = 1ull << 62;
// (Tests of the marks look at the high word alone: 64-bit mask tests with a
// mask in registers have compiled wrongly, and cost more.)
__host__ __device__ inline uint32_t ref_marks(ListRef r, uint32_t mask) { return (uint32_t)(r >> 32) & mask; }
constexpr uint32_t kMarkClosed = (uint32_t)(kRefClosed >> 32);
// A closed edge's lists have at most kCoreIds ids, so its length field holds
// the length in 16 bits and, above them, how much of the list's codes can
// match: the codes are ordered by degree class, highest first, and the ids
// past the first part(r) of them rank below the edge's head, so none of them
// is in N+(head).
constexpr uint32_t kPartAll = 255;
__host__ __device__ inline ListRef closed_ref(int64_t start, int64_t len, uint32_t part) {
  return kRefClosed | ((uint64_t)start << kLenBits) | (uint64_t)(part << 16) | (uint64_t)len;
}
__host__ __device__ inline int32_t list_len(ListRef r) {
  return (int32_t)((uint32_t)r & (ref_marks(r, kMarkClosed) ? 0xFFFFu : (1u << kLenBits) - 1u));
}
// Codes to stream of a closed edge's list (part: 1/256 of its length, less 1).
__host__ __device__ inline uint32_t closed_len(ListRef r) {
  const uint32_t x = (uint32_t)r;
  return ((x & 0xFFFFu) * ((x >> 16 & 0xFFu) + 1u) + 255u) >> 8;
}
__host__ __device__ inline int64_t list_start(ListRef r) { return (int64_t)(r << 2 >> (kLenBits + 2)); }

// A partner row: the owner's list (the set; 0 for an unused slot), the
// total length of its partners' lists (saturated at 2^32 - 1; only compared
// with the bin thresholds) and its graph, or where some of a single graph's
// ids have codes (core 2) whether the row has edges marked kRefClosed
// (kRowClosed) and others (kRowOpen).
constexpr int32_t kRowClosed = 1, kRowOpen = 2;
struct VRow {
  ListRef set;
  uint32_t work;
  int32_t g;
};

// Outputs of a local count (one graph only).  pedge / pvid: DAG edge
// position and partner vertex of every partner entry (parallel to the
// partner pool); pown: owner vertex of every partner row (per plan index);
// ecount: per DAG edge position, |N+(u) ∩ N+(v)| of edge (u, v); vcount: per
// vertex, the triangles with a corner there.  All null in a plain count.
// Attribution modes of a local count: none (the plain count); every
// triangle to its DAG edge, its three corners (slot hit counters for the
// third) and, through the edges, the parts of a split (full); to its DAG
// edge only (edges); or only to the part of a split that computes it, one
// sum per partner row (parts: no per-edge or per-vertex output).
constexpr int kLocalNone = 0, kLocalFull = 1, kLocalEdges = 2, kLocalParts = 3;

struct LocalOut {
  const int64_t* pedge;
  const int32_t* pvid;
  const int32_t* pown;
  uint32_t* ecount;
  unsigned long long* vcount;
  const int32_t* bounds = nullptr;  // kLocalParts: split points [parts + 1]
  int32_t parts = 0;
  uint64_t* pe = nullptr;           // kLocalParts: per-part sums [parts], zeroed by the caller
};

struct LaunchArgs {
  const GraphDesc* descs;
  int32_t ngraphs;
  int64_t P;            // partner-row slots = plan indices (sum of nv_max + 1)
  const int64_t* rp;    // DAG rowptr pool
  const int32_t* ci;    // DAG colidx pool
  const int32_t* lines; // null, or the lists of ci on cache lines (line_start), for streaming
  const ListRef* pci;   // partner pool: each partner's list
  const int64_t* vrp;   // [P + 1] partner-row offsets into the partner pool
  const VRow* vrow;     // [P] partner rows
  const int32_t* nv;    // [ngraphs] partner rows in use
  Tune tune;
  PlanBufs bufs;
  LocalOut local;
  const uint8_t* own;   // one graph only: null, or per row 1 if it is a pivot row
  // Bitmap counting (see core_kernel): 16-bit codes of the ids of every list
  // (at code_start); 2^core_kb bytes hold the bitmap of any set of codes.
  const uint16_t* c16;
  int32_t core;         // 0: no codes; 1: every id has one; 2: edges marked kRefClosed can use them
  int32_t core_kb;
  int32_t wide_ids;     // 1 when ids reach 2^24: hash sets fold the high id bits into the bucket
  int32_t out_slots;    // kOutSlots where bufs.outs holds a single graph's slots, else 0
  // A batch's bitmap kernels: null (they add to bufs.outs), or slots[g * nslots + i]
  // a cache line apart, i < nslots (a power of two), added by launch_batch_sums.
  uint64_t* slots;
  int32_t nslots;
  int32_t many_light;   // a batch (whose rows per bin the host does not know): over kManyLight times as many
                        // rows of the light bins as of the wave bin, by the lists' lengths
  int32_t gbase;        // partner build of a segment of graphs: index of descs[0] among all graphs
};

// Ids at or above this need the folded hash (the bucket multiply reads 24 bits).
constexpr int64_t kNarrowIds = (int64_t)1 << 24;

// Planning blocks of a launch over P plan indices.
inline int64_t plan_blocks(int64_t P) { return (P + 255) / 256; }

// Scratch of a partner build over RP row slots (the graphs' n_rows + 1
// slots, concatenated in graph order from row_base 0).
// Partners a row owns through in-edges are counted in kXcds stripes:
// workgroup i updates stripe i mod kXcds, and the dispatcher places it on
// XCD i mod kXcds, so each stripe's counters and cursors are touched by one
// XCD only (a hub's in-edges then spread over kXcds cache lines).  Both
// build passes use the same grid, so an edge falls in the same stripe in
// each whatever the placement.
constexpr int kXcds = 8;

struct BuildBufs {
  int32_t* c1;          // [RP] atomic path: partners owned through out-edges
  int32_t* c2;          // [kXcds * RP] atomic path: partners owned through in-edges, per stripe;
                        // radix path: pairs per owner of the big fine buckets
  unsigned long long* cur;  // [kXcds * RP] atomic path: fill cursor of each stripe;
                            // radix path: pool cursor of each owner of the big fine buckets
  int64_t* off;         // [RP] partner offsets (exclusive scan over the row slots)
  int32_t* kc;          // [RP] partner rows per DAG row
  int64_t* voff;        // [RP] partner-row offsets (pool-global exclusive scan)
  int64_t* part;        // [scan_partials(max(RP, ...))] scan partials
  int64_t* pedge;       // null, or [partner pool]: DAG edge position of each partner entry
  int32_t* pvid;        // with pedge: [partner pool] partner vertex of each entry
  int32_t* pown;        // null, or (one graph) [P] owner vertex of each partner row
  uint16_t* codes;          // null, or where to write the codes of all ids (core_code, a.core_kb)
  int32_t* lines;           // null, or where to write the lists at line_start
  const uint8_t* closed;    // null, or (one graph) per row kClosed | kOrdered
  const uint8_t* lpart;     // with closed: per DAG id e = (u, v), the part of u's codes that rank with v or above
  // Radix transpose (null when the scratch has no per-id part).  Build space:
  // M ids, graph g's at eb; row slots: RP.
  int32_t* gid;         // [RP] graph of each row slot; ~graph when the row is not split
  int64_t* erow;        // [RP + 1] first build-space id of each row slot; erow[RP] = M
  ListRef* lref;        // [RP] each row slot's own list
  uint16_t* deg16;      // [RP] out-degree of each row slot, saturated at 65535
  int32_t* key;         // [M] owner of each id's pair (-1: none); after level 2, fine-bucket order
  ListRef* ref;         // [M] partner list of each pair, in the order of key
  int32_t* pkey;        // [M] level-1 (coarse-bucket) order of key
  ListRef* pref;        // [M] and of ref
  int64_t* bq;          // [nmp + 1] rows consumed before each split block
  uint32_t* cnt1;       // [kCoarse * nmp + 1] pairs per (coarse bucket, split block) -> positions
  uint32_t* cnt2;       // [kFine * nt2 + 1] pairs per (fine digit, level-2 tile) -> positions
  int64_t* tstart;      // [kCoarse + 1] first level-2 tile of each coarse bucket
  int64_t* chstart;     // [kMaxFineBuckets + 1] first chunk of each big fine bucket
  int64_t* fst;         // [kMaxFineBuckets + 1] first pair of each fine bucket
  unsigned long long* wq;   // [RP] radix path: each owner's work (its partners' list lengths); else null
  // Radix path with pedge (a local rebuild of one graph): each pair's DAG id
  // position rides along the two levels (e1, e2) and lands in pedge beside
  // the partner's list; esrc[e] = the row of DAG id e gives the partner
  // vertices (pvid).  Either path of a local rebuild (the radix split, or
  // the atomic fill) sets bit 31 of esrc[e] where the edge's head owns it.
  // Null otherwise.
  uint32_t* e1;         // [M] level-1 order of the pairs' id positions
  uint32_t* e2;         // [M] level-2 (fine-bucket) order
  int32_t* esrc;        // [M]
  int64_t rows;         // capacity: row slots
  int64_t ids;          // capacity: ids
};
int64_t scan_partials(int64_t n);

// Radix transpose geometry.  Owner slots fall in fine buckets of 2^fs slots
// (at most kMaxFineBuckets), 64 fine buckets to a coarse bucket.  Split
// blocks take kMP merge-path items (row ends and ids), level-2 tiles kTile
// pairs.  A fine bucket of at most `cap` pairs is sorted whole in LDS; a
// bigger one goes by chunks of `chunk` pairs.  Dynamic LDS of the final
// passes stays within kRadixLds.
constexpr int kMP = 4096;
constexpr int kMPPer = kMP / kBlock;
constexpr int kTile = 4096;
constexpr int kTilePer = kTile / kBlock;
constexpr int kCoarse = 160;
constexpr int kFine = 64;
constexpr int kMaxFineBuckets = kCoarse * kFine;
constexpr int kMinFineShift = 5;
constexpr int kMaxFineShift = 11;
constexpr int kMaxFineOwners = 1 << kMaxFineShift;
constexpr int64_t kFineCapMax = 8192;
constexpr int64_t kChunkMax = 4096;
constexpr int kFinPer = (int)(kFineCapMax / kBlock);  // pairs per thread of a small bucket
constexpr int kChunkPer = (int)(kChunkMax / kBlock);  // pairs per thread of a chunk
constexpr int64_t kRadixLds = 64512;  // 63 KB: room for the kernels' static LDS within 64 KB
inline size_t radix_final_lds(int fs, int cap) { return 20 * ((size_t)1 << fs) + 4 * (size_t)cap; }
inline size_t radix_place_lds(int fs, int chunk) { return 24 * ((size_t)1 << fs) + 4 * (size_t)chunk; }
struct RadixGeom {
  int fs, nf, nc;
  int64_t nmp, nt2, nch;
  int cap, chunk;
};
// False when RP or M is beyond the radix path (the atomic path then builds).
inline bool radix_geom(int64_t RP, int64_t M, RadixGeom& x) {
  if (RP <= 0 || RP >= ((int64_t)1 << 31) || M < 0 || M >= ((int64_t)1 << 32)) return false;
  int fs = kMinFineShift;
  while (fs <= kMaxFineShift && ((RP + ((int64_t)1 << fs) - 1) >> fs) > kMaxFineBuckets) ++fs;
  if (fs > kMaxFineShift) return false;
  const int64_t no = (int64_t)1 << fs;
  x.fs = fs;
  x.nf = (int)((RP + no - 1) >> fs);
  x.nc = (x.nf + kFine - 1) / kFine;
  x.nmp = (RP + M + kMP - 1) / kMP;
  x.nt2 = (M + kTile - 1) / kTile + x.nc;
  const int64_t cap = (kRadixLds - 20 * no) / 4 / 256 * 256, chunk = (kRadixLds - 24 * no) / 4 / 256 * 256;
  x.cap = (int)(cap < kFineCapMax ? cap : kFineCapMax);
  x.chunk = (int)(chunk < kChunkMax ? chunk : kChunkMax);
  x.nch = (M + x.chunk - 1) / x.chunk + x.nf;
  return true;
}
// Upper bounds of the per-build arrays for up to `rows` slots and `ids` ids.
inline int64_t radix_split_blocks(int64_t rows, int64_t ids) { return (rows + ids + kMP - 1) / kMP; }
inline int64_t radix_tiles2(int64_t ids) { return (ids + kTile - 1) / kTile + kCoarse; }

// Builds the partner lists, rows and counts of every graph of `a` (descs,
// rp, ci, P as for a count; pci/vrp/vrow/nv are written); RP = sum of
// n_rows + 1 over the graphs, M = sum of their ids.  With the per-id
// scratch (b.key) and no local outputs (b.pedge null) the in-edge partners
// are placed by a bucketed transpose; otherwise by per-edge atomics.
hipError_t launch_partners(const LaunchArgs& a, int64_t RP, int64_t M, const BuildBufs& b, hipStream_t s);

// Launchers (stream-ordered; return the launch status).
hipError_t launch_zero(void* p, int64_t words32, hipStream_t s);

// One request's CSR on its way from pinned host memory (src, mapped for the
// device) to its extent of the device pool (dst): `bytes`, a multiple of 4,
// both ends 16-byte aligned; chunks [first, first + ceil(bytes / kStageChunk))
// of the staging copy move it.
struct StageCopy {
  const char* src;
  char* dst;
  int64_t bytes;
  int64_t first;
};
constexpr int64_t kStageChunk = (int64_t)64 << 10;  // bytes per chunk of the staging copy
inline int64_t stage_blocks(int64_t bytes) { return (bytes + kStageChunk - 1) / kStageChunk; }
// All copies of a launch in one kernel (`chunks` = the sum of their chunks;
// copies on the device, ordered by first), on at most kStageGrid workgroups.
constexpr int64_t kStageGrid = 128;
hipError_t launch_stage_copy(const StageCopy* copies, int32_t n, int64_t chunks, hipStream_t s);
// Re-arms a kept plan for another count: tile queue heads and the fallback
// counter to 0 (bin counts kept), outs[0..nouts) to 0.
hipError_t launch_rearm(uint32_t* counters, uint64_t* outs, int32_t nouts, hipStream_t s);
// The end of a single graph's count: its sum (of kOutSlots words) to host[0]
// and its hash fallbacks to host[1] (pinned memory, by its device address),
// and a rearm on the way, so that another count with the plan needs none.
// One launch instead of two copies and the next call's rearm, each ~5 us and
// as much again between launches (R-MAT n=30011: 85 -> 72 us a call, R-MAT-18
// 215 -> 200).
hipError_t launch_finish(uint32_t* counters, uint64_t* outs, uint64_t* host, hipStream_t s);
// outs[g] += the slots of graph g, for every graph of a batch with slots.
hipError_t launch_batch_sums(const LaunchArgs& a, hipStream_t s);
hipError_t launch_plan(const LaunchArgs& a, hipStream_t s);
// Bytes of a pool of ids with its lists on lines.
inline size_t line_bytes(int64_t ids) { return sizeof(int32_t) * (size_t)(2 * ids + kCiPad); }
// Bytes of the codes of a pool of ids.
inline size_t code_bytes(int64_t ids) { return sizeof(uint16_t) * (size_t)(2 * ids + kCorePad); }
// Codes for a graph of more than kCoreIds rows: the at most kCoreIds vertices
// of highest degree (in the uploaded rows) get one.  c16: the codes of each
// row's ids, at code_start; rows of more than kRankLeast ids have
// theirs in order of degree class, highest first, ids without a code last.
// closed[v]: kClosed | kOrdered; part[e]: see BuildBufs::lpart; *closed_edges = ids
// that name closed rows.  scratch: big_codes_bytes(n, m) bytes.
constexpr int kRankLeast = 32;
constexpr int kDegBucketBits = 14;
constexpr int64_t kDegBuckets = 1024;
inline bool big_codes_fit(int64_t n, int64_t m) {
  return n > kCoreIds && (n + ((int64_t)1 << kDegBucketBits) - 1) >> kDegBucketBits <= kDegBuckets && m > 0 && m < kCorePool;
}
int64_t big_codes_bytes(int64_t n, int64_t m);
hipError_t launch_big_codes(const int64_t* rp, const int32_t* ci, int64_t n, int64_t m, char* scratch, uint16_t* c16,
                            uint8_t* closed, uint8_t* part, unsigned long long* closed_edges, int cus, hipStream_t s);
// The hash kernel over all bins at full residency (grid > 0 overrides the size).
hipError_t launch_count(const LaunchArgs& a, int cus, int grid, hipStream_t s);
// A count with codes has up to three parts, each one persistent launch; they
// run side by side on streams of their own: the bitmap kernels of the rows
// that take a workgroup (kPartBlock) and a wave (kPartWave), and the hash
// kernel of all others (kPartHash; without codes of all rows, with codes of
// some ids the other edges of the heavy rows as well).  rows: per bin, null
// when the host does not know them; parts without rows launch nothing.
// The bitmap kernels take the bins that keep a wave busy, or all bins of a
// graph with few light rows (at most kCoreLightRows), where one more wide
// launch beats narrow groups (R-MAT n=30011 d=24: 0.17 -> 0.10 ms, ER n=32000
// d=16: 75 -> 45 us, R-MAT n=65003 d=32: 121 -> 82; ER n=40000 d=16 with all
// rows so: 78 -> 131) -- a wave per light row is slower from a few rows per
// resident wave on (the batch of 512 graphs, 215 K rows of the 32-lane bin:
// 0.53 ms there, 0.64 ms here).
constexpr int64_t kCoreLightRows = 32768;
// launch_core's comment has both sides measured.
constexpr int64_t kManyLight = 8;
constexpr int kPartBlock = 0, kPartWave = 1, kPartHash = 2, kCountParts = 3;
bool part_empty(const LaunchArgs& a, int part, const int64_t* rows);
hipError_t launch_count_part(const LaunchArgs& a, int cus, int grid, int part, const int64_t* rows, hipStream_t s);

// own: null, or per row 1 if it is a pivot row (rows outside
// [row_begin, row_end) are never pivots).  out must hold 0.  host: null, or
// where the last workgroup stores the sum (pinned memory, by its device
// address); out is then kOutWords words, left 0.  For sums below 2^kDoneShift
// and grids below 2^(64 - kDoneShift).
constexpr int kDoneShift = 48;
// single: ids are loaded one at a time, not kChunk (see tcr::DagShape::short_lists).
hipError_t launch_plain(const int64_t* rp, const int32_t* ci, int32_t row_begin, int32_t row_end,
                        const uint8_t* own, uint64_t* out, int grid, bool single, hipStream_t s,
                        uint64_t* host = nullptr);
// Count of one graph that also fills a.local: same plan, the local variants
// of the hash kernel over all bins.  mode kLocalFull: ecount and vcount (zeroed by the
// caller); kLocalEdges: ecount only (the kernels keep no slot hit counters:
// less LDS, more waves per SIMD); kLocalParts: pe only (bounds, parts, pe
// set; the plain count's kernels, each row's hits added to its owner's part).
hipError_t launch_count_local(const LaunchArgs& a, int cus, int mode, hipStream_t s);
// Per-graph table of launch_local_parts over rows [0, n): esrc[e] = the row
// u of DAG edge e = (u, v); the local rebuild (launch_build with pedge and
// esrc) then sets bit 31 where v owns the edge, i.e. d+(u) < d+(v).
hipError_t launch_local_prep(const int64_t* rp, int64_t n, int32_t* esrc, hipStream_t s);
// After launch_count_local: sums the ecount of every edge in [e0, e1) (the
// counted rows' edges; uncounted ones hold 0) into pe[owner] by the
// reference push/pull rule over the split bounds[0..parts] (1 <= parts <=
// kMaxParts, bounds[0] = 0, bounds[parts] = n, non-decreasing; pe zeroed by
// the caller).
constexpr int kMaxParts = 1024;
hipError_t launch_local_parts(const int32_t* ci, const int32_t* esrc, int64_t n, int64_t e0, int64_t e1,
                              const uint32_t* ecount, const int32_t* bounds, int32_t parts, unsigned long long* pe,
                              int cus, hipStream_t s);
hipError_t launch_copy(const void* src, void* dst, int64_t bytes, int grid, hipStream_t s);
// sink: grid * kBlock words (never written for a byte-filled source).
hipError_t launch_read(const void* src, int64_t bytes, uint32_t* sink, int grid, hipStream_t s);
// Resident workgroups per CU of the persistent and plain kernels.
int count_blocks_per_cu();
int plain_blocks_per_cu();

// Static plan scratch of the allocation-free count (tc_count_noalloc): a
// count over at most kNoAllocSlots plan indices keeps its bins, items, scan
// and counters there instead of in allocated memory.
constexpr int64_t kNoAllocSlots = (int64_t)1 << 21;
// Byte size of the scratch and the plan buffers laid out in it (base = its
// device address, from noalloc_scratch_address).
int64_t noalloc_scratch_bytes();
PlanBufs noalloc_plan_bufs(void* base);
// Device address of the scratch on the current device.
hipError_t noalloc_scratch_address(void** ptr);

}  // namespace tck
