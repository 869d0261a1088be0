// Internal state of the device library shared by tc_runtime.cpp, tc_copy.cpp,
// tc_batch.cpp, tc_server.cpp and tc_tune.cpp.
#pragma once

#include <hip/hip_runtime.h>

#include <chrono>
#include <memory>
#include <mutex>
#include <string>
#include <unordered_set>
#include <vector>

#include "tc.h"
#include "tc_kernels.hpp"

namespace tcr {

// Records the calling thread's error text and returns `st`.
tc_status fail(tc_status st, const std::string& msg);
// Called from a catch block: turns the exception in flight into a status, so
// that no C++ exception crosses the C ABI (a failed host allocation is
// TC_ENOMEM).
tc_status caught() noexcept;

#define TC_HIP_TRY(expr)                                                              \
  do {                                                                                \
    hipError_t e_ = (expr);                                                           \
    if (e_ != hipSuccess)                                                             \
      return ::tcr::fail(TC_EDEVICE, std::string(#expr) + ": " + hipGetErrorString(e_)); \
  } while (0)

inline double now_ms() {
  using namespace std::chrono;
  return duration<double, std::milli>(steady_clock::now().time_since_epoch()).count();
}

// Device allocation with an out-of-memory status instead of an abort.
tc_status dev_alloc(void** p, size_t bytes, const char* what);
void dev_free(void* p);

// Plan scratch (binning output and counters) sized for P pivots / k outputs.
struct PlanScratch {
  uint16_t* bin_of = nullptr;
  uint64_t* items = nullptr;
  uint32_t* blk = nullptr;
  int64_t* part = nullptr;
  int64_t cap = 0;
  uint32_t* counters = nullptr;
  uint64_t* outs = nullptr;
  int64_t outs_cap = 0;
  tc_status ensure(int64_t pivots, int64_t nouts);
  void release();
  tck::PlanBufs bufs() const { return tck::PlanBufs{bin_of, items, blk, part, counters, outs}; }
  // Device bytes per plan index, for footprint estimates.
  static int64_t bytes_for(int64_t pivots);
};

// Partner structure of pooled graphs (see tck::GraphDesc): partner list
// references (as many as the colidx pool has ids), partner-row slots (and
// one more row offset), rows in use per graph.
struct Partners {
  tck::ListRef* pci = nullptr;
  int64_t* vrp = nullptr;
  tck::VRow* vrow = nullptr;
  int32_t* nv = nullptr;
  int64_t bytes = 0;
  tc_status alloc(int64_t ci_slots, int64_t row_slots, int32_t ngraphs);
  static int64_t vrow_bytes(int64_t row_slots) { return (int64_t)sizeof(tck::VRow) * row_slots; }
  void release();
  void into(tck::LaunchArgs& a) const {
    a.pci = pci;
    a.vrp = vrp;
    a.vrow = vrow;
    a.nv = nv;
  }
  static int64_t bytes_for(int64_t ci_slots, int64_t row_slots, int32_t ngraphs);
};

// Buffers of a local count of one graph: the partner entries' DAG edge
// positions and partner vertices, per-edge and per-vertex counts, and
// per-part sums with their split points (a call with part sums alone
// allocates only those two; the partner rows' owners belong to the graph).
struct LocalBufs {
  int64_t* pedge = nullptr;
  int32_t* pvid = nullptr;
  uint32_t* ecount = nullptr;
  unsigned long long* vcount = nullptr;
  unsigned long long* pe = nullptr;  // [tck::kMaxParts]
  int32_t* bounds = nullptr;         // [tck::kMaxParts + 1]
  int32_t* esrc = nullptr;           // [nnz] row u of each DAG edge (u, v) | (d+(u) < d+(v)) << 31
  int64_t bytes = 0;
  void release();
};

// Temporary arrays of a partner build over RP rowptr slots and M DAG ids
// (the ids' part -- 24 bytes per id -- serves the bucketed transpose; with
// ids = 0 only the per-edge atomic path is available).
struct BuildScratch {
  char* mem = nullptr;
  int64_t cap = 0;
  char* emem = nullptr;  // the radix path's pair id positions (local rebuilds)
  int64_t ecap = 0;
  tck::BuildBufs b{};
  tc_status ensure(int64_t rp_slots, int64_t ids);
  // After ensure: room for the pairs' id positions (b.e1, b.e2) of ids ids.
  tc_status ensure_edges(int64_t ids);
  void release();
  static int64_t bytes_for(int64_t rp_slots, int64_t ids);
};

// Builds the partners of the graphs of `a` (descs on the device, pools and
// P set; RP row slots, M ids in all) on stream s.  Stream-ordered, no sync.
// loc: null, or where to write each partner entry's DAG edge position and
// partner vertex and each partner row's owner (pedge, pvid, pown).
tc_status launch_build(const tck::LaunchArgs& a, int64_t RP, int64_t M, BuildScratch& bs, hipStream_t s,
                       const LocalBufs* loc = nullptr, int32_t* pown = nullptr, const uint8_t* closed = nullptr,
                       const uint8_t* part = nullptr, uint16_t* codes = nullptr, int32_t* lines = nullptr);

// Large copies from the device to pageable host memory, by way of a ring of
// pinned buffers that a few threads empty while the copy engine fills the
// others.  The runtime's own path copies out on one thread, 10 GB/s where the
// process has not touched the memory yet (63 MB of edge counts on MI355X, PCIe
// 5 x16: 6.0 ms; so 1.9).  The threads live for one copy, the ring (16 MB) for
// its owner.  Copies below kLeast bytes take the runtime's path: below that
// starting the threads takes longer than they save.  (Uploads gain nothing:
// the runtime copies those at 24 GB/s, and a one-shot call of RMAT-20, which
// has to make the ring, went from 8.8 to 12 ms.)
struct Stager {
  static constexpr size_t kLeast = (size_t)8 << 20, kChunk = (size_t)4 << 20;
  static constexpr int kBufs = 4, kSlices = 8, kThreads = 8;
  char* mem = nullptr;
  hipEvent_t ev[kBufs] = {};
  // Synchronous; on stream s, so after what s has been given before.
  hipError_t to_host(void* dst, const void* src, size_t bytes, hipStream_t s);
  void release();

 private:
  hipError_t ring();
};

// What an upload's choices go by: one pass over the row offsets.
struct DagShape {
  int64_t max_out = 0;
  uint64_t squares = 0;  // sum of the out-degrees' squares: bounds the ids a count streams
  double mean = 0;       // squares per id: the mean length of the list an id is in
  double skew = 0;       // squares against those of lists of equal length
  DagShape() = default;
  explicit DagShape(const tc_csr_view& dag);  // (rowptr checked; squares stay below 2^64 where max_out passes)
  // ER graphs of mean out-degree 2 to 100 have 1.1 to 1.5, R-MAT graphs 3.5 and more.
  bool flat() const { return skew < 2.0; }
  // The plain kernel's loads of four ids waste much of themselves on short
  // lists; in uneven graphs most ids streamed are in longer ones (us, ids
  // loaded four at a time / singly: ER of mean 5.9, n=1000000 590 / 519, of
  // 9.5, n=1500000 930 / 852, of 14.3, n=1000000 687 / 689, of 24.1, n=600000
  // 554 / 623; R-MAT of 8.3, n=10000 25.6 / 27.0).
  bool short_lists() const { return flat() && mean < 12.0; }
};

// Threads that copy a server request of `bytes`, of `clients` that are copying
// one (this one among them).  One thread moves ~9 GB/s, so a request is split
// from 1 MB a thread on; but the clients share kCopyThreads, since more threads
// than that only cost their start (8 clients with requests of 1.2 M ids on
// MI355X: a thread per MB each 0.60 ms a submit, one each 0.31; one client
// 0.25 -> 0.18).  Requests of 16 MB and more have up to 4 whatever the others
// do: their copies outlast that.
constexpr size_t kCopySplit = (size_t)1 << 20, kCopySplitLarge = (size_t)8 << 20;
constexpr int kCopyThreads = 8, kCopyThreadsLarge = 4;
inline int copy_threads(size_t bytes, int clients) {
  const int64_t by_size = (int64_t)(bytes / kCopySplit), large = (int64_t)(bytes / kCopySplitLarge);
  const int64_t share = by_size < kCopyThreads / clients ? by_size : kCopyThreads / clients;
  const int64_t n = large < kCopyThreadsLarge ? large : kCopyThreadsLarge;
  return (int)(n > share ? n : share > 1 ? share : 1);
}

// Makes ctx's device current for the scope of one API call.
struct DeviceGuard {
  int prev = -1;
  explicit DeviceGuard(int dev) {
    if (hipGetDevice(&prev) != hipSuccess) prev = -1;
    if (prev != dev) (void)hipSetDevice(dev);
  }
  ~DeviceGuard() {
    int cur = -1;
    if (prev >= 0 && hipGetDevice(&cur) == hipSuccess && cur != prev) (void)hipSetDevice(prev);
  }
};

tck::Tune to_kernel_tune(const tc_tune& t);
tc_status check_tune(const tc_tune& t);
tc_tune default_tune();

// A graph or a batch that holds device memory its counts can do without: the
// 16-bit codes and the lists on lines.  Such memory is taken last, and when a
// context runs out it gives all of it back and tries again, so that it never
// takes the place of what a call needs.
struct Spare {
  // Gives it back; the context's streams are idle.
  virtual void shed() = 0;

 protected:
  ~Spare() = default;
};
bool shed_spares(tc_ctx* ctx);  // all of ctx's; whether there were any
// f's status; when f ran out of memory and spares could be shed, that of
// another try.  f leaves nothing behind when it fails.
template <class F>
tc_status with_room(tc_ctx* ctx, F f) {
  const tc_status st = f();
  return st == TC_ENOMEM && shed_spares(ctx) ? f() : st;
}

}  // namespace tcr

struct tc_ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  // A count's parts past the first run on side streams beside `stream`
  // (default priority); join[i]: side stream i done, fork: side streams may
  // start (events without timing).
  static constexpr int kSides = 2;
  hipStream_t side[kSides] = {};
  hipEvent_t join[kSides] = {};
  hipEvent_t fork = nullptr;
  hipEvent_t ev[4] = {nullptr, nullptr, nullptr, nullptr};
  int cus = 0;
  int count_grid = 0;   // full-residency grid of the persistent kernel
  int plain_grid = 0;   // full-residency grid of the plain kernel
  tc_tune tune{};
  std::recursive_mutex mu;
  std::string name;
  tcr::PlanScratch scratch;
  tcr::Stager stager;
  std::unordered_set<tcr::Spare*> spares;  // the graphs and batches that hold any
  uint64_t* pinned = nullptr;  // 256 B: a build's results and copied counts, plan counters, a count's sum
  uint64_t* pinned_dev = nullptr;  // its device address
  void* noalloc = nullptr;     // device address of the static scratch of tc_count_noalloc
  // device: the single-launch count's kOutWords words, which every call
  // leaves 0 (plain_dirty: unless it did not finish); then an upload's word
  uint64_t* plain_out = nullptr;
  bool plain_dirty = false;
  // tc_count_csr's copy of a small graph: rowptr, then colidx at the next
  // 256-byte boundary (grow-only, kept until destroy)
  uint8_t* once_dev = nullptr;
  size_t once_cap = 0;  // bytes
  int grid() const { return tune.grid > 0 ? tune.grid : count_grid; }
};

struct tc_graph final : tcr::Spare {
  tc_ctx* ctx = nullptr;
  int64_t* rp = nullptr;
  int32_t* ci = nullptr;
  int32_t n = 0;
  int64_t nnz = 0;
  int32_t row_begin = 0, row_end = 0;
  int64_t edge_begin = 0, edge_end = 0;  // DAG edge positions of rows [row_begin, row_end)
  uint8_t* own = nullptr;                 // null, or per row 1 if it is a pivot row
  int32_t* lines = nullptr; // ci with its lists on cache lines (null: none)
  uint16_t* c16 = nullptr;  // 16-bit codes of ci for the bitmap kernels (null: none)
  uint8_t* closed = nullptr;  // with c16, over kCoreIds rows: tck::BuildBufs::closed
  uint8_t* part = nullptr;    // with closed: tck::BuildBufs::lpart
  bool coded = false;         // whether enough edges can use the codes
  int64_t spare_bytes = 0;    // of those four
  void drop_codes() {
    tcr::dev_free(c16);
    tcr::dev_free(closed);
    tcr::dev_free(part);
    c16 = nullptr;
    closed = part = nullptr;
    coded = false;
  }
  void shed() override {
    drop_codes();
    tcr::dev_free(lines);
    lines = nullptr;
    bytes -= spare_bytes;
    spare_bytes = 0;
  }
  int32_t* pown = nullptr;  // [nv_max + 1] owner vertex of each partner row, written by every build
  int32_t max_out = 0;
  bool short_lists = false;  // DagShape::short_lists
  tcr::Partners partners;
  tcr::LocalBufs local;
  int32_t nv_max = 0;   // partner rows it may need (nv_max + 1 slots = plan indices)
  int32_t nv = 0;       // partner rows in use
  double build_ms = 0;  // partner build time on the device
  tck::GraphDesc* d_desc = nullptr;
  int64_t bytes = 0;
  // The binned count's plan, kept across calls: valid for plan_tune; its
  // rows per bin (which size the launches) on the host.
  tcr::PlanScratch plan;
  bool plan_valid = false;
  bool plan_armed = false;  // its queue heads and sums are 0
  tc_tune plan_tune{};
  int64_t plan_bins[tck::kNumBins] = {};
};
