// A stand-in for the GPU behind the device library's host code: device memory
// is host memory under a budget, copies are memcpy, streams run at once, and
// the kernel launches do nothing but note what they were given.  Linked with
// csrc/hip's .cpp files, so that their allocation order, fallbacks and routes
// can be tested on the CPU.  Counts are 0 throughout.
//
//   fake_device SCENARIO [arguments]   exits 0 when the scenario holds
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <mutex>
#include <thread>

#include "tc_internal.hpp"

// ---- device memory -----------------------------------------------------------
static std::mutex g_mu;
static std::map<void*, size_t> g_size;
static size_t g_used = 0, g_peak = 0, g_budget = ~(size_t)0;
static std::function<bool(size_t)> g_deny;  // sizes that are never to be had

extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
  std::lock_guard<std::mutex> lk(g_mu);
  if (g_used + n > g_budget || (g_deny && g_deny(n))) return hipErrorOutOfMemory;
  *p = std::calloc(1, n + 64);
  g_size[*p] = n;
  g_used += n;
  g_peak = std::max(g_peak, g_used);
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  std::lock_guard<std::mutex> lk(g_mu);
  auto it = g_size.find(p);
  if (it == g_size.end()) std::abort();  // freed twice, or never allocated
  g_used -= it->second;
  g_size.erase(it);
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return (*p = std::calloc(1, n)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipHostFree(void* p) { return std::free(p), hipSuccess; }
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned) { return *d = h, hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { return std::memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) { return std::memcpy(d, s, n), hipSuccess; }
hipError_t hipMemset(void* d, int v, size_t n) { return std::memset(d, v, n), hipSuccess; }
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { return std::memset(d, v, n), hipSuccess; }
// ---- streams, events, graphs, devices ------------------------------------------
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return *s = (hipStream_t)std::malloc(1), hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { return std::free(s), hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return *e = (hipEvent_t)std::malloc(1), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { return std::free(e), hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 0, hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { return *g = (hipGraph_t)std::malloc(1), hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t, hipGraphNode_t*, char*, size_t) { return *x = (hipGraphExec_t)std::malloc(1), hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t x) { return std::free(x), hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t g) { return std::free(g), hipSuccess; }
hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) { return std::memset(p, 0, sizeof *p), p->multiProcessorCount = 256, hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
}

// ---- launches -----------------------------------------------------------------
static tck::BuildBufs g_build;           // of the last partner build
static unsigned long long g_closed = 0;  // what launch_big_codes reports
static int g_big_codes = 0;              // its launches
static tck::LaunchArgs g_args;           // of the last count
static int g_sums = 0;                   // launches that add a batch's slots
static bool g_single = false, g_direct = false;  // of the last plain launch
static int g_launches = 0;               // plain, zero and rearm launches
namespace tck {
int64_t scan_partials(int64_t n) { return n / 1024 + 2; }
int64_t big_codes_bytes(int64_t n, int64_t m) { return 12 * n + 2 * m; }
hipError_t launch_big_codes(const int64_t*, const int32_t*, int64_t, int64_t, char*, uint16_t*, uint8_t*, uint8_t*,
                            unsigned long long* closed, int, hipStream_t) {
  return *closed = g_closed, ++g_big_codes, hipSuccess;
}
hipError_t launch_partners(const LaunchArgs&, int64_t, int64_t, const BuildBufs& b, hipStream_t) { return g_build = b, hipSuccess; }
hipError_t launch_zero(void* p, int64_t n, hipStream_t) { return ++g_launches, std::memset(p, 0, 4 * (size_t)n), hipSuccess; }
hipError_t launch_stage_copy(const StageCopy*, int32_t, int64_t, hipStream_t) { return hipSuccess; }
hipError_t launch_rearm(uint32_t*, uint64_t*, int32_t, hipStream_t) { return hipSuccess; }
hipError_t launch_finish(uint32_t*, uint64_t*, uint64_t* host, hipStream_t) { return host[0] = host[1] = 0, hipSuccess; }
hipError_t launch_plan(const LaunchArgs& a, hipStream_t) { return g_args = a, hipSuccess; }
hipError_t launch_count(const LaunchArgs& a, int, int, hipStream_t) { return g_args = a, hipSuccess; }
bool part_empty(const LaunchArgs&, int, const int64_t*) { return false; }
hipError_t launch_count_part(const LaunchArgs& a, int, int, int, const int64_t*, hipStream_t) { return g_args = a, hipSuccess; }
hipError_t launch_plain(const int64_t*, const int32_t*, int32_t, int32_t, const uint8_t*, uint64_t*, int, bool single, hipStream_t, uint64_t* host) {
  return g_single = single, g_direct = host != nullptr, ++g_launches, hipSuccess;
}
hipError_t launch_count_local(const LaunchArgs& a, int, int, hipStream_t) { return g_args = a, hipSuccess; }
hipError_t launch_local_prep(const int64_t*, int64_t, int32_t*, hipStream_t) { return hipSuccess; }
hipError_t launch_local_parts(const int32_t*, const int32_t*, int64_t, int64_t, int64_t, const uint32_t*, const int32_t*, int32_t, unsigned long long*, int, hipStream_t) { return hipSuccess; }
hipError_t launch_copy(const void*, void*, int64_t, int, hipStream_t) { return hipSuccess; }
hipError_t launch_read(const void*, int64_t, uint32_t*, int, hipStream_t) { return hipSuccess; }
hipError_t launch_batch_sums(const LaunchArgs& a, hipStream_t) { return ++g_sums, g_args = a, hipSuccess; }
int count_blocks_per_cu() { return 4; }
int plain_blocks_per_cu() { return 4; }
hipError_t noalloc_scratch_address(void** p) { return *p = nullptr, hipSuccess; }
PlanBufs noalloc_plan_bufs(void*) { return PlanBufs{}; }
}  // namespace tck

// ---- graphs ---------------------------------------------------------------------
struct Dag {
  std::vector<int64_t> rp;
  std::vector<int32_t> ci;
  tc_csr_view view() const { return tc_csr_view{rp.data(), ci.data(), (int32_t)rp.size() - 1, (int64_t)ci.size()}; }
};
// n rows; the first `rows` have `d` ids each, the next `hubs` have `long_d`.
static Dag make(int32_t n, int32_t rows, int32_t d, int32_t hubs = 0, int32_t long_d = 0) {
  Dag g;
  g.rp.assign((size_t)n + 1, 0);
  for (int32_t v = 0; v < n; ++v) {
    const int32_t k = v < rows ? d : v < rows + hubs ? long_d : 0;
    for (int32_t i = 0; i < k; ++i) g.ci.push_back(n - k + i);
    g.rp[(size_t)v + 1] = (int64_t)g.ci.size();
  }
  return g;
}

#define CHECK(x)                                                              \
  do {                                                                        \
    if (!(x)) {                                                               \
      std::printf("line %d: %s (%s)\n", __LINE__, #x, tc_last_error(nullptr)); \
      std::exit(1);                                                           \
    }                                                                         \
  } while (0)

struct Ctx {
  tc_ctx* c = nullptr;
  Ctx() { CHECK(tc_ctx_create(0, &c) == TC_OK); }
  ~Ctx() { tc_ctx_destroy(c); }
  operator tc_ctx*() const { return c; }
};

// ---- scenarios --------------------------------------------------------------------

// A graph counted once gets no lines, and codes only where one count repays
// them; a resident graph gets both.
static void one_shot(int, char**) {
  Ctx ctx;
  uint64_t total;
  const Dag flat = make(140000, 139000, 17), skewed = make(140000, 20000, 10, 2000, 500),
            heavy = make(140000, 40000, 20, 600, 10000);
  g_closed = ~0ull >> 3;
  auto once = [&](const Dag& g) {
    const tc_csr_view v = g.view();
    g_big_codes = 0;
    CHECK(tc_count_csr(ctx, &v, TC_CHECK_SHAPE, &total, nullptr) == TC_OK);
    return g_big_codes;
  };
  CHECK(once(flat) == 0 && !g_build.lines && !g_build.codes && !g_args.c16);
  CHECK(once(skewed) == 0 && !g_build.lines && !g_args.c16 && g_args.core == 0);
  CHECK(once(heavy) == 1 && g_args.c16 && g_args.core == 2);
  const Dag few = make(60000, 50000, 70);  // every id has a code: written on the way, in one shot too
  CHECK(once(few) == 0 && g_build.codes && g_args.core == 1);
  for (uint32_t hint : {0u, (uint32_t)TC_UPLOAD_ONCE}) {
    const std::vector<uint8_t> owned(140000, 1);
    for (int kind = 0; kind < 2; ++kind) {
      auto upload = [&](const Dag& g, tc_graph** dg) {
        const tc_csr_view v = g.view();
        return kind ? tc_graph_upload_rows(ctx, &v, owned.data(), TC_CHECK_SHAPE | hint, dg)
                    : tc_graph_upload(ctx, &v, TC_CHECK_SHAPE | hint, dg);
      };
      tc_graph* dg = nullptr;
      CHECK(upload(flat, &dg) == TC_OK && (g_build.lines != nullptr) == (hint == 0));
      tc_graph_free(ctx, dg);
      g_big_codes = 0;
      CHECK(upload(skewed, &dg) == TC_OK && g_big_codes == (hint ? 0 : 1));
      tc_graph_free(ctx, dg);
      CHECK(upload(heavy, &dg) == TC_OK && g_build.closed);
      tc_graph_free(ctx, dg);
    }
  }
}

// What a program does with one graph, at a budget of device memory; the first
// status that is not TC_OK.
static tc_status use_graph(const Dag& g, size_t budget, int64_t* bytes = nullptr) {
  Ctx ctx;
  g_budget = budget;
  const tc_csr_view v = g.view();
  tc_graph* dg = nullptr;
  uint64_t total;
  tc_status st = tc_graph_upload(ctx, &v, TC_CHECK_SHAPE, &dg);
  for (int i = 0; i < 2 && st == TC_OK; ++i) st = tc_count_binned(ctx, dg, &total, nullptr);
  std::vector<uint32_t> edges(g.ci.size());
  tc_local out{};
  out.edge_counts = edges.data();
  if (st == TC_OK) st = tc_count_local(ctx, dg, &total, &out, nullptr);
  if (st == TC_OK) st = tc_count_binned(ctx, dg, &total, nullptr);
  if (bytes && dg) *bytes = tc_graph_bytes(dg);
  tc_graph_free(ctx, dg);
  g_budget = ~(size_t)0;
  return st;
}
static tc_status use_batch(const Dag& g, size_t budget, int64_t* bytes = nullptr) {
  Ctx ctx;
  g_budget = budget;
  const tc_csr_view v[2] = {g.view(), g.view()};
  tc_batch* b = nullptr;
  uint64_t counts[2];
  tc_status st = tc_batch_create(ctx, v, 2, TC_CHECK_SHAPE, &b);
  if (st == TC_OK) st = tc_batch_count(ctx, b, counts, nullptr);
  if (bytes && b) *bytes = tc_batch_bytes(b);
  tc_batch_free(ctx, b);
  g_budget = ~(size_t)0;
  return st;
}

// Codes and lines never take the place of what a call needs: whatever memory
// holds the calls without them holds the calls.
static void memory(int, char**) {
  const Dag flat = make(140000, 139000, 17), skewed = make(140000, 20000, 10, 2000, 500), few = make(60000, 50000, 70);
  g_closed = ~0ull >> 3;
  for (const Dag* g : {&flat, &skewed, &few})
    for (const auto& use : {use_graph, use_batch}) {
      const size_t n = g->rp.size() - 1, m = g->ci.size();
      int64_t least = 0, most = 0;
      g_peak = 0;
      CHECK(use(*g, ~(size_t)0, &most) == TC_OK);
      const size_t with = g_peak;
      const bool batch = use == use_batch;
      g_deny = [=](size_t b) {
        return batch ? b == tck::code_bytes(2 * m) : b == tck::code_bytes(m) || b == tck::line_bytes(m) || b == n || b == m;
      };
      g_peak = 0;
      CHECK(use(*g, ~(size_t)0, &least) == TC_OK);
      const size_t without = g_peak;
      g_deny = nullptr;
      CHECK(most >= least && with >= without);
      CHECK(use(*g, without - 1, nullptr) == TC_ENOMEM);
      int64_t bytes = 0;
      CHECK(use(*g, without, &bytes) == TC_OK && bytes == least);
      for (int i = 1; i < 16; ++i) CHECK(use(*g, without + (with - without) * i / 16, &bytes) == TC_OK);
      CHECK(use(*g, with, &bytes) == TC_OK && bytes == most);
    }
  // beside others: a graph and a batch with codes give them up for a third
  Ctx ctx;
  const tc_csr_view v = skewed.view(), w = few.view(), x = flat.view();
  tc_graph *a = nullptr, *c = nullptr;
  tc_batch* b = nullptr;
  uint64_t total;
  CHECK(tc_graph_upload(ctx, &v, TC_CHECK_SHAPE, &a) == TC_OK && tc_batch_create(ctx, &w, 1, TC_CHECK_SHAPE, &b) == TC_OK);
  CHECK(tc_batch_count(ctx, b, &total, nullptr) == TC_OK);
  const int64_t had_a = tc_graph_bytes(a), had_b = tc_batch_bytes(b);
  g_peak = g_used;
  CHECK(tc_graph_upload(ctx, &x, TC_CHECK_SHAPE | TC_UPLOAD_ONCE, &c) == TC_OK);
  const size_t need = g_peak;
  tc_graph_free(ctx, c);
  g_budget = need;
  CHECK(tc_graph_upload(ctx, &x, TC_CHECK_SHAPE, &c) == TC_OK && tc_graph_bytes(a) == had_a);
  tc_graph_free(ctx, c);
  g_budget = need - 1;
  CHECK(tc_graph_upload(ctx, &x, TC_CHECK_SHAPE, &c) == TC_OK);
  CHECK(tc_graph_bytes(a) < had_a && tc_batch_bytes(b) < had_b);
  CHECK(tc_count_binned(ctx, a, &total, nullptr) == TC_OK && g_args.core == 0 && !g_args.c16);
  CHECK(tc_batch_count(ctx, b, &total, nullptr) == TC_OK && g_args.core == 0 && !g_args.c16);
  tc_graph_free(ctx, c);
  tc_graph_free(ctx, a);
  tc_batch_free(ctx, b);
  g_budget = ~(size_t)0;
}

// Which graphs get codes and which lines; codes that too few edges can use go.
static void choice(int, char**) {
  Ctx ctx;
  uint64_t total;
  struct Got {
    bool codes, lines;
    int64_t bytes;
  };
  auto got = [&](const Dag& g) {
    const tc_csr_view v = g.view();
    tc_graph* dg = nullptr;
    g_big_codes = 0;
    CHECK(tc_graph_upload(ctx, &v, TC_CHECK_SHAPE, &dg) == TC_OK);
    CHECK(tc_count_binned(ctx, dg, &total, nullptr) == TC_OK);
    const Got x{g_args.c16 != nullptr, g_args.lines != nullptr, tc_graph_bytes(dg)};
    CHECK((g_args.core != 0) == x.codes);
    tc_graph_free(ctx, dg);
    return x;
  };
  g_closed = ~0ull >> 3;
  const Dag skewed = make(140000, 20000, 10, 2000, 500);
  const int64_t m = (int64_t)skewed.ci.size();
  const Got with = got(skewed);
  CHECK(with.codes && !with.lines && g_big_codes == 1);
  g_closed = (unsigned long long)m / 4 - 1;
  const Got without = got(skewed);
  CHECK(!without.codes && g_big_codes == 1 && with.bytes - without.bytes == (int64_t)tck::code_bytes(m) + m + 140000);
  g_closed = ~0ull >> 3;
  for (const Dag& flat : {make(140000, 60000, 80), make(140000, 139000, 17, 1, 64), make(140000, 139000, 17, 3, 600)}) {
    const Got x = got(flat);
    CHECK(!x.codes && x.lines && g_big_codes == 0);
  }
  // the plain kernel's loads: one id where lists are short and even
  const struct {
    Dag g;
    bool single;
  } plain[] = {{make(9000, 8000, 11), true}, {make(9000, 8000, 12), false}, {make(9000, 8000, 1, 100, 300), false}, {make(9, 0, 0), true}};
  for (const auto& p : plain) {
    const tc_csr_view v = p.g.view();
    double ms;
    g_single = !p.single;
    CHECK(tc_count_csr(ctx, &v, TC_CHECK_SHAPE, &total, nullptr) == TC_OK && g_single == p.single);
    tc_graph* dg = nullptr;
    g_single = !p.single;
    CHECK(tc_graph_upload(ctx, &v, TC_CHECK_SHAPE, &dg) == TC_OK && tc_count_plain(ctx, dg, &total, nullptr) == TC_OK);
    CHECK(g_single == p.single);
    tc_graph_free(ctx, dg);
    tc_batch* b = nullptr;
    g_single = !p.single;
    CHECK(tc_batch_create(ctx, &v, 1, TC_CHECK_SHAPE, &b) == TC_OK && tc_batch_count_each(ctx, b, &total, &ms, nullptr) == TC_OK);
    CHECK(g_single == p.single);
    tc_batch_free(ctx, b);
  }
}

// A plain count is one launch, whatever the graph's size, unless its sum might
// not fit beside the count of workgroups; the one after such a count clears
// the words first.
static void plain(int, char**) {
  Ctx ctx;
  for (const Dag& g : {make(9000, 8000, 11), make(300000, 200000, 20), make(9000, 8000, 1, 1, 4000)}) {
    const tc_csr_view v = g.view();
    tc_graph* dg = nullptr;
    uint64_t total;
    CHECK(tc_graph_upload(ctx, &v, TC_CHECK_SHAPE, &dg) == TC_OK);
    for (int i = 0; i < 3; ++i) {
      g_launches = 0;
      CHECK(tc_count_plain(ctx, dg, &total, nullptr) == TC_OK && g_direct && (g_launches == 1 || i == 0));
    }
    dg->max_out = 1 << 25;  // as if of a list that long: 2^25 * ids may pass 2^48
    const bool fits = (uint64_t)dg->max_out * g.ci.size() < 1ull << tck::kDoneShift;
    g_launches = 0;
    CHECK(tc_count_plain(ctx, dg, &total, nullptr) == TC_OK && g_direct == fits && g_launches == (fits ? 1 : 2));
    dg->edge_end = (int64_t)1 << 30;
    CHECK(tc_count_plain(ctx, dg, &total, nullptr) == TC_OK && !g_direct);
    tc_graph_free(ctx, dg);
  }
}

// Threads that copy a request: never more than the clients' share, never fewer
// than a large request's own; concurrent submits all arrive.
static void clients(int, char**) {
  constexpr size_t MB = (size_t)1 << 20;
  for (int c = 1; c <= 64; ++c)
    for (size_t mb : {0, 1, 2, 3, 5, 8, 15, 16, 24, 31, 32, 70, 1000}) {
      const int n = tcr::copy_threads(mb * MB, c), large = (int)std::min<size_t>(4, mb / 8);
      CHECK(n >= 1 && n <= 8 && (n == 1 || n <= (int)mb) && n >= large);
      if (mb < 16) CHECK(n * std::min(c, 8) <= 8);      // 8 threads for all that copy at once
      if (c == 1) CHECK(n == (int)std::min<size_t>(8, std::max<size_t>(1, mb)));
    }
  Ctx ctx;
  tc_server_config cfg{};
  cfg.hbm_budget = (uint64_t)1 << 30;
  cfg.host_staging = (uint64_t)64 << 20;  // some requests fit it, others go pageable
  cfg.slots = 2;
  cfg.max_batch_graphs = 64;
  cfg.max_batch_rows = 1 << 22;
  cfg.max_queue = 1024;
  tc_server* s = nullptr;
  CHECK(tc_server_create(ctx, &cfg, &s) == TC_OK);
  const Dag big = make(60000, 50000, 70), small = make(3000, 2000, 9);
  Dag bad = make(60000, 50000, 70);
  bad.ci[bad.ci.size() - 5] = 60000;  // in the last thread's share
  std::atomic<int> refused{0};
  std::vector<std::thread> all;
  for (int c = 0; c < 8; ++c)
    all.emplace_back([&, c] {
      for (int i = 0; i < 6; ++i) {
        const tc_csr_view v = (i % 3 == 0 ? big : i % 3 == 1 ? small : bad).view();
        const tc_status st = tc_server_submit(s, &v, (uint64_t)(c * 6 + i), TC_CHECK_SHAPE);
        if (st != TC_OK) ++refused;
      }
    });
  for (std::thread& t : all) t.join();
  CHECK(refused == 16 && tc_server_drain(s, 60000) == TC_OK);
  tc_request_result r[64];
  int32_t n = 0;
  CHECK(tc_server_poll(s, r, 64, &n, 1000) == TC_OK && n == 32);
  for (int i = 0; i < n; ++i) CHECK(r[i].status == TC_OK && r[i].tag % 3 != 2);
  tc_server_destroy(s);
}

// The words of a batch's sums: several a graph where there are few graphs, each
// on a line of its own inside what the counts' buffer holds.
static void batch_words(int, char**) {
  Ctx ctx;
  const Dag one = make(2000, 1500, 30), wide = make(70000, 1500, 30);
  for (int n : {1, 2, 5, 15, 16, 17, 31, 33, 63, 64, 65, 200})
    for (const Dag* g : {&one, &wide}) {
      const std::vector<tc_csr_view> v((size_t)n, g->view());
      std::vector<uint64_t> counts((size_t)n);
      tc_batch* b = nullptr;
      CHECK(tc_batch_create(ctx, v.data(), n, TC_CHECK_SHAPE, &b) == TC_OK);
      g_sums = 0;
      CHECK(tc_batch_count(ctx, b, counts.data(), nullptr) == TC_OK);
      const bool slots = n > 1 && n < tck::kBatchGraphs && g == &one;  // (the other has no codes)
      CHECK(g_sums == (slots ? 1 : 0) && (g_args.slots != nullptr) == slots);
      if (slots) {
        const int s = g_args.nslots;
        CHECK(s > 1 && s <= tck::kOutSlots && (s & (s - 1)) == 0 && s * n <= tck::kBatchWords);
        CHECK(g_args.slots - g_args.bufs.outs >= n && (g_args.slots - g_args.bufs.outs) % tck::kOutStride == 0);
        CHECK((size_t)(g_args.slots - g_args.bufs.outs + (int64_t)n * s * tck::kOutStride) * 8 <= g_size[g_args.bufs.outs]);
      }
      tc_batch_free(ctx, b);
    }
}

// Whether a batch has many light rows to a wave row.
static void light(int, char**) {
  Ctx ctx;
  const struct {
    Dag g;
    int many;
  } all[] = {{make(3000, 2500, 30), 1}, {make(3000, 2500, 80), 0}, {make(3000, 800, 63, 100, 64), 0},
             {make(3000, 801, 63, 100, 64), 1}, {make(3000, 801, 63, 100, 127), 1}, {make(3000, 10, 5, 100, 128), 1}};
  for (const auto& x : all) {
    const tc_csr_view v[2] = {x.g.view(), x.g.view()};
    tc_batch* b = nullptr;
    uint64_t counts[2];
    CHECK(tc_batch_create(ctx, v, 2, TC_CHECK_SHAPE, &b) == TC_OK && tc_batch_count(ctx, b, counts, nullptr) == TC_OK);
    CHECK(g_args.many_light == x.many);
    tc_batch_free(ctx, b);
  }
}

int main(int argc, char** argv) {
  static const std::map<std::string, std::function<void(int, char**)>> all = {
      {"one_shot", one_shot},
      {"memory", memory},
      {"choice", choice},
      {"plain", plain},
      {"clients", clients},
      {"batch_words", batch_words},
      {"light", light},
  };
  const auto it = argc > 1 ? all.find(argv[1]) : all.end();
  if (it == all.end()) return 2;
  it->second(argc - 2, argv + 2);
  if (!g_size.empty()) return std::printf("%zu device allocations never freed\n", g_size.size()), 1;
  return 0;
}
