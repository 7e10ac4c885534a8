// Host paths of libraja_cdna4.so on a recording HIP runtime (no GPU): what is
// launched and copied, in which order, and what survives a failing call.
//   test_host_paths <libraja_cdna4.so> <test name>
#include "recording_hip.hpp"

#include <dlfcn.h>
#include <stdint.h>
#include <stdio.h>

#include <chrono>
#include <future>
#include <memory>
#include <string>
#include <thread>
#include <utility>
#include <vector>

#include "raja_cdna4.h"

namespace
{
int g_failed = 0;
#define CHECK(cond, ...)                                 \
  do                                                     \
  {                                                      \
    if (!(cond))                                         \
    {                                                    \
      ++g_failed;                                        \
      printf("line %d: %s  ", __LINE__, #cond);          \
      printf(__VA_ARGS__);                               \
      printf("\n");                                      \
    }                                                    \
  } while (0)

void* g_lib = nullptr;
template<typename F>
F* entry(const char* name)
{
  F* f = (F*)dlsym(g_lib, name);
  if (!f)
  {
    printf("no entry point %s\n", name);
    exit(2);
  }
  return f;
}
#define ENTRY(name) entry<decltype(name)>(#name)

// ---- a plan whose table upload fails ---------------------------------------------
// Segments of every kind of record (empty, one element, short ones of all
// classes, longer ones), and the first call of each batched operation with one
// allocation or copy failing: that call reports it, the plan holds nothing of
// the failed build, and the next call builds and uploads the whole table.
void failed_upload()
{
  const std::vector<int64_t> lens = {0, 1, 60, 500, 2000, 5000, 8000, 20000, 70000, 40};
  std::vector<int64_t> off = {0};
  for (int64_t n : lens) off.push_back(off.back() + n);
  std::vector<uint32_t> keys((size_t)off.back()), vals(keys.size());
  std::vector<double> x((size_t)off.back()), sums(lens.size());
  std::vector<int32_t> xi((size_t)off.back()), oi(xi.size());
  auto create = ENTRY(raja_cdna4_segments_create);
  auto destroy = ENTRY(raja_cdna4_segments_destroy);
  auto sort = ENTRY(raja_cdna4_segmented_sort_pairs);
  auto reduce = ENTRY(raja_cdna4_segmented_reduce);
  auto scan = ENTRY(raja_cdna4_segmented_exclusive_scan);
  const double zero = 0.0;
  const int32_t izero = 0;
  using Plan = raja_cdna4_segments_s*;
  std::vector<std::function<int(Plan)>> ops = {
      [&](Plan p) { return sort(p, RAJA_CDNA4_U32, keys.data(), vals.data(), 4, 0, nullptr); },
      [&](Plan p) { return reduce(p, RAJA_CDNA4_F64, RAJA_CDNA4_OP_PLUS, x.data(), &zero, sums.data(), nullptr); },
      [&](Plan p) { return scan(p, RAJA_CDNA4_I32, RAJA_CDNA4_OP_PLUS, xi.data(), oi.data(), &izero, nullptr); }};
  auto copies = [] {
    std::vector<size_t> b;
    for (const rec::Call& c : rec::g_calls)
      if (c.what == "copy") b.push_back(c.bytes);
    return b;
  };
  for (size_t o = 0; o < ops.size(); ++o)
  {
    // the stream's scratch exists before, so that only the plan's own uploads fail
    Plan warm = nullptr;
    CHECK(create(off.data(), (int64_t)lens.size(), &warm) == 0, "create");
    rec::clear();
    CHECK(ops[o](warm) == 0, "warm call %zu", o);
    const std::vector<size_t> want = copies();
    CHECK(!want.empty(), "operation %zu uploads nothing", o);
    CHECK(destroy(warm) == 0, "destroy");
    const size_t base = rec::live_blocks();
    for (int copy = 0; copy < 2; ++copy)
    {
      for (int k = 1; k <= (int)want.size(); ++k)
      {
        Plan p = nullptr;
        CHECK(create(off.data(), (int64_t)lens.size(), &p) == 0, "create");
        const size_t held = rec::live_blocks();
        (copy ? rec::g_fail_copy : rec::g_fail_malloc) = k;
        rec::clear();
        CHECK(ops[o](p) != 0, "operation %zu, failing %s %d went unreported", o, copy ? "copy" : "malloc", k);
        CHECK(rec::count("launch") == 0, "operation %zu launched after a failed upload", o);
        CHECK(rec::live_blocks() == held, "operation %zu, failing %s %d: %zu blocks kept of a failed build", o,
              copy ? "copy" : "malloc", k, rec::live_blocks() - held);
        rec::g_fail_copy = rec::g_fail_malloc = 0;
        rec::clear();
        CHECK(ops[o](p) == 0, "operation %zu after a failed upload", o);
        CHECK(copies() == want, "operation %zu, after failing %s %d: %zu uploads, not %zu", o,
              copy ? "copy" : "malloc", k, copies().size(), want.size());
        CHECK(destroy(p) == 0, "destroy");
        CHECK(rec::live_blocks() == base, "operation %zu leaks", o);
      }
    }
  }
}

// ---- the lookback gate -------------------------------------------------------------
// What a sort's kernels leave in pinned memory (arguments as in
// partition_sort.hip and digit_hist.hpp).
constexpr uint32_t kTwoDigits = 0x80000005u;  // the keys differ in digits 0 and 2
void answer(const std::string& kernel, void** args, bool sample, bool counts)
{
  auto host = [&](int arg) { return *(volatile uint32_t**)args[arg]; };
  auto is = [&](const char* name) { return kernel.find(name) != std::string::npos; };
  if (is("sample_kernel")) *host(10) = sample ? 2u : 1u;
  if (is("plan1_kernel"))
  {
    host(9)[0] = sample && counts ? 1u : 0u;
    host(9)[2] = sample ? 0u : kTwoDigits;
  }
  if (is("plan2_kernel")) *host(8) = counts ? 1u : 0u;
  if (is("digits_kernel")) *host(2) = kTwoDigits;
}
void take_partition(const std::string& k, void** a) { answer(k, a, true, true); }
void sample_refuses(const std::string& k, void** a) { answer(k, a, false, false); }
void counts_refuse(const std::string& k, void** a) { answer(k, a, true, false); }

// While a sort waits on the host, a scan of many tiles on another thread and
// stream must go through: the wait may be for work which that thread has yet
// to queue.  And the gate's event covers the scatters alone: the block sorts,
// which look back at nothing, are launched after it is recorded.
void gate_across_waits()
{
  auto sort = ENTRY(raja_cdna4_sort_pairs);
  auto scan = ENTRY(raja_cdna4_exclusive_scan);
  hipStream_t s1 = nullptr, s2 = nullptr;
  (void)hipStreamCreateWithFlags(&s1, 0);
  (void)hipStreamCreateWithFlags(&s2, 0);
  const int64_t n = 1 << 22;
  std::vector<int32_t> in((size_t)n), out((size_t)n);
  const int32_t zero = 0;
  auto scan_on_s2 = [&] {
    return scan(RAJA_CDNA4_I32, RAJA_CDNA4_OP_PLUS, in.data(), out.data(), n, &zero, s2);
  };
  CHECK(scan_on_s2() == 0, "scan");
  for (const auto& [dtype, len] : {std::pair<int, int64_t>{RAJA_CDNA4_U32, 1 << 20}, {RAJA_CDNA4_U64, 1 << 22}})
  {
    std::vector<uint64_t> keys((size_t)len);
    std::vector<uint32_t> vals((size_t)len);
    rec::on_launch = take_partition;
    CHECK(sort(dtype, keys.data(), vals.data(), 4, len, 0, s1) == 0, "sort");  // scratch
    int waits = 0, stuck = 0;
    std::thread::id me = std::this_thread::get_id();
    rec::on_wait = [&](const char*) {
      if (std::this_thread::get_id() != me) return;
      ++waits;
      auto done = std::make_shared<std::promise<int>>();
      std::future<int> f = done->get_future();
      std::thread([done, &scan_on_s2] { done->set_value(scan_on_s2()); }).detach();
      if (f.wait_for(std::chrono::seconds(5)) != std::future_status::ready) ++stuck;
    };
    rec::clear();
    CHECK(sort(dtype, keys.data(), vals.data(), 4, len, 0, s1) == 0, "sort");
    rec::on_wait = nullptr;
    CHECK(waits > 0, "the sort of %lld keys waits for nothing", (long long)len);
    CHECK(stuck == 0, "a scan on another thread stood still while the sort waited");
    if (stuck) std::this_thread::sleep_for(std::chrono::seconds(1));
    rec::on_launch = nullptr;
    std::lock_guard<std::recursive_mutex> g(rec::g_m);
    size_t scatter = 0, recorded = 0, groups = 0;
    for (size_t i = 0; i < rec::g_calls.size(); ++i)
    {
      const rec::Call& c = rec::g_calls[i];
      if (c.stream != (void*)s1) continue;
      if (c.kernel.find("onesweep_kernel") != std::string::npos) scatter = i;
      if (c.kernel.find("local_groups_kernel") != std::string::npos) groups = i;
      if (c.what == "event_record" && groups == 0) recorded = i;
    }
    CHECK(scatter > 0 && groups > scatter, "no partition");
    CHECK(recorded > scatter, "the gate's event is recorded after the block sorts");
  }
}

// ---- scratch of a batched sort ------------------------------------------------------
// All of a call's scratch grows before its first launch (growing waits for the
// stream), and a batch of short segments grows none: it can be captured on a
// stream that has run something else.
void batched_sort_scratch()
{
  auto create = ENTRY(raja_cdna4_segments_create);
  auto sort = ENTRY(raja_cdna4_segmented_sort_pairs);
  auto scan = ENTRY(raja_cdna4_exclusive_scan);
  std::vector<int64_t> off = {0};
  for (int g = 0; g < 3000; ++g) off.push_back(off.back() + 1 + 37 * g % 8192);
  const int64_t nshort = (int64_t)off.size() - 1;
  for (int g = 0; g < 40; ++g) off.push_back(off.back() + 100000);
  std::vector<uint32_t> keys((size_t)off.back()), vals(keys.size());
  raja_cdna4_segments_s *all = nullptr, *few = nullptr;
  CHECK(create(off.data(), (int64_t)off.size() - 1, &all) == 0, "create");
  CHECK(create(off.data(), nshort, &few) == 0, "create");
  CHECK(sort(few, RAJA_CDNA4_U32, keys.data(), vals.data(), 4, 0, nullptr) == 0, "tables");
  CHECK(sort(all, RAJA_CDNA4_U32, keys.data(), vals.data(), 4, 0, nullptr) == 0, "tables");
  hipStream_t s1 = nullptr, s2 = nullptr;
  (void)hipStreamCreateWithFlags(&s1, 0);
  (void)hipStreamCreateWithFlags(&s2, 0);
  // scratch that a call of another kind left small
  CHECK(sort(few, RAJA_CDNA4_U32, keys.data(), vals.data(), 4, 0, s1) == 0, "sort");
  rec::clear();
  CHECK(sort(all, RAJA_CDNA4_U32, keys.data(), vals.data(), 4, 0, s1) == 0, "sort");
  size_t launched = 0;
  for (const rec::Call& c : rec::g_calls)
  {
    launched += c.what == "launch";
    CHECK(launched == 0 || (c.what != "malloc" && c.what != "free" && c.what != "stream_wait"),
          "%s after %zu launches", c.what.c_str(), launched);
  }
  CHECK(launched > 6, "launches");

  std::vector<int32_t> in(100), out(100);
  const int32_t zero = 0;
  CHECK(scan(RAJA_CDNA4_I32, RAJA_CDNA4_OP_PLUS, in.data(), out.data(), 100, &zero, s2) == 0, "scan");
  rec::g_capturing = true;
  rec::clear();
  CHECK(sort(few, RAJA_CDNA4_U32, keys.data(), vals.data(), 4, 0, s2) == 0, "captured sort");
  CHECK(rec::count("malloc") + rec::count("free") + rec::count("stream_wait") + rec::count("copy") == 0,
        "a captured sort of short segments grows the stream's scratch");
  rec::g_capturing = false;
}

// The allocation-free scan's descriptors are one array per device: calls on
// different streams run one after the other, one-tile calls too.
void noalloc_order()
{
  auto scan = ENTRY(raja_cdna4_exclusive_scan_noalloc);
  hipStream_t s[2] = {nullptr, nullptr};
  for (hipStream_t& x : s) (void)hipStreamCreateWithFlags(&x, 0);
  const int32_t zero = 0;
  std::vector<int32_t> in(200000), out(200000);
  for (int64_t n : {1, 1000, 200000})
  {
    for (int i = 0; i < 4; ++i)
    {
      rec::clear();
      CHECK(scan(RAJA_CDNA4_I32, RAJA_CDNA4_OP_PLUS, in.data(), out.data(), n, &zero, s[i % 2]) == 0, "scan");
      CHECK(i == 0 || rec::count("wait_event") == 1, "n = %lld: no wait for the other stream's scan", (long long)n);
      CHECK(rec::count("event_record") == 1, "n = %lld: the next stream has nothing to wait for", (long long)n);
    }
  }
}

// A small batch is one launch, whatever its segments' lengths; a large one a
// launch per length class and one for what those leave to the passes.
void batched_sort_launches()
{
  auto create = ENTRY(raja_cdna4_segments_create);
  auto destroy = ENTRY(raja_cdna4_segments_destroy);
  auto sort = ENTRY(raja_cdna4_segmented_sort_pairs);
  for (int count : {1, 60, 512, 513})
  {
    std::vector<int64_t> off = {0};
    for (int g = 0; g < count; ++g) off.push_back(off.back() + 2 + 1297 * g % 8190);
    std::vector<uint32_t> keys((size_t)off.back()), vals(keys.size());
    raja_cdna4_segments_s* p = nullptr;
    CHECK(create(off.data(), count, &p) == 0, "create");
    rec::clear();
    CHECK(sort(p, RAJA_CDNA4_U32, keys.data(), vals.data(), 4, 0, nullptr) == 0, "sort");
    const size_t want = count <= 512 ? 1 : 6;
    CHECK(rec::count("launch") == want, "%d segments: %zu launches", count, rec::count("launch"));
    CHECK(destroy(p) == 0, "destroy");
  }
}

// Two threads' batches of short segments on one stream: the launches of one come
// in a row, so neither reads marks that the other has written over.
void batched_sorts_of_two_threads()
{
  auto create = ENTRY(raja_cdna4_segments_create);
  auto sort = ENTRY(raja_cdna4_segmented_sort_pairs);
  std::vector<int64_t> off = {0};
  for (int g = 0; g < 3000; ++g) off.push_back(off.back() + 2 + 37 * g % 8190);
  std::vector<uint32_t> keys((size_t)off.back()), vals(keys.size());
  raja_cdna4_segments_s* p = nullptr;
  CHECK(create(off.data(), (int64_t)off.size() - 1, &p) == 0, "create");
  auto one = [&](int descending) {
    return sort(p, RAJA_CDNA4_U32, keys.data(), vals.data(), 4, descending, nullptr);
  };
  CHECK(one(0) == 0, "sort");
  std::vector<std::thread::id> order;
  std::mutex m;
  std::thread other;
  rec::on_launch = [&](const std::string&, void**) {
    bool first = false;
    {
      std::lock_guard<std::mutex> g(m);
      first = order.empty();
      order.push_back(std::this_thread::get_id());
    }
    if (!first) return;
    other = std::thread([&] { CHECK(one(0) == 0, "sort"); });
    std::this_thread::sleep_for(std::chrono::milliseconds(300));
  };
  CHECK(one(0) == 0, "sort");
  other.join();
  rec::on_launch = nullptr;
  size_t turns = 0;
  for (size_t i = 1; i < order.size(); ++i) turns += order[i] != order[i - 1];
  CHECK(order.size() == 12 && turns == 1, "%zu launches, %zu changes of thread", order.size(), turns);
}

// ---- a stream with a long queue --------------------------------------------------------
// The answers of a sort's kernels come late: the queries in between are no
// errors, the calls after them succeed, and a stream that ends without an answer
// is reported.
void late_answers()
{
  auto sort = ENTRY(raja_cdna4_sort_pairs);
  const int64_t n = 1 << 22;
  std::vector<uint64_t> keys((size_t)n);
  std::vector<uint32_t> vals((size_t)n);
  std::vector<std::function<void()>> late;
  bool never = false;
  rec::on_launch = [&](const std::string& kernel, void** args) {
    volatile uint32_t* w = nullptr;
    if (kernel.find("sample_kernel") != std::string::npos) w = *(volatile uint32_t**)args[10];
    if (kernel.find("digits_kernel") != std::string::npos) w = *(volatile uint32_t**)args[2];
    const uint32_t v = kernel.find("sample_kernel") != std::string::npos ? 1u : kTwoDigits;
    if (w && !never)
    {
      rec::g_not_ready = 3;
      late.push_back([w, v] { *w = v; });
    }
  };
  rec::on_wait = [&](const char*) {
    if (rec::g_not_ready == 1 && !late.empty())
    {
      late.back()();
      late.pop_back();
    }
  };
  for (const auto& [dtype, len] : {std::pair<int, int64_t>{RAJA_CDNA4_U64, n}, {RAJA_CDNA4_U32, 2000000}})
  {
    rec::clear();
    CHECK(sort(dtype, keys.data(), vals.data(), 4, len, 0, nullptr) == 0, "sort with late answers");
    CHECK(rec::count("launch", "onesweep_kernel") == 2, "%zu passes", rec::count("launch", "onesweep_kernel"));
  }
  never = true;
  CHECK(sort(RAJA_CDNA4_U64, keys.data(), vals.data(), 4, n, 0, nullptr) != 0, "a missing answer goes unreported");
  rec::on_launch = nullptr;
  rec::on_wait = nullptr;
}

// ---- shape tuning --------------------------------------------------------------------
// The tuner's candidates run the kernels that they name, and a recorded full
// tile is taken, not the tile that untuned spans of that length take.
void tuner_shapes()
{
  auto tune = ENTRY(raja_cdna4_autotune);
  auto forget = ENTRY(raja_cdna4_tune_forget);
  auto path = ENTRY(raja_cdna4_tune_cache_path);
  auto sort = ENTRY(raja_cdna4_sort_pairs);
  auto scan = ENTRY(raja_cdna4_exclusive_scan);
  auto shapes = [](const char* kernel) {  // grid sizes of a kernel's launches
    std::set<unsigned> g;
    for (const rec::Call& c : rec::g_calls)
      if (c.kernel.find(kernel) != std::string::npos) g.insert(c.grid);
    return g;
  };
  rec::on_launch = take_partition;
  for (int64_t n : {int64_t(5000), int64_t(100000), int64_t(1) << 20})
  {
    rec::clear();
    CHECK(tune(2, RAJA_CDNA4_U32, n, nullptr) == 0, "tune");
    const std::set<unsigned> want = {(unsigned)((n + 16383) / 16384), (unsigned)((n + 8191) / 8192),
                                     (unsigned)((n + 4095) / 4096)};
    CHECK(shapes("onesweep_kernel") == want, "n = %lld: %zu tiles measured", (long long)n,
          shapes("onesweep_kernel").size());
    CHECK(rec::count("launch", "sample_kernel") + rec::count("launch", "span_sort_kernel") == 0,
          "n = %lld: not the digit passes", (long long)n);
  }
  rec::on_launch = sample_refuses;
  rec::clear();
  CHECK(tune(1, RAJA_CDNA4_I32, 1 << 20, nullptr) == 0, "tune");
  CHECK(shapes("scan_kernel") == (std::set<unsigned>{32, 64, 128}), "%zu scan tiles measured",
        shapes("scan_kernel").size());

  char file[1024];
  CHECK(path(file, sizeof(file)) == 0, "path");
  FILE* f = fopen(file, "w");
  CHECK(f != nullptr, "%s", file);
  if (!f) return;
  fprintf(f, "sort_pairs 2 20 0 0.0\nexclusive_scan 0 20 0 0.0\n");
  fclose(f);
  std::vector<uint32_t> a(1 << 20), b(1 << 20);
  const int32_t zero = 0;
  for (int tuned = 1; tuned >= 0; --tuned)
  {
    CHECK(forget() == 0, "forget");
    if (!tuned) remove(file);
    rec::clear();
    CHECK(sort(RAJA_CDNA4_U32, a.data(), b.data(), 4, 1 << 20, 0, nullptr) == 0, "sort");
    // the partition's refused scatter has the small tile: count the digit passes' grid
    size_t full = 0;
    for (const rec::Call& c : rec::g_calls) full += c.kernel.find("onesweep_kernel") != std::string::npos && c.grid == 64;
    CHECK((full > 0) == (tuned == 1), "full radix tile %s", tuned ? "not taken" : "taken untuned");
    rec::clear();
    CHECK(scan(RAJA_CDNA4_I32, RAJA_CDNA4_OP_PLUS, a.data(), b.data(), 1 << 20, &zero, nullptr) == 0, "scan");
    CHECK(shapes("scan_kernel") == std::set<unsigned>{tuned ? 32u : 128u}, "scan tile");
  }
}

// ---- spans that the partition refuses -------------------------------------------------
// A span that the sample refuses has its digits counted once, by the kernel
// after the sample, and goes on with the digit passes: nothing is copied back
// and the host waits once.  One that only the counts refuse starts over.
void refused_spans()
{
  auto sort = ENTRY(raja_cdna4_sort_pairs);
  const int64_t most = 1 << 22;
  std::vector<uint64_t> keys((size_t)most);
  std::vector<uint32_t> vals((size_t)most);
  for (const auto& [dtype, n] : {std::pair<int, int64_t>{RAJA_CDNA4_U32, 1 << 20}, {RAJA_CDNA4_U64, 1 << 22}})
  {
    const bool one_level = n == 1 << 20;
    for (int how = 0; how < 2; ++how)
    {
      rec::on_launch = how == 0 ? sample_refuses : counts_refuse;
      for (int rep = 0; rep < 2; ++rep)  // the first call grows the scratch
      {
        rec::clear();
        CHECK(sort(dtype, keys.data(), vals.data(), 4, n, 0, nullptr) == 0, "sort");
      }
      const size_t hists = rec::count("launch", "11hist_kernel");
      const size_t scatters = rec::count("launch", "MapDigit");
      const size_t passes = rec::count("launch", "onesweep_kernel") - scatters;
      CHECK(passes == 2, "%zu passes for two digits", passes);
      CHECK(rec::count("copy_async") == 0 && rec::count("stream_wait") == 0, "%zu copies, %zu waits",
            rec::count("copy_async"), rec::count("stream_wait"));
      CHECK(rec::count("launch", "local_groups") == 0, "block sorts");
      if (how == 0)
      {
        CHECK(hists == (one_level ? 0 : 1), "%zu digit histograms after the sample", hists);
        CHECK(rec::count("launch", "clear_words") == 0, "cleared again");
        CHECK(scatters == (one_level ? 1 : 0), "%zu scatters", scatters);
        CHECK(rec::count("launch", "hist1_kernel") == (one_level ? 1 : 0) && rec::count("launch", "hist2_kernel") == 0,
              "counts");
      }
      else
      {
        CHECK(hists == (one_level ? 1 : 2), "%zu digit histograms after the counts", hists);
      }
    }
  }
  rec::on_launch = nullptr;
}
}  // namespace

int main(int argc, char** argv)
{
  if (argc < 3) return 2;
  g_lib = dlopen(argv[1], RTLD_NOW | RTLD_LOCAL);
  if (!g_lib)
  {
    printf("%s\n", dlerror());
    return 2;
  }
  if (ENTRY(raja_cdna4_init)(0) != 0) return 2;
  const std::map<std::string, void (*)()> tests = {{"failed_upload", failed_upload},
                                                      {"gate_across_waits", gate_across_waits},
                                                      {"batched_sort_scratch", batched_sort_scratch},
                                                      {"noalloc_order", noalloc_order},
                                                      {"tuner_shapes", tuner_shapes},
                                                      {"refused_spans", refused_spans},
                                                      {"late_answers", late_answers},
                                                      {"batched_sort_launches", batched_sort_launches},
                                                      {"batched_sorts_of_two_threads", batched_sorts_of_two_threads}};
  const auto it = tests.find(argv[2]);
  if (it == tests.end()) return 2;
  it->second();
  printf("%s: %d failed\n", argv[2], g_failed);
  fflush(stdout);
  _Exit(g_failed ? 1 : 0);
}
