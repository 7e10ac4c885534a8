// Host paths of libraja_cdna4.so on a recording HIP runtime (no GPU): what is
// launched and copied, in which order, and what survives a failing call.
//   test_host_paths <libraja_cdna4.so> <test name>
#include "recording_hip.hpp"

#include <dlfcn.h>
#include <stdint.h>
#include <stdio.h>

#include <string>
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
  const std::map<std::string, void (*)()> tests = {{"failed_upload", failed_upload}};
  const auto it = tests.find(argv[2]);
  if (it == tests.end()) return 2;
  it->second();
  printf("%s: %d failed\n", argv[2], g_failed);
  fflush(stdout);
  _Exit(g_failed ? 1 : 0);
}
