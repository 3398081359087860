// The library's calls where device memory holds their tables but not what they are merely faster with.
// Usage: memory_limit_check LIBRARY CASE BUDGET_KIB; prints the status and what ran.
#include <dlfcn.h>

#include "hip_stub.hpp"
#include "../include/stwo_hip.h"

static void* lib;
template <class F>
static F* entry(F*, const char* name) {
  return (F*)dlsym(lib, name);
}
#define ENTRY(name) entry((decltype(&name))nullptr, #name)

int main(int argc, char** argv) {
  lib = dlopen(argv[1], RTLD_NOW);
  if (!lib) {
    fprintf(stderr, "%s\n", dlerror());
    return 2;
  }
  const std::string what = argv[2];
  stub::budget = (size_t)atol(argv[3]) << 10;
  auto fake = [](uint32_t n, uint64_t stride, uint64_t base) {  // column pointers that nothing reads here
    std::vector<uint32_t*> p;
    for (uint32_t i = 0; i < n; i++) p.push_back((uint32_t*)(base + i * stride));
    return p;
  };
  uint32_t* const tree = (uint32_t*)0x500000000000ull;
  int st = -1;
  if (what == "lde" || what == "plan" || what == "plan_tuned") {
    const uint32_t n = 64, log = 20, blowup = 1;
    auto ev = fake(n, 4 << log, 0x600000000000ull), co = fake(n, 4 << log, 0x610000000000ull),
         ld = fake(n, 8 << log, 0x620000000000ull);
    std::vector<uint32_t> logs(n, log);
    if (what == "lde") {
      st = ENTRY(stwo_hip_lde_columns_async)((const uint32_t* const*)ev.data(), co.data(), ld.data(), logs.data(), n, blowup,
                                             tree, tree, 1ull << (log + blowup - 1));
    } else {
      std::vector<StwoBlake2sHash*> layers;
      for (uint32_t k = 0; k <= log + blowup; k++) layers.push_back((StwoBlake2sHash*)(0x630000000000ull + ((uint64_t)k << 32)));
      StwoCommitPlan* plan = nullptr;
      st = ENTRY(stwo_hip_commit_plan_create)(&plan, n, (const uint32_t* const*)ev.data(), co.data(), ld.data(), logs.data(),
                                              blowup, tree, tree, 1ull << (log + blowup - 1), layers.data(), log + blowup,
                                              what == "plan_tuned");
      stub::launched.clear();
      if (!st) st = ENTRY(stwo_hip_commit_plan_run)(plan, 0);
    }
  } else {  // whole small columns
    const uint32_t n = 20000, log = 12;
    auto a = fake(n, 4 << log, 0x600000000000ull), b = fake(n, 4 << log, 0x610000000000ull);
    std::vector<uint32_t> logs(n, log);
    if (what == "interpolate")
      st = ENTRY(stwo_hip_interpolate_columns_async)(a.data(), logs.data(), n, tree, 1ull << (log - 1));
    else if (what == "evaluate")
      st = ENTRY(stwo_hip_evaluate_columns_async)((const uint32_t* const*)a.data(), logs.data(), b.data(), logs.data(), n,
                                                  tree, 1ull << (log - 1));
  }
  printf("status %d matrices %d butterflies %d\n", st, stub::find("matrix_kernel") >= 0,
         stub::find("fft_pass_kernel") >= 0 || stub::find("fft_lde_strided_kernel") >= 0);
  return 0;
}
