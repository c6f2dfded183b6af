// Host-side check of launch rules that pick a kernel or an order by size, built with asserts on and
// run on the CPU by tests/test_index_math.py from the headers that the launches use.
#undef NDEBUG
#include <cassert>
#include <cstdio>

#include "plz_gemv_split.h"

static long checks = 0;

// Split bit-plane GEMVs: every plan is one that the kernel can run, and the launches whose both
// sides are known (256 CUs) take the faster one.
static void check_gemv_split() {
  using namespace plz::gv;
  for (int64_t cus : {1, 80, 256, 304})
    for (int64_t items = 1; items <= cus + 2; ++items)
      for (int64_t stages : {1, 2, 4, 10, 16, 38, 64, 300})
        for (int M = 1; M <= 16; ++M) {
          const SplitPlan p = split_plan_on(items, stages, M, cus);
          ++checks;
          if (p.rbw == 0) continue;
          assert(M <= 8 && items <= cus);
          assert(p.rbw == 1 || p.rbw == 2 || (p.rbw == 4 && M == 1));
          assert(p.waves >= p.rbw * sp_ni(M) / 2 && p.waves <= SP_WAVES);
          assert(p.waves * sp_wave_bytes(sp_ni(M), p.rbw, M) <= SP_LDS);
        }
  struct { int64_t items, K; int M; bool split; } known[] = {
      // one layer's groups: q/k/v, o, gate/up, down
      {48, 2560, 1, true}, {20, 4096, 1, true}, {152, 2560, 1, true}, {20, 9728, 1, true},
      {48, 2560, 8, true}, {20, 4096, 8, true}, {20, 9728, 8, true},
      {152, 2560, 4, true}, {160, 2560, 8, false}, {160, 1024, 8, true}, {160, 256, 8, true},
      {76, 9728, 3, true}, {76, 9728, 5, false}, {76, 9728, 8, false}, {140, 9728, 2, false},
      {140, 9728, 4, false}, {140, 9728, 8, false}, {140, 4096, 3, true}, {140, 4096, 5, false},
      {240, 2560, 1, true}, {200, 9728, 1, true}, {257, 2560, 1, false}, {161, 256, 2, false}};
  for (const auto& k : known) {
    const bool split = split_plan_on(k.items, k.K / 256, k.M, 256).rbw > 0;
    if (split != k.split)
      printf("items %ld K %ld M %d: split %d\n", (long)k.items, (long)k.K, k.M, (int)split);
    assert(split == k.split);
    ++checks;
  }
}

int main() {
  check_gemv_split();
  printf("launch rules: %ld checks passed\n", checks);
  return 0;
}
