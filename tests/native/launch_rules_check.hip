// Host-side check of launch rules that pick a kernel or an order by size, built with asserts on and
// run on the CPU by tests/test_index_math.py from the headers that the launches use.
#undef NDEBUG
#include <cassert>
#include <cstdio>
#include <set>

#include "plz_attn_items.h"
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

// Attention items: every (query block, batch, query head) once, the longest first, the kv head its
// own; the heads of a pair on one XCD (id % 8) where the pairs divide by 8, and one query head per
// kv head in batch-major order, as the dK/dV kernel's.
static void check_attn_items() {
  using namespace plz::attn;
  for (int nqb : {1, 3, 4})
    for (int B : {1, 2, 3, 8, 16})
      for (const auto& heads : {std::pair<int, int>{1, 1}, {8, 8}, {6, 2}, {32, 8}, {16, 2}, {2, 1}}) {
        const int Hq = heads.first, Hkv = heads.second, G = Hq / Hkv;
        std::set<int> seen;
        for (int id = 0; id < nqb * B * Hq; ++id) {
          const QItem q = q_item(id, nqb, B, Hq, Hkv);
          assert(q.qb == nqb - 1 - id / (B * Hq) && q.b >= 0 && q.b < B && q.h >= 0 && q.h < Hq);
          assert(q.hk == q.h / G);
          assert(seen.insert((q.qb * B + q.b) * Hq + q.h).second);
          if (G == 1) assert(q.b * Hq + q.h == id % (B * Hq));
          if (G > 1 && B * Hkv % 8 == 0) assert((q.b * Hkv + q.hk) / (B * Hkv / 8) == id % 8);
          ++checks;
        }
      }
}

int main() {
  check_attn_items();
  check_gemv_split();
  printf("launch rules: %ld checks passed\n", checks);
  return 0;
}
