// Order of the attention kernels' work items (plz_attn.hip).
#pragma once
#include "plz_common.h"

namespace plz {
namespace attn {

// Work item (query block, batch, kv head, query head of it) of a workgroup of the forward and the
// dQ kernel, longest first (the last query blocks see the most kv blocks). Workgroup id runs on
// XCD id % 8, each with its own L2: where the (batch, kv head) pairs divide by 8, each XCD takes
// an eighth of them and the G query heads of a pair, which walk the same K and V, are neighbours
// there: with a pair's heads on different XCDs every workgroup fetched its own K and V past the
// L2s, 0.8 GB in the forward and 1.1 GB in dQ at B32 S512 Hq32 Hkv8 (6 TB/s), which are 0.30 and
// 0.57 now. Forward 147 -> 141 us, dQ 188 -> 179 there; B8 S2048 355 -> 328 and 424 -> 399; one
// long sequence (B1 S4096) the same. With one query head per kv head every order here keeps a pair on one XCD, and the plain one
// is also the dK/dV kernel's, which finds the pair's Q and dO in that L2: backward at B16 S128
// 8/8 heads 20.4 us against 21.8, B8 S256 26.2 against 27.8. The dK/dV kernel keeps batch-major
// pairs: the kv blocks of a pair side by side on an XCD (they walk the same Q and dO) took 211 us
// for 214 at B32 S512, but 282 for 273 at B2 S4096.
struct QItem {
  int qb, b, hk, h;
};
__host__ __device__ __forceinline__ QItem q_item(int id, int nqb, int B, int Hq, int Hkv) {
  const int G = Hq / Hkv, pairs = B * Hkv;
  int pair, g, lev;
  if (pairs % 8 == 0 && G > 1) {
    const int n = pairs / 8, s = id >> 3;
    lev = s / (n * G);
    const int r = s - lev * (n * G);
    pair = (id & 7) * n + r / G;
    g = r % G;
  } else {
    lev = id / (pairs * G);
    const int r = id - lev * (pairs * G);
    pair = r / G;
    g = r % G;
  }
  const int b = pair / Hkv, hk = pair - b * Hkv;
  return QItem{nqb - 1 - lev, b, hk, hk * G + g};
}

}  // namespace attn
}  // namespace plz
