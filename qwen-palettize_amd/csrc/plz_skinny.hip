// Hard LUT-linear forward of few rows: y[M, N] = x W^T (+ bias) (+ t B^T), M <= 64.
//
// At these M the 256x256 GEMM core spends its time on padding: a tile's 256 rows are mostly past
// M, and filling the chip with N / 256 tiles takes a split reduction whose fp32 partials of whole
// tiles go through HBM. Here a workgroup owns 16 * RB rows of W for all M tokens, its 8 waves
// split the reduction, and the partial sums meet in LDS:
//
// * A unit of work is 128 k of one palette group; wave w takes units w, w + 8, ... Lane 16 q + n
//   dequantises words q and q + 4 of row n's eight (k = 16 q and 64 + 16 q, 16 each) into four A
//   fragments of v_mfma_f32_16x16x32_bf16, which serve every token block: each weight is
//   dequantised once per launch.
// * x is the B operand, read straight from the caches in the same k order: a load of a wave is 16
//   tokens x 4 pieces of 16 bytes of one 128-byte line. Two waves per SIMD and the compiler's own
//   order of loads cover their latency: loads pinned a unit ahead, through one or two register
//   buffers, were slower (2560 -> 4096 at M = 48: 11.5 us, 14.0 and 15.4), since the vector L1's
//   16-byte accesses, not latency, are the limit.
// * The waves' C blocks are added in wave order (deterministic); the LoRA product t B^T is one
//   more MFMA per 32 ranks in the last wave, which has the fewest units.
//
// Bound: a few dependent phases, then the reads of x, all of it by every workgroup: RB is the least
// that leaves at most one workgroup per CU. At M = 48 one layer's seven linears take 114 us
// (296 us as split 256-row tiles with whole-tile partials).
#include "plz_skinny.h"

namespace plz {
namespace sk {

constexpr int WAVES = 8;

struct Args {
  const uint16_t* x; const int32_t* packed; const float* pal;
  const uint16_t* bias; const uint16_t* t; const uint16_t* b; int rank;
  uint16_t* y; int M; int64_t N, K;
};

template <int RB, int MB>
__global__ __launch_bounds__(64 * WAVES) void skinny_fwd_kernel(const Args g) {
  extern __shared__ uint4 smem[];
  const int lane = threadIdx.x & 63, nl = lane & 15, q = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t row0 = (int64_t)blockIdx.x * (16 * RB);
  const int units = (int)(g.K / 128);
  // this lane's W rows (past N: the last one, never stored) and x rows (past M: the last one)
  const uint32_t* wp[RB];
  const float4* pp[RB];
#pragma unroll
  for (int r = 0; r < RB; ++r) {
    int64_t n = row0 + 16 * r + nl;
    n = n < g.N ? n : g.N - 1;
    wp[r] = reinterpret_cast<const uint32_t*>(g.packed) + n * (g.K / 16) + q;
    pp[r] = reinterpret_cast<const float4*>(g.pal) + n * (g.K / 256);
  }
  uint32_t xo[MB];  // in uint4
#pragma unroll
  for (int m = 0; m < MB; ++m) {
    const int t = 16 * m + nl;
    xo[m] = (uint32_t)((t < g.M ? t : g.M - 1) * (g.K / 8) + 2 * q);
  }
  const uint4* xb = reinterpret_cast<const uint4*>(g.x);

  f32x4 acc[RB][MB];
#pragma unroll
  for (int r = 0; r < RB; ++r)
#pragma unroll
    for (int m = 0; m < MB; ++m) acc[r][m] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int u = wave; u < units; u += WAVES) {
    uint32_t wf[RB][2][8];  // the words' bf16 pairs: word i's two fragments
#pragma unroll
    for (int r = 0; r < RB; ++r) {
      const float4 p = pp[r][u >> 1];
      const PalLut lut = make_lut(p.x, p.y, p.z, p.w);
      dequant16(wp[r][u * 8], lut, wf[r][0]);
      dequant16(wp[r][u * 8 + 4], lut, wf[r][1]);
    }
#pragma unroll
    for (int f = 0; f < 4; ++f) {
      uint4 xv[MB];
#pragma unroll
      for (int m = 0; m < MB; ++m)
        xv[m] = xb[xo[m] + (uint32_t)(u * 16 + 8 * (f >> 1) + (f & 1))];
#pragma unroll
      for (int r = 0; r < RB; ++r) {
        const uint32_t* o = &wf[r][f >> 1][4 * (f & 1)];
        const bf16x8 a = __builtin_bit_cast(bf16x8, u32x4{o[0], o[1], o[2], o[3]});
#pragma unroll
        for (int m = 0; m < MB; ++m)
          acc[r][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              a, __builtin_bit_cast(bf16x8, xv[m]), acc[r][m], 0, 0, 0);
      }
    }
  }
  if (wave == WAVES - 1)
    for (int k = 8 * q, k0 = 0; k0 < g.rank; k0 += 32, k += 32) {
      // fragments of t [M, rank] and B [N, rank]; zero past the rank
      uint4 tv[MB], bv[RB];
#pragma unroll
      for (int m = 0; m < MB; ++m) {
        const int t = 16 * m + nl;
        tv[m] = make_uint4(0, 0, 0, 0);
        if (k < g.rank && t < g.M)
          tv[m] = *reinterpret_cast<const uint4*>(g.t + (int64_t)t * g.rank + k);
      }
#pragma unroll
      for (int r = 0; r < RB; ++r) {
        const int64_t n = row0 + 16 * r + nl;
        bv[r] = make_uint4(0, 0, 0, 0);
        if (k < g.rank && n < g.N)
          bv[r] = *reinterpret_cast<const uint4*>(g.b + n * g.rank + k);
      }
#pragma unroll
      for (int r = 0; r < RB; ++r)
#pragma unroll
        for (int m = 0; m < MB; ++m)
          acc[r][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(bf16x8, bv[r]), __builtin_bit_cast(bf16x8, tv[m]), acc[r][m], 0,
              0, 0);
    }

  // C lane 16 q + nl: rows 4 q .. 4 q + 3 of the row block, token nl of the token block. LDS
  // [wave][row block][token block][lane]
  f32x4* part = reinterpret_cast<f32x4*>(smem);
#pragma unroll
  for (int r = 0; r < RB; ++r)
#pragma unroll
    for (int m = 0; m < MB; ++m) part[((wave * RB + r) * MB + m) * 64 + lane] = acc[r][m];
  __syncthreads();
  for (int e = threadIdx.x; e < RB * MB * 64; e += 64 * WAVES) {
    const int l = e & 63, m = (e >> 6) % MB, r = (e >> 6) / MB;
    f32x4 s = part[e];
#pragma unroll
    for (int v = 1; v < WAVES; ++v) s += part[v * (RB * MB * 64) + e];
    const int t = 16 * m + (l & 15);
    const int64_t n = row0 + 16 * r + 4 * (l >> 4);
    if (t >= g.M || n >= g.N) continue;  // N % 8 == 0: four columns are in or out together
    if (g.bias)
#pragma unroll
      for (int i = 0; i < 4; ++i) s[i] += bf2f(g.bias[n + i]);
    const uint32_t lo = f2bf2(s[0], s[1]), hi = f2bf2(s[2], s[3]);
    uint16_t* dst = g.y + (int64_t)t * g.N + n;
    if (((uintptr_t)dst & 7) == 0) {
      *reinterpret_cast<uint2*>(dst) = make_uint2(lo, hi);
    } else {
      dst[0] = (uint16_t)lo; dst[1] = (uint16_t)(lo >> 16);
      dst[2] = (uint16_t)hi; dst[3] = (uint16_t)(hi >> 16);
    }
  }
}

template <int RB, int MB>
static int launch(const Args& g, hipStream_t stream, const char* what) {
  auto kern = skinny_fwd_kernel<RB, MB>;
  const size_t lds = (size_t)WAVES * RB * MB * 1024;
  static uint64_t lds_done = 0;
  if (int rc = reserve_lds((const void*)kern, lds, lds_done, what)) return rc;
  hipLaunchKernelGGL(kern, dim3((unsigned)((g.N + 16 * RB - 1) / (16 * RB))), dim3(64 * WAVES),
                     lds, stream, g);
  return check_launch(what);
}
template <int MB>
static int launch_mb(const Args& g, int rb, hipStream_t stream, const char* what) {
  if (rb == 1) return launch<1, MB>(g, stream, what);
  if (rb == 2) return launch<2, MB>(g, stream, what);
  return launch<4, MB>(g, stream, what);
}

int fwd(const uint16_t* x, const int32_t* packed, const float* palette, const uint16_t* bias,
        const uint16_t* lora_t, const uint16_t* lora_b, int rank, uint16_t* y, int64_t M,
        int64_t N, int64_t K, int64_t cus, hipStream_t stream, const char* what) {
  const Args g = {x, packed, palette, bias, lora_t, lora_b, rank, y, (int)M, N, K};
  // the fewest row blocks that leave at most one workgroup per CU
  const int rb = N <= 16 * cus ? 1 : N <= 32 * cus ? 2 : 4;
  switch ((M + 15) / 16) {
    case 1: return launch_mb<1>(g, rb, stream, what);
    case 2: return launch_mb<2>(g, rb, stream, what);
    case 3: return launch_mb<3>(g, rb, stream, what);
    default: return launch_mb<4>(g, rb, stream, what);
  }
}

}  // namespace sk
}  // namespace plz
