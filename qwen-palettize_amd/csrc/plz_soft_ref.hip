// Soft linear in the reference's own layouts: logits (4, K, N) planes, palette (G, 4) with one
// group per group_size output columns, the Gumbel noise of its LCG samplers
// (fused_lut_kernel.cu:1245-1256, 1946-2004; triton_soft_forward.py:51-181).
//
// Everything stays in (K, N) order, in which the logits arrive and the gradients leave:
//   plz_soft_ref_build_w  W [K, N] bf16 from the planes, the noise drawn in the kernel
//   (y = x W and grad_x = grad_y W^T are then the dense GEMMs with W's two roles exchanged)
//   plz_soft_ref_bwd      dW^T = x^T grad_y [K, N] as fp32 partials from the dW GEMM, then one
//                         streaming pass that draws the noise again, recomputes P in fp32, writes
//                         grad_logits (4, K, N) and sums the palette gradient
// so no plane is transposed and no noise tensor exists: per weight 8 B of logits read and 2 B (with
// the logits as read, 10 B) written forward; 8 B + 4 B per split read and 8 B written backward. Both passes are bound by
// their VALU, half of it quarter-rate (per weight 8 logs, 4 exponentials, 9 32-bit multiplies):
// 2560 x 4096 in 52 us forward, 58 with the copy, and 67 us backward (105, 189 and 210 MB). A training
// pass of that linear with LoRA at 2048 rows: 920 us through the native layout (two plane
// transposes of 206 us, noise drawn into and read from an fp32 tensor) -> 350 us.
#include "plz_soft_ref.h"
#include "palettize_hip.h"

namespace plz {
namespace sref {

// The LCG draw of class c of weight (k, n): idx = (k N + n) 4 + c in uint32 arithmetic. ARITH: the
// Triton hash (shifts of a signed value). -log(-log u) of u in [1e-7, 1 - 2^-24] sees normal
// inputs only, for which log_normal is logf.
template <bool ARITH>
__device__ __forceinline__ float lcg_noise(uint32_t seed, uint32_t idx) {
  auto shr = [](uint32_t x, int s) { return ARITH ? (uint32_t)((int32_t)x >> s) : x >> s; };
  uint32_t x = seed ^ (idx * 0x9E3779B9u);
  x ^= shr(x, 13);
  x = x * 1103515245u + 12345u;
  x ^= shr(x, 17);
  x = x * 1103515245u + 12345u;
  const float u = fmaxf((float)(x & 0xFFFFFFu) * (1.0f / 16777216.0f), 1e-7f);
  return -log_normal(-log_normal(u));
}

// P_c = softmax_c((l_c + z_c) / tau), one reciprocal of the sum, as build_w_two computes it
__device__ __forceinline__ void probs4(const float (&l)[4], const float (&z)[4], float inv_tau,
                                       float (&P)[4]) {
  float a[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) a[c] = (l[c] + z[c]) * inv_tau;
  const float m = fmaxf(fmaxf(a[0], a[1]), fmaxf(a[2], a[3]));
  float s = 0.f;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    P[c] = __expf(a[c] - m);
    s += P[c];
  }
  const float rs = 1.f / s;
#pragma unroll
  for (int c = 0; c < 4; ++c) P[c] *= rs;
}

struct Weights {
  const uint16_t* logits;  // (4, K, N)
  const void* pal;         // (G, 4), pal_dtype
  int64_t K, N, group_size;
  float inv_tau;
  uint32_t seed;
  int f16, pal_dtype;
};
__device__ __forceinline__ float elem(const void* p, int dtype, int64_t i) {
  if (dtype == PLZ_DT_FP32) return reinterpret_cast<const float*>(p)[i];
  const uint32_t b = reinterpret_cast<const uint16_t*>(p)[i];
  return dtype == PLZ_DT_FP16 ? h2f(b) : bf2f(b);
}
__device__ __forceinline__ void store_elem(void* p, int dtype, int64_t i, float v) {
  if (dtype == PLZ_DT_FP32) reinterpret_cast<float*>(p)[i] = v;
  else reinterpret_cast<uint16_t*>(p)[i] = (uint16_t)(dtype == PLZ_DT_FP16 ? f2h(v) : f2bf(v));
}
// the palettes of columns n .. n + 3
__device__ __forceinline__ void load_palettes(const Weights& w, int64_t n, float (&pal)[4][4]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int64_t g = (n + i) / w.group_size;
#pragma unroll
    for (int c = 0; c < 4; ++c) pal[i][c] = elem(w.pal, w.pal_dtype, 4 * g + c);
  }
}
// l[i][c]: the logits of weights e .. e + 3 of the flat (K, N) index
__device__ __forceinline__ void load_logits(const Weights& w, int64_t e, uint2 (&v)[4]) {
#pragma unroll
  for (int c = 0; c < 4; ++c)
    v[c] = *reinterpret_cast<const uint2*>(w.logits + c * w.K * w.N + e);
}
__device__ __forceinline__ void unpack_logits(const Weights& w, const uint2 (&v)[4],
                                              float (&l)[4][4]) {
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const uint32_t b[4] = {v[c].x & 0xffffu, v[c].x >> 16, v[c].y & 0xffffu, v[c].y >> 16};
#pragma unroll
    for (int i = 0; i < 4; ++i) l[i][c] = w.f16 ? h2f(b[i]) : bf2f(b[i]);
  }
}

// A workgroup covers 256 columns (4 per lane) and KR rows, its wave w rows w, w + 4, ...
constexpr int KR = 32;

// keep (optional): the logits as read
template <bool ARITH>
__global__ __launch_bounds__(256) void build_kernel(const Weights w, int mode,
                                                    uint16_t* __restrict__ out,
                                                    uint16_t* __restrict__ keep) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t n = (int64_t)blockIdx.x * 256 + 4 * lane;
  if (n >= w.N) return;
  float pal[4][4];
  load_palettes(w, n, pal);
  const int64_t k0 = (int64_t)blockIdx.y * KR;
#pragma unroll 2
  for (int kk = wave; kk < KR; kk += 4) {
    const int64_t k = k0 + kk;
    if (k >= w.K) break;
    const int64_t e = k * w.N + n;
    uint2 v[4];
    load_logits(w, e, v);
    if (keep)
#pragma unroll
      for (int c = 0; c < 4; ++c) *reinterpret_cast<uint2*>(keep + c * w.K * w.N + e) = v[c];
    float l[4][4];
    unpack_logits(w, v, l);
    uint32_t o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t idx = (uint32_t)(e + i) * 4u;
      float r;
      if (mode == PLZ_W_HARD_PLAIN) {
        // argmax of the plain logits, first maximum wins
        r = pal[i][0];
        float best = l[i][0];
#pragma unroll
        for (int c = 1; c < 4; ++c)
          if (l[i][c] > best) { best = l[i][c]; r = pal[i][c]; }
      } else {
        float z[4], P[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) z[c] = lcg_noise<ARITH>(w.seed, idx + c);
        probs4(l[i], z, w.inv_tau, P);
        r = pal[i][0];
        float best = P[0], ws = P[0] * pal[i][0];
#pragma unroll
        for (int c = 1; c < 4; ++c) {
          if (P[c] > best) { best = P[c]; r = pal[i][c]; }
          ws += P[c] * pal[i][c];
        }
        if (mode == PLZ_W_SOFT) r = ws;
      }
      o[i] = f2bf(r);
    }
    *reinterpret_cast<uint2*>(out + e) = make_uint2(o[0] | (o[1] << 16), o[2] | (o[3] << 16));
  }
}

// grad_logits (optional) and the per-column palette sums of KR rows, [row block][N][4] fp32
template <bool ARITH>
__global__ __launch_bounds__(256) void bwd_kernel(const Weights w, const float* __restrict__ part,
                                                  int Z, float glog_scale,
                                                  uint16_t* __restrict__ grad_logits,
                                                  float* __restrict__ cols) {
  __shared__ float4 red[3][4][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t n = (int64_t)blockIdx.x * 256 + 4 * lane, KN = w.K * w.N;
  const bool live = n < w.N;
  float pal[4][4], sp[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int c = 0; c < 4; ++c) pal[i][c] = sp[i][c] = 0.f;
  if (live) load_palettes(w, n, pal);
  const int64_t k0 = (int64_t)blockIdx.y * KR;
#pragma unroll 2
  for (int kk = wave; kk < KR; kk += 4) {
    const int64_t k = k0 + kk;
    if (k >= w.K || !live) break;
    const int64_t e = k * w.N + n;
    uint2 v[4];
    load_logits(w, e, v);
    float4 g4 = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int z = 0; z < Z; ++z) {  // the splits in order
      const float4 d = *reinterpret_cast<const float4*>(part + z * KN + e);
      g4.x += d.x; g4.y += d.y; g4.z += d.z; g4.w += d.w;
    }
    const float gw[4] = {g4.x, g4.y, g4.z, g4.w};
    float l[4][4];
    unpack_logits(w, v, l);
    uint32_t o[4][4];  // [class][weight]
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t idx = (uint32_t)(e + i) * 4u;
      float z[4], P[4], ws = 0.f;
#pragma unroll
      for (int c = 0; c < 4; ++c) z[c] = lcg_noise<ARITH>(w.seed, idx + c);
      probs4(l[i], z, w.inv_tau, P);
#pragma unroll
      for (int c = 0; c < 4; ++c) ws += P[c] * pal[i][c];
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const float gp = gw[i] * P[c];
        sp[i][c] += gp;
        const float gl = glog_scale * gp * (pal[i][c] - ws);
        o[c][i] = w.f16 ? f2h(gl) : f2bf(gl);
      }
    }
    if (grad_logits)
#pragma unroll
      for (int c = 0; c < 4; ++c)
        *reinterpret_cast<uint2*>(grad_logits + c * KN + e) =
            make_uint2(o[c][0] | (o[c][1] << 16), o[c][2] | (o[c][3] << 16));
  }
  // the four waves' sums of a column, in wave order
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (wave > 0) red[wave - 1][i][lane] = make_float4(sp[i][0], sp[i][1], sp[i][2], sp[i][3]);
  __syncthreads();
  if (wave > 0 || !live) return;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
#pragma unroll
    for (int u = 0; u < 3; ++u) {
      const float4 d = red[u][i][lane];
      sp[i][0] += d.x; sp[i][1] += d.y; sp[i][2] += d.z; sp[i][3] += d.w;
    }
    *reinterpret_cast<float4*>(cols + ((int64_t)blockIdx.y * w.N + n + i) * 4) =
        make_float4(sp[i][0], sp[i][1], sp[i][2], sp[i][3]);
  }
}

// Palette gradient (G, 4): group g = its columns' sums over all row blocks, fixed order; groups that
// no column uses are zero. One workgroup per group.
__global__ __launch_bounds__(512) void pal_kernel(const float4* __restrict__ cols, int64_t blocks,
                                                  int64_t N, int64_t group_size, void* out,
                                                  int dtype) {
  __shared__ float4 red[512];
  const int64_t g = blockIdx.x, n0 = g * group_size;
  const int64_t nc = n0 >= N ? 0 : (n0 + group_size < N ? group_size : N - n0);
  float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
  if (blocks == 1) {
#pragma unroll 8
    for (int64_t c = threadIdx.x; c < nc; c += 512) {
      const float4 d = cols[n0 + c];
      s.x += d.x; s.y += d.y; s.z += d.z; s.w += d.w;
    }
  } else {
    for (int64_t c = threadIdx.x & 255; c < nc; c += 256) {  // two row blocks of 256 columns a step
      const float4* p = cols + n0 + c;
#pragma unroll 8
      for (int64_t b = threadIdx.x >> 8; b < blocks; b += 2) {
        const float4 d = p[b * N];
        s.x += d.x; s.y += d.y; s.z += d.z; s.w += d.w;
      }
    }
  }
  red[threadIdx.x] = s;
  for (int h = 256; h >= 1; h >>= 1) {
    __syncthreads();
    if ((int)threadIdx.x < h) {
      const float4 a = red[threadIdx.x], b = red[threadIdx.x + h];
      red[threadIdx.x] = make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w);
    }
  }
  __syncthreads();
  if (threadIdx.x < 4)
    store_elem(out, dtype, 4 * g + threadIdx.x, reinterpret_cast<const float*>(red)[threadIdx.x]);
}

// One thread per native palette entry: a 16-byte store of its row's group.
__global__ void expand_kernel(const void* pal, int dtype, float4* __restrict__ out, int64_t total,
                              int64_t kg, int64_t group_size) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= total) return;
  const int64_t g = t / kg / group_size * 4;
  out[t] = make_float4(elem(pal, dtype, g), elem(pal, dtype, g + 1), elem(pal, dtype, g + 2),
                       elem(pal, dtype, g + 3));
}

static int64_t row_blocks(int64_t K) { return (K + KR - 1) / KR; }
static size_t cols_bytes(int64_t N, int64_t K) { return (size_t)row_blocks(K) * N * 16; }

static int check(const uint16_t* logits, int logits_dtype, const void* palette, int pal_dtype,
                 int64_t group_size, float tau, int64_t K, int64_t N, const char* what) {
  PLZ_REQUIRE(K > 0 && N > 0 && K % 8 == 0 && N % 8 == 0,
              "%s: K (%lld) and N (%lld) must be positive multiples of 8", what, (long long)K,
              (long long)N);
  PLZ_REQUIRE(logits_dtype == PLZ_DT_BF16 || logits_dtype == PLZ_DT_FP16,
              "%s: logits dtype must be bf16 or fp16", what);
  PLZ_REQUIRE(pal_dtype == PLZ_DT_BF16 || pal_dtype == PLZ_DT_FP16 || pal_dtype == PLZ_DT_FP32,
              "%s: palette dtype must be bf16, fp16 or fp32", what);
  PLZ_REQUIRE(group_size > 0 && tau > 0.f, "%s: group_size and tau must be positive", what);
  PLZ_REQUIRE(logits && palette && ((uintptr_t)logits & 7) == 0 &&
                  ((uintptr_t)palette & (pal_dtype == PLZ_DT_FP32 ? 3 : 1)) == 0,
              "%s: null or misaligned logits or palette", what);
  PLZ_REQUIRE(row_blocks(K) <= 65535, "%s: K (%lld) is too large", what, (long long)K);
  return PLZ_OK;
}

}  // namespace sref
}  // namespace plz

using namespace plz;
using namespace plz::sref;

extern "C" {

int plz_palette_expand(const void* palette, int dtype, float* out, int64_t N, int64_t kg,
                       int64_t group_size, void* stream) {
  PLZ_REQUIRE(N >= 0 && kg >= 0 && group_size > 0, "plz_palette_expand: bad shape");
  PLZ_REQUIRE(dtype == PLZ_DT_BF16 || dtype == PLZ_DT_FP16 || dtype == PLZ_DT_FP32,
              "plz_palette_expand: palette must be bf16, fp16 or fp32");
  if (N == 0 || kg == 0) return PLZ_OK;
  PLZ_REQUIRE(palette && out && ((uintptr_t)out & 15) == 0,
              "plz_palette_expand: null or misaligned pointer");
  const int64_t total = N * kg;
  hipLaunchKernelGGL(expand_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0,
                     (hipStream_t)stream, palette, dtype, reinterpret_cast<float4*>(out), total, kg,
                     group_size);
  return check_launch("plz_palette_expand");
}

int plz_palette_fold(const float* grad, void* out, int dtype, int64_t n_groups, int64_t N,
                     int64_t kg, int64_t group_size, void* stream) {
  PLZ_REQUIRE(N > 0 && kg > 0 && group_size > 0 && n_groups <= 0x7fffffff &&
                  n_groups >= (N + group_size - 1) / group_size,
              "plz_palette_fold: bad shape");
  PLZ_REQUIRE(dtype == PLZ_DT_BF16 || dtype == PLZ_DT_FP16 || dtype == PLZ_DT_FP32,
              "plz_palette_fold: out must be bf16, fp16 or fp32");
  PLZ_REQUIRE(grad && out && ((uintptr_t)grad & 15) == 0,
              "plz_palette_fold: null or misaligned pointer");
  // [N, kg, 4] as one block of N kg columns in groups of group_size kg
  hipLaunchKernelGGL(pal_kernel, dim3((unsigned)n_groups), dim3(512), 0, (hipStream_t)stream,
                     reinterpret_cast<const float4*>(grad), (int64_t)1, N * kg, group_size * kg,
                     out, dtype);
  return check_launch("plz_palette_fold");
}

int plz_soft_ref_build_w_copy(const uint16_t* logits, int logits_dtype, const void* palette,
                              int palette_dtype, int64_t group_size, int triton_hash, uint32_t seed,
                              float tau, int mode, uint16_t* w, uint16_t* logits_copy, int64_t K,
                              int64_t N, void* stream) {
  const char* what = "plz_soft_ref_build_w";
  if (int rc = check(logits, logits_dtype, palette, palette_dtype, group_size, tau, K, N, what))
    return rc;
  PLZ_REQUIRE(mode == PLZ_W_SOFT || mode == PLZ_W_HARD_NOISY || mode == PLZ_W_HARD_PLAIN,
              "%s: unknown mode %d", what, mode);
  PLZ_REQUIRE(w && (((uintptr_t)w | (uintptr_t)logits_copy) & 7) == 0,
              "%s: w must be non-null, w and logits_copy 8-byte aligned", what);
  const Weights g = {logits, palette, K, N, group_size, 1.f / tau, seed,
                     logits_dtype == PLZ_DT_FP16, palette_dtype};
  const dim3 grid((unsigned)((N + 255) / 256), (unsigned)row_blocks(K));
  auto kern = triton_hash ? build_kernel<true> : build_kernel<false>;
  hipLaunchKernelGGL(kern, grid, dim3(256), 0, (hipStream_t)stream, g, mode, w, logits_copy);
  return check_launch(what);
}

int plz_soft_ref_build_w(const uint16_t* logits, int logits_dtype, const void* palette,
                         int palette_dtype, int64_t group_size, int triton_hash, uint32_t seed,
                         float tau, int mode, uint16_t* w, int64_t K, int64_t N, void* stream) {
  return plz_soft_ref_build_w_copy(logits, logits_dtype, palette, palette_dtype, group_size,
                                   triton_hash, seed, tau, mode, w, nullptr, K, N, stream);
}

size_t plz_soft_ref_bwd_workspace(int64_t M, int64_t N, int64_t K) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  return cols_bytes(N, K) + (size_t)g2::dw_splits(K, N, M) * K * N * sizeof(float);
}

int plz_soft_ref_bwd(const uint16_t* x, const uint16_t* grad_y, const uint16_t* logits,
                     int logits_dtype, const void* palette, int palette_dtype, int64_t n_groups,
                     int64_t group_size, int triton_hash, uint32_t seed, float tau,
                     int scale_grad_by_inv_tau, uint16_t* grad_logits, void* grad_palette,
                     void* workspace, size_t workspace_bytes, int64_t M, int64_t N, int64_t K,
                     void* stream) {
  const char* what = "plz_soft_ref_bwd";
  if (int rc = check(logits, logits_dtype, palette, palette_dtype, group_size, tau, K, N, what))
    return rc;
  PLZ_REQUIRE(M > 0, "%s: M must be positive", what);
  PLZ_REQUIRE(n_groups >= (N + group_size - 1) / group_size && n_groups <= 0x7fffffff,
              "%s: %lld groups for %lld columns in groups of %lld", what, (long long)n_groups,
              (long long)N, (long long)group_size);
  PLZ_REQUIRE(x && grad_y && grad_palette && (((uintptr_t)x | (uintptr_t)grad_y) & 15) == 0 &&
                  ((uintptr_t)grad_logits & 7) == 0 &&
                  ((uintptr_t)grad_palette & (palette_dtype == PLZ_DT_FP32 ? 3 : 1)) == 0,
              "%s: null or misaligned pointer", what);
  const size_t need = plz_soft_ref_bwd_workspace(M, N, K);
  if (!workspace || ((uintptr_t)workspace & 15) || workspace_bytes < need) {
    set_error("%s: workspace of %zu bytes (16-byte aligned) needed, %zu given", what, need,
              workspace_bytes);
    return PLZ_EWORKSPACE;
  }
  hipStream_t st = (hipStream_t)stream;
  float* cols = reinterpret_cast<float*>(workspace);
  float* part = reinterpret_cast<float*>(static_cast<uint8_t*>(workspace) + cols_bytes(N, K));
  const int z = g2::dw_splits(K, N, M);
  if (int rc = g2::dw_partials(x, grad_y, part, z, K, N, M, st, what)) return rc;
  const Weights g = {logits, palette, K, N, group_size, 1.f / tau, seed,
                     logits_dtype == PLZ_DT_FP16, palette_dtype};
  const float gs = scale_grad_by_inv_tau ? 1.f / tau : 1.f;
  const dim3 grid((unsigned)((N + 255) / 256), (unsigned)row_blocks(K));
  if (triton_hash)
    hipLaunchKernelGGL(bwd_kernel<true>, grid, dim3(256), 0, st, g, part, z, gs, grad_logits, cols);
  else
    hipLaunchKernelGGL(bwd_kernel<false>, grid, dim3(256), 0, st, g, part, z, gs, grad_logits, cols);
  hipLaunchKernelGGL(pal_kernel, dim3((unsigned)n_groups), dim3(512), 0, st,
                     reinterpret_cast<const float4*>(cols), row_blocks(K), N, group_size,
                     grad_palette, palette_dtype);
  return check_launch(what);
}

}  // extern "C"
