// Dense MFMA GEMM on 128x128 tiles: the forward and grad_x GEMMs (rows x rows, rows x columns) of
// a few hundred to a few thousand rows.
//
// The 256x256 core (plz_gemm2) fills 256 CUs with 256 tiles; a 1000 x 4096 output has 64, so it
// splits their reduction and moves 256 KB of fp32 partials per part through HBM, and its rows are
// padded to 256. Tiles of 128x128 make four times as many workgroups (4 waves of 64x64), at the
// price of twice the operand bytes and LDS reads per MFMA (4 fragments per 4
// v_mfma_f32_32x32x16_bf16). Only launches that still leave CUs idle split the reduction (fp32
// partials [split][I][J] without padding, summed in split order by reduce_kernel).
//
// The stage loop is the 256 core's: slots of BK = 64, the barrier that completes the next stage's
// copies before a stage's last k-step, a later stage's copies behind it. Two slots (64 KB) where
// two workgroups share a CU, one's waits covered by the other's MFMAs; four, copied three stages
// ahead, where a launch has at most one per CU (1000 x 4096 x 2560: 31.4 us with two, 28.0 with
// four). Bound by the operands' way from L2 (13 TB/s over the chip there, 750 TFLOP/s). Dense
// forward, 256 core -> this one: 2560 -> 4096 at M = 128 / 777 / 2048 32.0 / 47.5 / 60.8 ->
// 17.3 / 26.4 / 44.8 us, 2560 -> 1024 30.1 / 34.5 / 37.3 -> 13.9 / 19.8 / 24.1.
#include "plz_gemm2.cuh"
#include "plz_mid.h"

namespace plz {
namespace mid {

using g2::BK;
using g2::f32x16;
using g2::lds_u8;
using g2::row_chunk;
using g2::row_swz;
using g2::stage_barrier;
using g2::wait_vmcnt;

constexpr int T = 128, NT = 256;
constexpr int OPB = T * BK * 2;        // bytes of an operand's stage (16 KB)
constexpr int CI = OPB / 16 / NT;      // 16-byte copies per thread and operand (4)
constexpr int RS = T * 2 + 16;         // output staging row in bytes

// Col tile [r][128]: 16-byte chunk c of reduction row kr at c ^ col_swz(kr) (free of bank
// conflicts for the transposing reads: four rows x four chunks of a 32-lane half are distinct)
__device__ __forceinline__ int col_chunk(int kr, int c) { return kr * 16 + (c ^ g2::col_swz(kr)); }

struct Dma {
  BufRsrc r;
  uint32_t off[CI];
};
__device__ __forceinline__ Dma row_dma(const uint16_t* p, int64_t ld, int64_t row0, int64_t nrows) {
  Dma d;
  d.r = make_rsrc(p, (uint32_t)(nrows * ld * 2));
#pragma unroll
  for (int it = 0; it < CI; ++it) {
    const int pch = it * NT + threadIdx.x, row = pch >> 3, c = (pch & 7) ^ row_swz(row);
    int64_t gr = row0 + row;
    gr = gr < nrows ? gr : nrows - 1;  // rows past the end: any valid row
    d.off[it] = (uint32_t)((gr * ld + c * 8) * 2);
  }
  return d;
}
__device__ __forceinline__ Dma col_dma(const uint16_t* p, int64_t ld, int64_t col0, int64_t ncols,
                                       int64_t rtotal) {
  Dma d;
  d.r = make_rsrc(p, (uint32_t)(rtotal * ld * 2));
#pragma unroll
  for (int it = 0; it < CI; ++it) {
    const int pch = it * NT + threadIdx.x, kr = pch >> 4, c = (pch & 15) ^ g2::col_swz(kr);
    int64_t gc = col0 + c * 8;
    gc = gc < ncols ? gc : 0;  // chunks past the end: any valid chunk
    d.off[it] = (uint32_t)((kr * ld + gc) * 2);
  }
  return d;
}
__device__ __forceinline__ void copy_tile(lds_u8* lds, const Dma& d, uint32_t soff) {
  const int wbase = __builtin_amdgcn_readfirstlane((threadIdx.x >> 6) * 1024);
#pragma unroll
  for (int it = 0; it < CI; ++it)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(d.r, lds + it * NT * 16 + wbase, 16, d.off[it], soff,
                                             0, 0);
}
// register copies of a partial stage or the rank segment (zero past the reduction and the rows)
__device__ __forceinline__ void masked_rows(uint4* lds, const uint16_t* p, int64_t ld, int64_t row0,
                                            int64_t nrows, int64_t r0, int64_t rend) {
#pragma unroll
  for (int it = 0; it < CI; ++it) {
    const int ch = it * NT + threadIdx.x, row = ch >> 3, c = ch & 7;
    const int64_t gr = row0 + row, gk = r0 + 8 * c;
    uint4 v = make_uint4(0, 0, 0, 0);
    if (gr < nrows && gk < rend) v = *reinterpret_cast<const uint4*>(p + gr * ld + gk);
    lds[row_chunk(row, c)] = v;
  }
}
__device__ __forceinline__ void masked_cols(uint4* lds, const uint16_t* p, int64_t ld, int64_t col0,
                                            int64_t ncols, int64_t r0, int64_t rend) {
#pragma unroll
  for (int it = 0; it < CI; ++it) {
    const int ch = it * NT + threadIdx.x, kr = ch >> 4, c = ch & 15;
    const int64_t gc = col0 + 8 * c, gk = r0 + kr;
    uint4 v = make_uint4(0, 0, 0, 0);
    if (gc < ncols && gk < rend) v = *reinterpret_cast<const uint4*>(p + gk * ld + gc);
    lds[col_chunk(kr, c)] = v;
  }
}

__device__ __forceinline__ bf16x8 frag_col(const lds_u8* lds, int rowbase, int ks, int lane) {
  const int j = lane >> 4, i = lane & 15, t = i >> 2, q = i & 3;
  const int row = rowbase + 16 * (j & 1) + 4 * q;
  const int kr1 = 16 * ks + 8 * (j >> 1) + t, c = row >> 3, off = (row & 7) * 2;
  const g2::v4i16 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (g2::lds_v4i16*)(lds + col_chunk(kr1, c) * 16 + off));
  const g2::v4i16 v2 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (g2::lds_v4i16*)(lds + col_chunk(kr1 + 4, c) * 16 + off));
  typedef short v8i16 __attribute__((ext_vector_type(8)));
  const v8i16 v = __builtin_shufflevector(v1, v2, 0, 1, 2, 3, 4, 5, 6, 7);
  return __builtin_bit_cast(bf16x8, v);
}
template <bool B_COL>
__device__ __forceinline__ void frags(const lds_u8* a_s, const lds_u8* b_s, int ks, int wi, int wj,
                                      int lane, bf16x8 (&a)[2], bf16x8 (&b)[2]) {
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    a[i] = g2::frag_row((const uint4*)a_s, wi * 64 + 32 * i, ks, lane);
    b[i] = B_COL ? frag_col(b_s, wj * 64 + 32 * i, ks, lane)
                 : g2::frag_row((const uint4*)b_s, wj * 64 + 32 * i, ks, lane);
  }
}
__device__ __forceinline__ void mma(f32x16 (&acc)[2][2], const bf16x8 (&a)[2], const bf16x8 (&b)[2]) {
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
      acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
}

// One stage (plz_gemm2's mma_stage_pipe): as_, bs_ this stage's tiles with k-step 0 already in
// a0 / b0, na, nb the next stage's; bar() completes the next stage's copies, dma() refills this
// stage's slot (da: the same LDS as as_, written only after the barrier).
template <bool B_COL, typename Bar, typename DmaF>
__device__ __forceinline__ void stage_pipe(const lds_u8* __restrict__ as_,
                                           const lds_u8* __restrict__ bs_,
                                           const lds_u8* __restrict__ na,
                                           const lds_u8* __restrict__ nb, lds_u8* __restrict__ da,
                                           f32x16 (&acc)[2][2], int wi, int wj, int lane,
                                           bf16x8 (&a0)[2], bf16x8 (&b0)[2], Bar&& bar,
                                           DmaF&& dma) {
  bf16x8 a1[2], b1[2];
  frags<B_COL>(as_, bs_, 1, wi, wj, lane, a1, b1);
  __builtin_amdgcn_sched_barrier(0);
  mma(acc, a0, b0);
  frags<B_COL>(as_, bs_, 2, wi, wj, lane, a0, b0);
  __builtin_amdgcn_sched_barrier(0);
  mma(acc, a1, b1);
  frags<B_COL>(as_, bs_, 3, wi, wj, lane, a1, b1);
  __builtin_amdgcn_sched_barrier(0);
  mma(acc, a0, b0);
  __builtin_amdgcn_sched_barrier(0);
  bar();
  __builtin_amdgcn_sched_barrier(0);
  dma(da);
  frags<B_COL>(na, nb, 0, wi, wj, lane, a0, b0);
  __builtin_amdgcn_sched_barrier(0);
  mma(acc, a1, b1);
  __builtin_amdgcn_sched_barrier(0);
}

// eight rounded outputs at (i, j), as plz_gemm2 stores them
__device__ __forceinline__ void store8(const Args& g, u32x4 v, int64_t i, int64_t j) {
  if (g.res) v = g2::add_residual8(v, g.res + i * g.ldres + j);
  __builtin_nontemporal_store(v, reinterpret_cast<u32x4*>(g.c + i * g.ldc + j));
}

template <bool B_COL, int NS>
__global__ __launch_bounds__(NT, NS == 2 ? 2 : 1) void mid_kernel(const Args g) {
  extern __shared__ uint4 smem[];
  lds_u8* lbase = (lds_u8*)smem;
  // items (split, tile) in XCD-contiguous ranges; tile-columns within groups of 4 tile-rows
  const int tiles = g.tiles_i * g.tiles_j;
  const g2::Item itm = g2::map_item(tiles, false, 0, 0, (int)blockIdx.x, (int)blockIdx.z,
                                    (int)gridDim.z);
  int ti, tj;
  g2::tile_coords(4, g.tiles_i, g.tiles_j, itm.bid, ti, tj);
  const int z = itm.zsl;
  const int64_t i0 = (int64_t)ti * T, j0 = (int64_t)tj * T;
  const int64_t rbeg = (int64_t)z * g.r_split, rend = min(g.R, rbeg + g.r_split);
  const int64_t rlen = rend > rbeg ? rend - rbeg : 0;
  const int nfull = (int)(rlen / BK);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, wi = wave >> 1, wj = wave & 1;

  f32x16 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  const Dma dA = row_dma(g.a, g.lda, i0, g.I);
  const Dma dB = B_COL ? col_dma(g.b, g.ldb, j0, g.J, g.R) : row_dma(g.b, g.ldb, j0, g.J);
  auto slot = [&](int kt) { return lbase + (kt & (NS - 1)) * 2 * OPB; };
  auto copy = [&](int kt, lds_u8* s) {  // past the last stage: that one again
    const int64_t r0 = rbeg + (int64_t)(kt < nfull ? kt : nfull - 1) * BK;
    copy_tile(s, dA, (uint32_t)(r0 * 2));
    copy_tile(s + OPB, dB, (uint32_t)(B_COL ? r0 * g.ldb * 2 : r0 * 2));
  };
  bf16x8 a0[2], b0[2];
  if (nfull > 0) {
#pragma unroll
    for (int u = 0; u < NS; ++u) copy(u, slot(u));
    wait_vmcnt<(NS - 1) * 2 * CI>();  // stage 0 has landed; the others may be in flight
    stage_barrier();
    frags<B_COL>(slot(0), slot(0) + OPB, 0, wi, wj, lane, a0, b0);
  }
  for (int kt = 0; kt < nfull; ++kt) {
    lds_u8* const cs = slot(kt);
    const lds_u8* const ns = slot(kt + 1);
    stage_pipe<B_COL>(
        cs, cs + OPB, ns, ns + OPB, cs, acc, wi, wj, lane, a0, b0,
        [&] {
          wait_vmcnt<(NS - 2) * 2 * CI>();  // this wave's copies of stage kt + 1
          stage_barrier();
        },
        [&](lds_u8* d) { copy(kt + NS, d); });
  }
  __builtin_amdgcn_s_waitcnt(0);  // the repeated copies past the last stage
  __syncthreads();
  // the partial stage and the rank segment, synchronously through slot 0
  const bool tail = rlen % BK != 0, lora = g.R2 > 0 && z == 0;
  for (int s = 0; s < 2; ++s) {
    if (!(s == 0 ? tail : lora)) continue;  // uniform
    uint4* As = (uint4*)lbase;
    uint4* Bs = (uint4*)(lbase + OPB);
    int len;
    if (s == 0) {
      const int64_t r0 = rbeg + (int64_t)nfull * BK;
      masked_rows(As, g.a, g.lda, i0, g.I, r0, rend);
      if (B_COL) masked_cols(Bs, g.b, g.ldb, j0, g.J, r0, rend);
      else masked_rows(Bs, g.b, g.ldb, j0, g.J, r0, rend);
      len = (int)(rend - r0);
    } else {
      masked_rows(As, g.a2, g.R2, i0, g.I, 0, g.R2);
      if (B_COL) masked_cols(Bs, g.b2, g.J, j0, g.J, 0, g.R2);
      else masked_rows(Bs, g.b2, g.R2, j0, g.J, 0, g.R2);
      len = g.R2;
    }
    __syncthreads();
    for (int ks = 0; ks < (len + 15) / 16; ++ks) {
      bf16x8 a[2], b[2];
      frags<B_COL>(lbase, lbase + OPB, ks, wi, wj, lane, a, b);
      mma(acc, a, b);
    }
    __syncthreads();
  }

  // acc[x][y][e]: row wi*64 + 32 x + 8 (e / 4) + 4 (lane / 32) + e % 4, col wj*64 + 32 y + lane % 32
  if (g.splits > 1) {
    float* dst = g.part + (int64_t)z * g.I * g.J;
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int y = 0; y < 2; ++y) {
        const int64_t j = j0 + wj * 64 + 32 * y + (lane & 31);
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int64_t i = i0 + wi * 64 + 32 * x + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3);
          if (i < g.I && j < g.J) dst[i * g.J + j] = acc[x][y][e];
        }
      }
    return;
  }
#pragma unroll
  for (int y = 0; y < 2; ++y) {
    const int col = wj * 64 + 32 * y + (lane & 31);
    const float bj = g.bias && j0 + col < g.J ? bf2f(g.bias[j0 + col]) : 0.f;
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int row = wi * 64 + 32 * x + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3);
        *reinterpret_cast<__attribute__((address_space(3))) uint16_t*>(lbase + row * RS + col * 2) =
            (uint16_t)f2bf(acc[x][y][e] + bj);
      }
  }
  __syncthreads();
#pragma unroll
  for (int it = 0; it < T * T / 8 / NT; ++it) {
    const int ch = it * NT + threadIdx.x, row = ch >> 4, c8 = (ch & 15) * 8;
    const int64_t i = i0 + row, j = j0 + c8;
    if (i < g.I && j < g.J) {
      u32x4 v = *reinterpret_cast<const __attribute__((address_space(3))) u32x4*>(lbase + row * RS + c8 * 2);
      store8(g, v, i, j);
    }
  }
}

// C = the splits' partials in order (+ bias), rounded (+ res, rounded): 8 columns per thread
__global__ __launch_bounds__(256) void reduce_kernel(const Args g) {
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x, n8 = g.J / 8;
  if (t >= g.I * n8) return;
  const int64_t i = t / n8, j = (t - i * n8) * 8, IJ = g.I * g.J;
  const float* p = g.part + i * g.J + j;
  float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  for (int z = 0; z < g.splits; ++z) {
    const float4 u = *reinterpret_cast<const float4*>(p + z * IJ);
    const float4 v = *reinterpret_cast<const float4*>(p + z * IJ + 4);
    s[0] += u.x; s[1] += u.y; s[2] += u.z; s[3] += u.w;
    s[4] += v.x; s[5] += v.y; s[6] += v.z; s[7] += v.w;
  }
  if (g.bias)
#pragma unroll
    for (int e = 0; e < 8; ++e) s[e] += bf2f(g.bias[j + e]);
  u32x4 v;
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = f2bf2(s[2 * e], s[2 * e + 1]);
  store8(g, v, i, j);
}

size_t workspace(int64_t I, int64_t J, int z) {
  return z > 1 ? (size_t)z * I * J * sizeof(float) : 0;
}

// Modelled time of z splits: a workgroup alone on its CU takes 0.64 us per stage, one of two
// 1.08 (1000 and 2048 x 4096 x 2560: 28.0 us of 256 workgroups, 44.8 of 512); a launch moves from
// one rate to the other over its first half wave of second workgroups (512 x 9728 x 2560, 304
// workgroups: 36 us). Splits add 3 us of launch and 8 B per output and split at 5 TB/s.
Plan plan(int64_t I, int64_t J, int64_t R, int64_t cus) {
  const int64_t tiles = ((I + T - 1) / T) * ((J + T - 1) / T);
  Plan best{1, 1e300};
  for (int z = 1; z <= 16; ++z) {
    const int64_t len = g2::split_len(R, z);
    if (z > 1 && (len < 4 * BK || (int64_t)(z - 1) * len >= R)) break;  // >= 4 stages, none empty
    const int64_t wg = tiles * z, full = wg / (2 * cus), rest = wg % (2 * cus);
    const double st = (double)((len + BK - 1) / BK), over = 2.0 * (double)(rest - cus) / (double)cus;
    double t = (double)full * (1.08 * st + 4.0) + (z > 1 ? 3.0 + z * 8.0 * (double)I * J / 5.0e6 : 0.0);
    if (rest > 0) t += (0.64 + 0.44 * (over < 0.0 ? 0.0 : over > 1.0 ? 1.0 : over)) * st + 3.0;
    if (t < best.us * 0.97) best = Plan{z, t};
    if (wg > 4 * cus) break;
  }
  return best;
}

template <bool B_COL, int NS>
static int start(const Args& g, int z, hipStream_t stream, const char* what) {
  constexpr size_t lds = (size_t)NS * 2 * OPB;
  static_assert(lds >= (size_t)T * RS, "the output tile is staged in the ring");
  auto kern = mid_kernel<B_COL, NS>;
  static uint64_t done = 0;
  if (int rc = reserve_lds((const void*)kern, lds, done, what)) return rc;
  hipLaunchKernelGGL(kern, dim3((unsigned)(g.tiles_i * g.tiles_j), 1, (unsigned)z), dim3(NT), lds,
                     stream, g);
  return check_launch(what);
}

int launch(Args g, bool b_col, int z, int64_t cus, void* ws, hipStream_t stream,
           const char* what) {
  g.tiles_i = (int)((g.I + T - 1) / T);
  g.tiles_j = (int)((g.J + T - 1) / T);
  g.splits = z;
  g.r_split = z > 1 ? g2::split_len(g.R, z) : g.R;
  g.part = reinterpret_cast<float*>(ws);
  const int64_t lim = (int64_t)1 << 32;  // copies address each operand through a 32-bit offset
  if (g.I * g.lda * 2 >= lim || (b_col ? g.R : g.J) * g.ldb * 2 >= lim) {
    set_error("%s: an operand spans 4 GiB or more", what);
    return PLZ_EUNSUPPORTED;
  }
  int rc;
  if ((int64_t)g.tiles_i * g.tiles_j * z <= cus)
    rc = b_col ? start<true, 4>(g, z, stream, what) : start<false, 4>(g, z, stream, what);
  else
    rc = b_col ? start<true, 2>(g, z, stream, what) : start<false, 2>(g, z, stream, what);
  if (rc != PLZ_OK) return rc;
  if (z == 1) return PLZ_OK;
  const int64_t n = g.I * (g.J / 8);
  hipLaunchKernelGGL(reduce_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, g);
  return check_launch(what);
}

}  // namespace mid
}  // namespace plz
