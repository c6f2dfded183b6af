// Dense MFMA GEMM on 128x128 tiles for launches of few output tiles (plz_mid.hip).
#pragma once
#include "plz_common.h"

namespace plz {
namespace mid {

// C[I, J] = sum_r A(i, r) B(j, r) (+ A2 B2) (+ bias) (+ res), bf16 in and out, fp32 sums.
struct Args {
  const uint16_t* a; int64_t lda;  // [I, R] rows
  const uint16_t* b; int64_t ldb;  // [J, R] rows, or with b_col [R, J] (J contiguous)
  int64_t I, J, R;
  // rank-R2 second segment (R2 <= 64): a2 [I, R2]; b2 [J, R2], or with b_col [R2, J]
  const uint16_t* a2; const uint16_t* b2; int R2;
  uint16_t* c; int64_t ldc; const uint16_t* bias;
  const uint16_t* res; int64_t ldres;  // added to the rounded bf16 values and rounded again
  // set by launch
  float* part; int splits; int64_t r_split; int tiles_i, tiles_j;
};

// The reduction splits this core runs the shape with, and the time its model gives them (us).
struct Plan {
  int z;
  double us;
};
Plan plan(int64_t I, int64_t J, int64_t R, int64_t cus);
size_t workspace(int64_t I, int64_t J, int z);
// z from plan(); the workspace holds workspace(I, J, z) bytes (none for z = 1).
int launch(Args g, bool b_col, int z, int64_t cus, void* ws, hipStream_t stream, const char* what);

}  // namespace mid
}  // namespace plz
