// Pieces of the reference-layout soft linear shared by plz_soft_ref.hip and the GEMM core.
#pragma once
#include "plz_common.h"

namespace plz {
namespace g2 {

// fp32 partials [z][I][J] of C[i][j] = sum_r a[r][i] b[r][j] (a [R, I], b [R, J] bf16) over z
// splits of R, by the dW GEMM (plz_gemm2.hip); I, J, R > 0, I and J multiples of 8.
int dw_splits(int64_t I, int64_t J, int64_t R);
int dw_partials(const uint16_t* a, const uint16_t* b, float* out, int z, int64_t I, int64_t J,
                int64_t R, hipStream_t stream, const char* what);

}  // namespace g2
}  // namespace plz
