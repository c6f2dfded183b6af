// Hard LUT-linear forward of few rows (plz_skinny.hip).
#pragma once
#include "plz_common.h"

namespace plz {
namespace sk {

constexpr int64_t kMaxRows = 64;

// The operands have passed plz_lut_linear_fwd's checks; 1 <= M <= kMaxRows, N, K > 0.
int fwd(const uint16_t* x, const int32_t* packed, const float* palette, const uint16_t* bias,
        const uint16_t* lora_t, const uint16_t* lora_b, int rank, uint16_t* y, int64_t M,
        int64_t N, int64_t K, int64_t cus, hipStream_t stream, const char* what);

}  // namespace sk
}  // namespace plz
