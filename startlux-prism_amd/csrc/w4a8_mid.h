// The W4A8 kernels for batches between the decode kernels and projections that fill the chip with 128 x 128 tiles
// (w4a8_mid.hip); any M from 1.
#pragma once

#include "common.h"

namespace prism {

// Whether the offsets inside a workgroup's operands fit 32 bits.
inline bool w4_mid_fits(int64_t M, int64_t K) { return M <= 4096 && K <= (1 << 23); }

// Whether the mid kernel takes the shape by default (it fits, and is faster than the tile kernel).
bool w4_mid_faster(bool q6k, int64_t M, int64_t N, int64_t K);

// Q4_K (xs given) or Q6_K (xs null) weights.
void w4_mid_launch(const int8_t* xq, const float* a, int64_t a_sb, const int8_t* xs, const uint8_t* qv,
                   const uint8_t* meta, void* out, int64_t ldo, const int32_t* n_rows, int M, int N, int K, int epi,
                   hipStream_t st);

}  // namespace prism
