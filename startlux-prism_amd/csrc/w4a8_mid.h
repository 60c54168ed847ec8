// The W4A8 kernels for 17 and more activation rows on projections too narrow to fill the chip with 128 x 128 tiles
// (w4a8_mid.hip).
#pragma once

#include "common.h"

namespace prism {

// Whether the mid kernel takes the shape by default (its offsets fit, and it is faster than the tile kernel).
bool w4_mid_faster(bool q6k, int64_t M, int64_t N, int64_t K);

// Q4_K (xs given) or Q6_K (xs null) weights.
void w4_mid_launch(const int8_t* xq, const float* a, int64_t a_sb, const int8_t* xs, const uint8_t* qv,
                   const uint8_t* meta, void* out, int64_t ldo, const int32_t* n_rows, int M, int N, int K, int epi,
                   hipStream_t st);

}  // namespace prism
