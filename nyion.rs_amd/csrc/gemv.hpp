// gemv.hpp — what the two k-quant weight product sources share.
#pragma once

#include "common.hpp"

namespace nyion {

constexpr int kKqBlockElems = 256;
constexpr int kQ4kBlockBytes = 144;
constexpr int kQ6kBlockBytes = 210;
constexpr int kGemvMaxMats = 4;

// out[m][b][r] = sum_j W_m[r][j] x[b][j] for n_mats (1..kGemvMaxMats) Q4_K
// matrices of nb blocks per row that share `batch` inputs.  Arguments are
// checked by the caller.
int gemv_q4k_launch(const uint8_t* const* ws, const float* x, long long x_stride, float* const* outs,
                    long long out_stride, const int32_t* row_counts, int n_mats, int nb, int batch,
                    hipStream_t st);

}  // namespace nyion
