// PQ2_0 products of many tokens on the block-scaled matrix cores (pq2_mx.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

namespace bh {

// Y[n_tok][n_rows] = X[n_tok][ne0] * W^T: ne0 a multiple of 256, w 4-byte and
// x 16-byte aligned.  Uses the matmul scratch.
int pq2_mx_gemm(const uint8_t *w, size_t ne0, size_t n_rows, const float *x, size_t n_tok, float *y,
                hipStream_t st);

}  // namespace bh
