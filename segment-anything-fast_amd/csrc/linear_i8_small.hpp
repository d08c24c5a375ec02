// A quantised Linear over few rows in one launch (linear_i8_small.hip).
#pragma once

#include "gemm_i8_shared.hpp"
#include <type_traits>

namespace samfast {

// whether the form covers the shape (and is the faster one there)
bool linear_i8_small_covers(int64_t M, int N, int K);
// shapes and alignment have been checked; `layout` is the layout of wq
int linear_i8_small_launch(const unsigned short* x, int64_t ldx, const int8_t* wq, const float* sw, const float* bias, unsigned short* y,
                           int64_t ldy, int M, int N, int K, int layout, hipStream_t stream);

// The product with scale + bias epilogue for few rows (the codes come from a quantiser launch).
bool gemm_i8_skinny_covers(const GemmArgs& a);
int gemm_i8_skinny_launch(const GemmArgs& a, hipStream_t stream);

}  // namespace samfast
