// A quantised Linear over few rows in one launch (linear_i8_small.hip).
#pragma once

#include "gemm_i8_shared.hpp"
#include <type_traits>

namespace samfast {

// whether the form covers the shape (and is the faster one there)
bool linear_i8_small_covers(int64_t M, int N, int K, bool sparse);
// whether dense calls of this size are taken with scales and bias of any alignment (at every N; the products want 16 bytes)
bool linear_i8_small_any_alignment(int64_t M, int K);
// shapes and alignment have been checked; `layout` is the layout of dense weights (widx null)
int linear_i8_small_launch(const unsigned short* x, int64_t ldx, const int8_t* w, const int32_t* widx, const float* sw, const float* bias,
                           unsigned short* y, int64_t ldy, int M, int N, int K, int layout, hipStream_t stream);

// The same over more rows, a band of them and a range of columns per workgroup (linear_i8_band.hip).
bool linear_i8_band_covers(int64_t M, int N, int K, bool sparse);
int linear_i8_band_launch(const unsigned short* x, int64_t ldx, const int8_t* w, const int32_t* widx, const float* sw, const float* bias, unsigned short* y,
                          int64_t ldy, int M, int N, int K, int layout, hipStream_t stream);

// The product with scale + bias epilogue for few rows (the codes come from a quantiser launch).
bool gemm_i8_skinny_covers(const GemmArgs& a);
int gemm_i8_skinny_launch(const GemmArgs& a, hipStream_t stream);

}  // namespace samfast
