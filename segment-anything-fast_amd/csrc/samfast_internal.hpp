// Shared device/host helpers of the samfast HIP kernels (gfx950 only).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "samfast.h"

namespace samfast {

// ---- error reporting (host) -------------------------------------------------
void set_error(const char* fmt, ...);
#define SF_FAIL(code, ...)              \
  do {                                  \
    ::samfast::set_error(__VA_ARGS__);  \
    return (code);                      \
  } while (0)
#define SF_REQUIRE(cond, ...)                              \
  do {                                                     \
    if (!(cond)) SF_FAIL(SAMFAST_E_INVALID, __VA_ARGS__);  \
  } while (0)

int check_launch(const char* what);

// Tuning knobs: each is an environment variable read ONCE (at the first query of any knob), after
// which samfast_bench_set_knob (include/samfast_bench.h) is the only way to change it.
enum Knob {
  KNOB_GEMM_TM,           // SAMFAST_GEMM_TM: 4 = 256 x 256 tiles in the two-per-CU kernel
  KNOB_GEMM_WG3,          // SAMFAST_GEMM_WG3: 0 = two workgroups per CU instead of three
  KNOB_GEMM_TILE,         // SAMFAST_GEMM_TILE: 64 / 96 / 128 forces 64 x 128 / 128 x 128 / 128 x 256 tiles in the three-per-CU kernel
  KNOB_GEMM_PERSIST,      // SAMFAST_GEMM_PERSIST: 0 off, 1 where it pays, 2 wherever it is built
  KNOB_GEMM_PERSIST_SKEW, // SAMFAST_GEMM_PERSIST_SKEW: start delay of every second resident workgroup, 64 cycles per k tile
  KNOB_GEMM_PERSIST_PRIO, // SAMFAST_GEMM_PERSIST_PRIO: 0 = no wave priority changes in the persistent kernel
  KNOB_GEMM_PINGPONG,     // SAMFAST_GEMM_PINGPONG: 256-row tiles by turns (gemm_pingpong.hpp), 0 off, 1 where it pays, 2 wherever built
  KNOB_GEMM_HALF,         // SAMFAST_GEMM_HALF: the half types' products, 0 the library's, 1 ours where they pay; 3, 4, 5 (K halves summed apart), 8, 10: columns / 32 of the tile, 58: 320 x 256, 192: 256 x 192; others: the library's
  KNOB_GEMM_SPLITK,       // SAMFAST_GEMM_SPLITK: 0 off, 1 where it pays (launches that leave the GPU half empty; 2:4: one tile per CU), 2 wherever built
  KNOB_GEMM_ONCE,         // SAMFAST_GEMM_ONCE: 0 = off, 1 where it pays, rows * 16 + columns / 32 = that tile of the one-tile-per-CU kernel
  KNOB_GEMM_STRIP,        // SAMFAST_GEMM_STRIP: 0 = off, 1 where it pays, 2 = wherever built (gemm_i8_strip.hip)
  KNOB_LINEAR_SMALL,      // SAMFAST_GEMM_LINEAR_SMALL: 0 = whole Linears (2:4 ones too) as two launches throughout: over few rows and over a band of rows
  KNOB_LINEAR_BAND,       // SAMFAST_GEMM_LINEAR_BAND: whole Linears over a band of rows in one launch, 0 off, 1 where it pays, row tiles * 8 + column tiles (of 16) of a wavefront: that tile, and no Linear by the few-row form
  KNOB_GEMM_SKINNY,       // SAMFAST_GEMM_SKINNY: 0 = products over few rows through the tiled kernels
  KNOB_ATTN_WAVES,        // SAMFAST_ATTN_WAVES: 4 / 8 wavefronts per global-attention workgroup
  KNOB_ATTN_SPLIT,        // SAMFAST_ATTN_SPLIT: global attention with the keys split between two wavefronts (other bits), 0 = never, 1 = head_dim 64, 2 = always
  KNOB_ATTN_WINDOW_ROWS,  // SAMFAST_ATTN_WINDOW_ROWS: 1 = window keys as grid rows padded to 16 (attn_window_rows_kernel) where built
  KNOB_SPARSE_PERSIST,    // SAMFAST_SPARSE_PERSIST: 2:4 GEMM, 0 = one workgroup per tile (default), 1 = resident workgroups from two tiles each on, 2 wherever built
  KNOB_SPARSE_TURNS,      // SAMFAST_SPARSE_TURNS: 2:4 GEMM by turns (gemm_i8_sp24_turns.hip), 0 off, 1 where it pays, 8 / 10 wherever built, channels / 32 of the tile
  KNOB_COUNT
};
constexpr int kKnobUnset = INT32_MIN;
int knob(Knob k);                      // kKnobUnset when neither the environment nor a setter gave a value
static inline int knob_or(Knob k, int dflt) {
  const int v = knob(k);
  return v == kKnobUnset ? dflt : v;
}

static inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// ---- vector types -------------------------------------------------------------
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef int i32x16 __attribute__((ext_vector_type(16)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

#define SF_DEVICE __device__ __forceinline__

// bf16 <-> fp32 on raw bits
SF_DEVICE float bf16_lo_to_f32(unsigned int w) { return __uint_as_float(w << 16); }
SF_DEVICE float bf16_hi_to_f32(unsigned int w) { return __uint_as_float(w & 0xffff0000u); }
SF_DEVICE float bf16_bits_to_f32(unsigned short h) { return __uint_as_float(((unsigned int)h) << 16); }

// round-to-nearest-even fp32 -> bf16 bits (finite inputs; NaN kept quiet)
SF_DEVICE unsigned int f32_to_bf16_bits(float f) {
  unsigned int u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (u >> 16) | 0x40u;
  u += 0x7fffu + ((u >> 16) & 1u);
  return u >> 16;
}
// two fp32 -> packed bf16 pair, round to nearest even, one v_cvt_pk_bf16_f32
SF_DEVICE unsigned int pack_bf16x2(float lo, float hi) {
  const f32x2 v = {lo, hi};
  return __builtin_bit_cast(unsigned int, __builtin_convertvector(v, bf16x2));
}

SF_DEVICE float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// value held by lane (lane ^ 32) of the same wavefront
SF_DEVICE float xor32(float v) { return __shfl_xor(v, 32, 64); }

// GELU(x) = x * Phi(x), written so that the negative side keeps its relative accuracy:
//   gelu(x) = max(x, 0) - |x| * h,   h = Phi(-|x|) = 2^P(|x|),
// P = degree-7 least-squares fit (Chebyshev nodes) of log2 Phi(-z) on [0, 6]: |P - log2 Phi|
// < 7e-6, i.e. h to 5e-6 relative in fp32 Horner form - a result that differs from the
// correctly rounded bf16 value in about one of a thousand cases, by one step.  Beyond |x| = 6
// h is held at Phi(-6) = 1e-9.  One transcendental and ten other instructions per value: the two
// clamps are median-of-three instructions (|x| as a source modifier), which unlike fminf / fmaxf
// need no separate instruction to quiet a signalling NaN first.
SF_DEVICE float gelu_erf(float x) {
#pragma clang fp contract(fast)  // an approximation anyway: let the polynomial use FMAs
  const float ax = fabsf(x);
  const float z = __builtin_amdgcn_fmed3f(ax, 0.0f, 6.0f);
  float p = -1.88962623e-06f;
  p = fmaf(p, z, 6.26814010e-05f);
  p = fmaf(p, z, -9.38867933e-04f);
  p = fmaf(p, z, 8.53946133e-03f);
  p = fmaf(p, z, -5.40206871e-02f);
  p = fmaf(p, z, -4.58409777e-01f);
  p = fmaf(p, z, -1.15126915e+00f);
  p = fmaf(p, z, -9.99994340e-01f);
  const float h = __builtin_amdgcn_exp2f(p);
  return fmaf(-ax, h, __builtin_amdgcn_fmed3f(x, 0.0f, 3.4028234664e38f));
}

// GELU(x) = x * Phi(x) for values that arrive and leave in the half types.  h = Phi(-|x|) = 2^P(|x|), so that the negative
// side keeps its relative accuracy; P is a degree-7 least-squares fit (Chebyshev nodes, reweighted towards the least
// maximum) of log2 Phi(-z) on [0, 5.5] with P(0) = -1 exactly, within 5.4e-6 there.  Odd, with a negative leading coefficient,
// it falls beyond that without a clamp, and h runs into zero as Phi does.  Of all fp16 values 45 are not rounded correctly (577
// with erf in fp32, where 1 + erf cancels), of all bf16 values 89 (340).  The infinities are x * Phi's: +inf for the positive
// one, NaN for the negative one, as x * 0.5 * (1 + erf) gives them.
SF_DEVICE float gelu_value(float x) {
  const float z = fabsf(x);
  float p = -1.73511671e-06f;
  p = fmaf(p, z, 5.9744074e-05f);
  p = fmaf(p, z, -0.000916868041f);
  p = fmaf(p, z, 0.00845726952f);
  p = fmaf(p, z, -0.0538610406f);
  p = fmaf(p, z, -0.458561927f);
  p = fmaf(p, z, -1.15120995f);
  p = fmaf(p, z, -1.f);
  const float h = fast_exp2(p);
  return x * (x > 0.f ? 1.f - h : h);
}

// Consecutive workgroup ids are dealt round-robin to the 8 XCDs, each with its
// own L2.  Map the hardware id to a logical id so that every XCD walks one
// contiguous range of logical ids (neighbours then share an L2).
SF_DEVICE unsigned int xcd_contiguous_id(unsigned int hw_id, unsigned int total) {
  const unsigned int per = (total + 7u) >> 3;
  return (hw_id & 7u) * per + (hw_id >> 3);
}

}  // namespace samfast
