// Measurement aid: what the gfx950 matrix pipe sustains with no data movement at all.
//
// Every wavefront runs `iters` rounds of eight independent MFMAs (eight accumulator sets, so no
// instruction waits for another's result) on operands that sit in registers for the whole kernel:
// no global loads, no LDS, no barriers.  The operands are read once from a caller-filled buffer,
// four different (A, B) pairs per lane that rotate over the accumulator sets, so the caller decides
// what the multipliers see: zeros / small constants, or random data like a real GEMM's.  The
// rate of this loop is the ceiling any kernel built from the same instruction can approach on
// the same data; on this part it depends on the data (the power limit lowers the clock when the
// operands toggle), which is why the buffer is an argument.
//
// The accumulators are folded into one word that is stored only if it equals a fixed pattern -
// a condition on the data that the compiler cannot decide, so the arithmetic stays, and that in
// practice never holds, so the kernel writes nothing.
#include "samfast_internal.hpp"
#include "samfast_bench.h"

namespace samfast {

constexpr int kCeilSets = 8;   // independent accumulator sets per wavefront
constexpr int kCeilPairs = 4;  // distinct (A, B) operand pairs per lane

// The instructions, by the number the entry point takes: result type, its words, operations of one instruction.
template <int> struct CeilInstr;
template <> struct CeilInstr<0> {
  typedef i32x16 acc_t;
  static constexpr int WORDS = 16, OPS = 2 * 32 * 32 * 32;
  static SF_DEVICE acc_t mma(u32x4 a, u32x4 b, acc_t c) {
    return __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_bit_cast(i32x4, a), __builtin_bit_cast(i32x4, b), c, 0, 0, 0);
  }
};
template <> struct CeilInstr<1> {
  typedef f32x16 acc_t;
  static constexpr int WORDS = 16, OPS = 2 * 32 * 32 * 16;
  static SF_DEVICE acc_t mma(u32x4 a, u32x4 b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
};
template <> struct CeilInstr<2> {
  typedef i32x4 acc_t;
  static constexpr int WORDS = 4, OPS = 2 * 16 * 16 * 64;
  static SF_DEVICE acc_t mma(u32x4 a, u32x4 b, acc_t c) {
    return __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(i32x4, a), __builtin_bit_cast(i32x4, b), c, 0, 0, 0);
  }
};
template <> struct CeilInstr<3> {
  typedef f32x4 acc_t;
  static constexpr int WORDS = 4, OPS = 2 * 16 * 16 * 32;
  static SF_DEVICE acc_t mma(u32x4 a, u32x4 b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
};

// operands: (kCeilPairs, 2, 256) 16-byte vectors, indexed [pair][a|b][thread of the workgroup]
template <int I>
__global__ __launch_bounds__(256, 2) void mfma_ceiling_kernel(const u32x4* __restrict__ operands,
                                                               int iters, int* out) {
  using L = CeilInstr<I>;
  const int tid = threadIdx.x;
  u32x4 av[kCeilPairs], bv[kCeilPairs];
#pragma unroll
  for (int p = 0; p < kCeilPairs; ++p) {
    av[p] = operands[(2 * p) * 256 + tid];
    bv[p] = operands[(2 * p + 1) * 256 + tid];
  }
  int check = 0;
  typename L::acc_t acc[kCeilSets];
#pragma unroll
  for (int j = 0; j < kCeilSets; ++j) acc[j] = typename L::acc_t{};
  for (int it = 0; it < iters; ++it) {
#pragma unroll
    for (int j = 0; j < kCeilSets; ++j) acc[j] = L::mma(av[j % kCeilPairs], bv[(j + j / kCeilPairs) % kCeilPairs], acc[j]);
  }
#pragma unroll
  for (int j = 0; j < kCeilSets; ++j)
#pragma unroll
    for (int r = 0; r < L::WORDS; ++r) {
      const auto v = acc[j][r];
      check ^= __builtin_bit_cast(int, v);
    }
  if (check == 0x5a17c0de) out[tid] = check;
}

// Second question: how much vector work runs in the shadow of another wavefront's MFMAs on the same
// SIMD?  512-thread workgroups, one per CU: wavefronts 0-3 run `mfma_rounds` rounds of eight
// independent v_mfma_f32_32x32x16_bf16, wavefronts 4-7 - their SIMD partners - run `vector_rounds`
// rounds of 64 independent vector instructions (v_fma_f32, or v_exp_f32 followed by a v_mul_f32
// that keeps the value in range).  Either count may be 0; timing the kernel with one side, the
// other side and both gives the overlap.
template <bool EXP>
__global__ __launch_bounds__(512, 1) void mfma_valu_overlap_kernel(const u32x4* __restrict__ operands,
                                                                   int mfma_rounds, int vector_rounds, int* out) {
  const int tid = threadIdx.x;
  int check = 0;
  if ((tid >> 6) < 4) {  // uniform per wavefront
    if (mfma_rounds <= 0) return;
    const bf16x8 a = __builtin_bit_cast(bf16x8, operands[tid]);
    const bf16x8 b = __builtin_bit_cast(bf16x8, operands[256 + tid]);
    f32x16 acc[kCeilSets];
#pragma unroll
    for (int j = 0; j < kCeilSets; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[j][r] = 0.f;
    for (int it = 0; it < mfma_rounds; ++it) {
#pragma unroll
      for (int j = 0; j < kCeilSets; ++j) acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc[j], 0, 0, 0);
    }
#pragma unroll
    for (int j = 0; j < kCeilSets; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) check ^= __float_as_int(acc[j][r]);
  } else {
    if (vector_rounds <= 0) return;
    const u32x4 o = operands[tid & 255];
    float x[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) x[i] = __uint_as_float((o[i & 3] & 0x007fffffu) | 0x3f000000u) + 0.01f * i;  // [0.5, 1.2)
    const float c0 = __uint_as_float((o[0] & 0x007fffffu) | 0x3a000000u), c1 = 0.999f;  // data the compiler cannot fold
    for (int it = 0; it < vector_rounds; ++it) {
#pragma unroll
      for (int rep = 0; rep < (EXP ? 2 : 4); ++rep)
#pragma unroll
        for (int i = 0; i < 16; ++i)
          x[i] = EXP ? __builtin_amdgcn_exp2f(x[i]) * 0.5f : fmaf(x[i], c1, c0);
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) check ^= __float_as_int(x[i]);
  }
  if (check == 0x5a17c0de) out[tid] = check;
}

}  // namespace samfast

extern "C" int samfast_bench_mfma_valu_overlap(int vector_kind, const void* operands, int workgroups,
                                               int mfma_rounds, int vector_rounds, void* scratch_out, void* stream) {
  using namespace samfast;
  SF_REQUIRE(vector_kind == 0 || vector_kind == 1, "bench_mfma_valu_overlap: vector_kind must be 0 (fma) or 1 (exp + mul)");
  SF_REQUIRE(operands && scratch_out && aligned16(operands), "bench_mfma_valu_overlap: null or unaligned buffer");
  SF_REQUIRE(workgroups > 0 && workgroups <= (1 << 20) && mfma_rounds >= 0 && mfma_rounds <= (1 << 24) &&
                 vector_rounds >= 0 && vector_rounds <= (1 << 24),
             "bench_mfma_valu_overlap: bad workgroup or round count");
  // a launch stays below about a second of GPU time
  SF_REQUIRE((int64_t)workgroups * ((int64_t)mfma_rounds + vector_rounds) <= (1ll << 27),
             "bench_mfma_valu_overlap: workgroups * rounds must not exceed 2^27");
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const u32x4* ops = reinterpret_cast<const u32x4*>(operands);
  if (vector_kind == 0)
    hipLaunchKernelGGL((mfma_valu_overlap_kernel<false>), dim3(workgroups), dim3(512), 0, s, ops, mfma_rounds,
                       vector_rounds, (int*)scratch_out);
  else
    hipLaunchKernelGGL((mfma_valu_overlap_kernel<true>), dim3(workgroups), dim3(512), 0, s, ops, mfma_rounds,
                       vector_rounds, (int*)scratch_out);
  return check_launch("mfma_valu_overlap_kernel");
}

extern "C" int samfast_bench_mfma_ceiling(int instruction, const void* operands, int workgroups,
                                          int iters, int64_t* host_ops_out, void* scratch_out, void* stream) {
  using namespace samfast;
  SF_REQUIRE(instruction >= 0 && instruction <= 3, "bench_mfma_ceiling: instruction must be 0 or 2 (int8), 1 or 3 (bf16)");
  SF_REQUIRE(operands && scratch_out && aligned16(operands), "bench_mfma_ceiling: null or unaligned buffer");
  SF_REQUIRE(workgroups > 0 && workgroups <= (1 << 20) && iters > 0 && iters <= (1 << 24),
             "bench_mfma_ceiling: bad workgroup or iteration count");
  // a launch stays below about a second of GPU time
  SF_REQUIRE((int64_t)workgroups * iters <= (1ll << 27), "bench_mfma_ceiling: workgroups * iters must not exceed 2^27");
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const u32x4* ops = reinterpret_cast<const u32x4*>(operands);
  int instruction_ops = 0;
#define SF_CEIL(I)                                                                                             \
  case I:                                                                                                      \
    hipLaunchKernelGGL((mfma_ceiling_kernel<I>), dim3(workgroups), dim3(256), 0, s, ops, iters, (int*)scratch_out); \
    instruction_ops = CeilInstr<I>::OPS;                                                                       \
    break
  switch (instruction) {
    SF_CEIL(0);
    SF_CEIL(1);
    SF_CEIL(2);
    SF_CEIL(3);
  }
#undef SF_CEIL
  // arithmetic operations the launch executes
  if (host_ops_out) *host_ops_out = (int64_t)workgroups * 4 * iters * kCeilSets * instruction_ops;
  return check_launch("mfma_ceiling_kernel");
}
