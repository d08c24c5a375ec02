/*
 * samfast_bench - measurement and tuning aids exported by libsamfast.so beside the path's C ABI
 * (include/samfast.h).  Nothing here has a counterpart in the reference and nothing here is needed
 * to run the path: bench.py and the tests use these entry points to time bare matrix-instruction
 * loops and to switch kernel variants inside one process.
 */
#ifndef SAMFAST_BENCH_H
#define SAMFAST_BENCH_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/*
 * Kernel variants are chosen by knobs, each named like the environment variable that gives its
 * initial value (read once per process): SAMFAST_GEMM_TM, SAMFAST_GEMM_WG3, SAMFAST_GEMM_TILE,
 * SAMFAST_GEMM_PERSIST, SAMFAST_GEMM_PERSIST_SKEW, SAMFAST_GEMM_PERSIST_PRIO,
 * SAMFAST_GEMM_PINGPONG, SAMFAST_GEMM_HALF, SAMFAST_GEMM_SPLITK, SAMFAST_GEMM_ONCE, SAMFAST_GEMM_STRIP, SAMFAST_GEMM_LINEAR_SMALL, SAMFAST_GEMM_LINEAR_BAND, SAMFAST_GEMM_SKINNY,
 * SAMFAST_ATTN_WAVES, SAMFAST_ATTN_SPLIT, SAMFAST_ATTN_WINDOW_ROWS, SAMFAST_SPARSE_PERSIST, SAMFAST_SPARSE_TURNS.  This
 * call sets one (`unset` != 0: back to "not given", `value` ignored).  The knobs move time; every
 * variant of a kernel returns the same bits, with three exceptions that sum in another order:
 * SAMFAST_ATTN_SPLIT, SAMFAST_ATTN_WINDOW_ROWS and SAMFAST_GEMM_HALF (the framework's products, tiles that sum K in one
 * order, tiles that sum its halves apart).  The first two defaults do not look at the number of slices: a slice's
 * attention does not depend on its batch.  A half-type product's kernel does follow its rows (samfast_linear_half_pays).
 * Returns SAMFAST_E_INVALID for an unknown name.
 */
int samfast_bench_set_knob(const char* name, int value, int unset);

/*
 * Columns of the tile (192, 256 or 320) in which samfast_gemm_i8_fused or samfast_gemm_i8_sparse24_fused forms this output by
 * turns, 0 where the rule leaves it to other kernels: no launch, for rows of the output and the residual
 * `row_stride` elements apart that start on a cache line.  SAMFAST_E_INVALID for a bad shape.
 */
int samfast_bench_gemm_i8_turns(int64_t M, int N, int K, int epilogue, int64_t row_stride);
int samfast_bench_sparse24_turns(int64_t M, int N, int K, int epilogue, int64_t row_stride);

/*
 * 1000 times the rows plus the columns of the tile in which samfast_gemm_i8_fused without a step behind it forms an output of few rows
 * with K dealt over a workgroup's wavefronts, 0 where the rule leaves it to other kernels: no launch.  SAMFAST_E_INVALID for a bad shape.
 */
int samfast_bench_gemm_i8_few_rows(int64_t M, int N, int K, int x_layout, int w_layout);

/*
 * The same of a Linear (samfast_linear_i8, or samfast_linear_i8_sparse24 for `layout` SAMFAST_LAYOUT_SPARSE24) whose workgroups quantise
 * a few rows themselves: 1000 times those rows plus the columns of one, 0 for other forms.
 */
int samfast_bench_linear_i8_few_rows(int64_t M, int N, int K, int layout);

/* 1000 times the rows plus the columns of the tile of samfast_linear_half, 0 where samfast_linear_half_pays says no. */
int samfast_bench_linear_half(int64_t M, int N, int K, int epilogue);

/*
 * Measurement aid, no counterpart in the reference: one launch of a kernel that does nothing
 * but matrix instructions on operands held in registers (no global loads, no LDS, no barriers)
 * - the rate a GEMM or attention kernel built from the same instruction can approach at best
 * on the same kind of data.  instruction 0 = v_mfma_i32_32x32x32_i8, 1 =
 * v_mfma_f32_32x32x16_bf16, 2 = v_mfma_i32_16x16x64_i8, 3 = v_mfma_f32_16x16x32_bf16.  `operands` holds 4 (A, B) pairs of 16 bytes for each of 256 lanes
 * (8 * 256 * 16 bytes, [pair][A|B][lane]); their values decide what the multipliers toggle.
 * `workgroups` of 256 threads run `iters` rounds of 8 independent instructions per wavefront
 * (workgroups * iters <= 2^27, about a second of GPU time; more returns SAMFAST_E_INVALID);
 * *host_ops_out (may be NULL) receives the arithmetic operations of the launch.  `scratch_out`
 * (>= 1 KiB) receives nothing in practice (see the kernel).  Timing is the caller's (events on `stream`).
 */
int samfast_bench_mfma_ceiling(
    int instruction, const void* operands, int workgroups, int iters,
    int64_t* host_ops_out, void* scratch_out, void* stream);

/*
 * Measurement aid, no counterpart in the reference: how much vector work runs in the shadow of
 * another wavefront's matrix instructions on the same SIMD.  Workgroups of 512 threads, one per
 * CU: wavefronts 0-3 run `mfma_rounds` rounds of eight independent v_mfma_f32_32x32x16_bf16 on
 * operands held in registers, wavefronts 4-7 (their SIMD partners) `vector_rounds` rounds of 64
 * independent vector instructions - vector_kind 0: v_fma_f32, 1: v_exp_f32 + v_mul_f32.  Either
 * count may be 0, which times one side alone; workgroups * (mfma_rounds + vector_rounds) <= 2^27.  `operands`: at least 8 KiB (two 16-byte vectors for
 * each of 256 lanes); `scratch_out`: 2 KiB the kernel may write.  bench.py --mfma-ceiling uses it.
 */
int samfast_bench_mfma_valu_overlap(
    int vector_kind, const void* operands, int workgroups, int mfma_rounds, int vector_rounds,
    void* scratch_out, void* stream);

#ifdef __cplusplus
}
#endif
#endif /* SAMFAST_BENCH_H */
