// Per-row symmetric int8 quantiser (bf16 -> int8 + fp32 scale), optionally preceded
// by LayerNorm over the row and a row gather (window partition).  HBM-bound: 65536 rows of 5120 through GELU 216 us, of 1280
// plain 46, with LayerNorm 54, codes written into new memory each time (4.7, 5.5 and 4.6 TB/s; a copy reaches 4.9 from HBM); rows that lie in the
// caches by the vector ALU as well: 144 vector instructions per row of 1280 plain, 338 with LayerNorm, 1374 per row of 5120 with GELU, by the hardware
// counters, for a wavefront per row (with LayerNorm 291 where wavefronts walk the rows of 65536).  us with the quotient made exact in three steps / codes from one product (quant_row.hpp): 4096 x 1024 3.52 / 3.30, with LayerNorm
// 4.63 / 4.36, 4096 x 4096 9.9 / 9.7, with GELU 14.6 / 13.8, 5003 x 5120 with GELU 20.1 / 18.9, 20480 x 1024 with LayerNorm 15.2 / 14.2, 65536 x 5120 with GELU 212 / 213,
// 65536 x 1280 with LayerNorm 53.4 / 53.6.
//
// One wavefront owns one output row: the source row is read once with 16- or 8-byte loads
// and unpacked to fp32 registers, (normalised,) reduced to its absmax across the 64 lanes
// (DPP within rows of 16 lanes, lane swaps between them: no LDS), then scaled, rounded
// half-to-even and written back as 8- or 4-byte packs of int8.
// Algorithmic traffic: 2 bytes read + 1 byte written per element + 4 bytes of scale.
//
// q = rint(x / s) must equal the IEEE division bit for bit (quant_row.hpp).
// |x| <= absmax makes |x / s| <= 127 by construction, so no clamp is needed.
#include "quant_row.hpp"

namespace samfast {

constexpr int kQuantWavesPerBlock = 4;

// workgroups for M rows, a multiple of 8
__host__ SF_DEVICE unsigned int quant_blocks(int64_t M, int rpb) { return ((unsigned int)((M + rpb - 1) / rpb) + 7u) & ~7u; }

// Which RPB rows workgroup b takes, of quant_blocks(M, RPB): every XCD (workgroup modulo 8) a contiguous eighth, and that from its end.
// The products on either side walk such eighths from their starts: what one of them has written last, and the last-level cache still holds, is read
// first here, and what is written last here is read first by the next one.  us in the ViT-H encoder, 16 images, row by row / so: rows with LayerNorm 53.2 / 51.9, proj
// and lin2 behind them 232.8 / 227.4 on average, rows with GELU, whose producer streams past the cache, 176 / 179; of
// the present rows the whole 57620 / 57410 and 57760 / 57370, 32 images with 2:4 MLPs 108610 / 107490 and 108530 / 107390, ViT-L in bf16, whose rows are not these, level; single images level.
// A Linear's own rows, without LayerNorm or GELU, are taken as they come by one wavefront (65536 x 1280 -> 3840 306.6 so, 309.4 from the ends) and by two through the cache (32768 x 2048
// -> 2048 148 / 151); the other shared rows from the ends (65536 x 4096 -> 1024 378 / 338, 16384 x 5120 -> 1280 126.3 / 121.0, 65536 x 2560 -> 1280 268 / 260, 20480 x 3072 -> 768 72 / 69.8).
SF_DEVICE unsigned int row_block(unsigned int b, int64_t M, int rpb) {
  const unsigned int eighth = quant_blocks(M, rpb) >> 3;
  return (b & 7u) * eighth + eighth - 1u - (b >> 3);
}

// GELU of values that lie in bf16, back in bf16, as the GEMM's epilogue makes it
template <int NCH, typename in_t>
SF_DEVICE void gelu_chunks(in_t (&xw)[NCH]) {
#pragma unroll
  for (int i = 0; i < NCH; ++i)
#pragma unroll
    for (int j = 0; j < (int)(sizeof(in_t) / 4); ++j) xw[i][j] = pack_bf16x2(gelu_erf(bf16_lo_to_f32(xw[i][j])), gelu_erf(bf16_hi_to_f32(xw[i][j])));
}

// ACT: the values are GELU's of what lies in memory.  Between an MLP's two Linears the activation runs here rather than in
// the first one's epilogue: this kernel waits for memory and the vector ALU is free (65536 x 5120: 175 us without, 215 with it),
// while a GEMM's wavefronts multiply nothing in the meantime (65536 x 1280 -> 5120: 465 us with GELU, 375 without).
// EXACT: the row fills every lane's chunks (nothing is tested per chunk, and the loads' addresses are one and constants).
template <int NCH, int EPC, bool LN, bool ACT, bool EXACT>
__global__ __launch_bounds__(64 * kQuantWavesPerBlock) void quant_rowwise_bf16_kernel(QuantArgs a) {
  using RQ = RowQuantizer<NCH, EPC, LN>;
  const int lane = threadIdx.x & 63;
  // the wavefront index is uniform: telling the compiler so keeps the row and everything derived from it
  // (row pointers, output offsets) in scalar registers instead of 64-bit arithmetic per lane
  const unsigned int block = LN || ACT ? row_block(blockIdx.x, a.M, kQuantWavesPerBlock) : blockIdx.x;
  const int64_t row = (int64_t)block * kQuantWavesPerBlock + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (row >= a.M) return;  // whole wavefront leaves together
  const int nchunk = EXACT ? 64 * NCH : a.K / EPC;

  int64_t srow = row;
  if (LN && a.src_row) {
    srow = a.src_row[row];
    if (srow < 0) {  // a padding token: LayerNorm output replaced by zeros
      RQ::zero_row(a, row, nchunk, lane);
      return;
    }
  }
  // all global loads first: the row, and (LN) the lane's slices of gamma and beta, which do not
  // depend on the statistics and would otherwise add a second memory latency to the chain
  typename RQ::in_t xw[NCH], gw[NCH], bw[NCH];
  // long rows (the 671 MB lin1 output at ViT-H batch 16) are read once and never again: streamed
  RQ::template load_row<(!LN && NCH >= 8)>(a.x + srow * a.ldx, nchunk, lane, xw);
  if (LN) RQ::load_affine(a.gamma, a.beta, nchunk, lane, gw, bw);
  if (ACT) gelu_chunks(xw);
  RQ::finish_row(a, row, nchunk, lane, xw, gw, bw);
}

// Many rows with LayerNorm: the wavefronts stay and walk the rows, gamma and beta unpacked once, the next row's loads under the
// present one's arithmetic: five workgroups per CU, what 84 registers a lane admit.  Bound: memory and the vector ALU level.  us, a wavefront per row / so
// (8 workgroups per CU): 65536 x 1280 62.7 / 54.2 (55.4), 131072 x 1280 128 / 118 (115), 32768 x 1280 32.9 / 29.2, 16384 x 1280 15.7 / 15.3, 65536 x 768 37.1 / 34.8, 65536 x 1024
// 43.3 / 42.2, 20480 x 1024 15.6 / 15.6; fewer values than that are no faster (16384 x 768 11.8 / 12.1, 8192 x 1024 7.9 / 8.0).
template <int NCH, int EPC>
__global__ __launch_bounds__(64 * kQuantWavesPerBlock) void layernorm_quant_rows_kernel(QuantArgs a) {
  using RQ = RowQuantizer<NCH, EPC, true>;
  const int lane = threadIdx.x & 63;
  constexpr int NCHUNK = 64 * NCH;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // (gridDim.x is a multiple of 8; a row behind the last one is none)
  const unsigned int blocks = quant_blocks(a.M, kQuantWavesPerBlock);
  unsigned int b = blockIdx.x;
  auto row_of = [&](unsigned int block) { return (int64_t)row_block(block, a.M, kQuantWavesPerBlock) * kQuantWavesPerBlock + wave; };
  int64_t row = row_of(b);
  typename RQ::in_t xw[NCH], next[NCH], gw[NCH], bw[NCH];
  const int64_t last = a.M - 1;
  RQ::template load_row<false>(a.x + min(row, last) * a.ldx, NCHUNK, lane, xw);
  RQ::load_affine(a.gamma, a.beta, NCHUNK, lane, gw, bw);
  const typename RQ::PlainAffine affine(gw, bw);
  while (b < blocks) {
    b += gridDim.x;
    const int64_t ahead = row_of(min(b, blocks - 1u));
    RQ::template load_row<false>(a.x + min(ahead, last) * a.ldx, NCHUNK, lane, next);
    if (row < a.M) RQ::finish_row(a, row, NCHUNK, lane, xw, affine);
    row = ahead;
#pragma unroll
    for (int i = 0; i < NCH; ++i) xw[i] = next[i];
  }
}

// WPR wavefronts share a row: fewer registers per lane for long rows (one wavefront with 4096 values needs 238: two
// per SIMD and 2.2 TB/s at 65536 rows, 5.1 TB/s with four sharing), and for few rows more wavefronts with
// fewer loads each to wait for.  The shares' maxima meet in LDS.  Bound: memory, at the rate of a copy, from 8192 rows on.
// NTL: rows larger than the cache, read past it.
template <int NCH, int EPC, int WPR, bool ACT, bool NTL>
__global__ __launch_bounds__(64 * kQuantWavesPerBlock) void quant_rowshare_bf16_kernel(QuantArgs a) {
  constexpr int RPB = kQuantWavesPerBlock / WPR;  // rows per workgroup
  using RQ = RowQuantizer<NCH, EPC, false>;
  typedef typename RQ::in_t in_t;
  __shared__ float part[kQuantWavesPerBlock];
  __shared__ int nan_seen[kQuantWavesPerBlock];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int sub = wave % WPR;
  const unsigned int block = ACT || NTL || WPR == 4 ? row_block(blockIdx.x, a.M, RPB) : blockIdx.x;
  const int64_t row = (int64_t)block * RPB + wave / WPR;
  const bool live = row < a.M;  // uniform over the wavefront
  const int nchunk = a.K / EPC;
  // chunk i of the lane: (i * WPR + sub) * 64 + lane, so that the wavefronts of a row read it side by side
  in_t xw[NCH];
  float amax;
#pragma unroll
  for (int i = 0; i < NCH; ++i) {
    const int c = (i * WPR + sub) * 64 + lane;
    const in_t z = {};
    xw[i] = z;
    if (live && c < nchunk) {
      const in_t* src = reinterpret_cast<const in_t*>(a.x + row * a.ldx) + c;
      xw[i] = NTL ? __builtin_nontemporal_load(src) : *src;
    }
  }
  if (ACT) gelu_chunks(xw);
  float f[NCH][EPC];
#pragma unroll
  for (int i = 0; i < NCH; ++i)
#pragma unroll
    for (int e = 0; e < RQ::W; ++e) {
      f[i][2 * e] = bf16_lo_to_f32(xw[i][e]);
      f[i][2 * e + 1] = bf16_hi_to_f32(xw[i][e]);
    }
  const bool own_nan = wave_absmax(f, amax);
  if (lane == 0) {
    part[wave] = amax;
    nan_seen[wave] = own_nan;
  }
  __syncthreads();
  int any_nan = 0;
#pragma unroll
  for (int w = 0; w < WPR; ++w) {
    amax = fmaxf(amax, part[wave / WPR * WPR + w]);
    any_nan |= nan_seen[wave / WPR * WPR + w];
  }
  const QuantScale q(amax);
#pragma unroll
  for (int i = 0; i < NCH; ++i)
    if (live && (i * WPR + sub) * 64 + lane < nchunk) {
      unsigned int codes[EPC / 4];
      quantize_chunk<EPC>(f[i], q, codes);
      RQ::store_chunk(a, row, i * WPR + sub, lane, codes);
    }
  if (live && sub == 0 && lane == 0) a.sx[row] = any_nan ? __uint_as_float(0x7fc00000u) : q.scale;
}

template <int NCH, int EPC, int WPR, bool ACT, bool NTL>
static int launch_rowshare(const QuantArgs& a, hipStream_t stream) {
  constexpr int RPB = kQuantWavesPerBlock / WPR;
  hipLaunchKernelGGL((quant_rowshare_bf16_kernel<NCH, EPC, WPR, ACT, NTL>), dim3(quant_blocks(a.M, RPB)), dim3(64 * kQuantWavesPerBlock), 0, stream, a);
  return check_launch("quant_rowshare_bf16_kernel");
}

template <int NCH, int EPC, bool LN, bool ACT>
static int launch_quant(const QuantArgs& a, hipStream_t stream) {
  const dim3 grid(quant_blocks(a.M, kQuantWavesPerBlock)), block(64 * kQuantWavesPerBlock);
  // (the widths of the encoders' rows: built for those)
  constexpr bool MAY_FIT = EPC == 4 || NCH == 2 || NCH == 10;
  if constexpr (LN && (EPC == 4 || NCH == 2)) {
    if (a.K == 64 * EPC * NCH && !a.src_row && a.M * a.K >= (20ll << 20)) {
      hipLaunchKernelGGL((layernorm_quant_rows_kernel<NCH, EPC>), dim3(min(grid.x, 256u * 5u)), block, 0, stream, a);
      return check_launch("layernorm_quant_rows_kernel");
    }
  }
  if (MAY_FIT && a.K == 64 * EPC * NCH) hipLaunchKernelGGL((quant_rowwise_bf16_kernel<NCH, EPC, LN, ACT, MAY_FIT>), grid, block, 0, stream, a);
  else hipLaunchKernelGGL((quant_rowwise_bf16_kernel<NCH, EPC, LN, ACT, false>), grid, block, 0, stream, a);
  return check_launch("quant_rowwise_bf16_kernel");
}

template <int WPR, bool ACT, bool NTL>
static int launch_shares(const QuantArgs& a, hipStream_t s) {
  // shares that 4-element chunks divide among the 64 lanes exactly and 8-element chunks do not
  if (a.K == 3 * 256 * WPR) return launch_rowshare<3, 4, WPR, ACT, NTL>(a, s);
  if (a.K == 5 * 256 * WPR) return launch_rowshare<5, 4, WPR, ACT, NTL>(a, s);
  const int need = (a.K / 8 + 64 * WPR - 1) / (64 * WPR);
  if (need <= 1) return launch_rowshare<1, 8, WPR, ACT, NTL>(a, s);
  if (need <= 2) return launch_rowshare<2, 8, WPR, ACT, NTL>(a, s);
  if (WPR == 2 || need <= 3) return launch_rowshare<3, 8, WPR, ACT, NTL>(a, s);
  return launch_rowshare<4, 8, WPR, ACT, NTL>(a, s);
}

template <bool LN, bool ACT>
static int dispatch_quant(const QuantArgs& a, hipStream_t s) {
  // rows that 4-element chunks divide among the 64 lanes exactly and 8-element chunks do not
  if (a.K == 768) return launch_quant<3, 4, LN, ACT>(a, s);
  if (a.K == 1280) return launch_quant<5, 4, LN, ACT>(a, s);
  const int need = (a.K / 8 + 63) / 64;
  if constexpr (!LN) {
    // Rows of more than 1024.  Where the rows and their codes fit the 256 MB last-level cache together (a producer has just put
    // them there), they are read as such and shared: by two wavefronts up to 2560 values, by four above and for few rows, in which the
    // wavefronts, not their loads, are scarce.  us, streamed and by the rules below / so: 4096 x 3072 10.8 / 9.5, 20480 x 3072 37.5 / 31.4, 4096 x 5120 15.6 /
    // 13.1, 5003 x 5120 17.3 / 15.4, 8192 x 5120 27.9 / 21.9, 16384 x 5120 46.6 / 40.2, 20480 x 4096 47.5 / 40.0, 12288 x 1536 14.7 / 12.2, 32768 x
    // 2048 42.3 / 32.8, 8192 x 8192 44.0 / 37.5 (168 MB of rows: the last that gain; inside an
    // encoder, where lin1 has just written them, neither way is ahead); beyond, 20480 x 5120 56.2 / 68.7, 65536 x 5120 198 / 248.
    // (Three loads of a wavefront, the third less than three quarters full, are as well alone from 8192 rows on: 12000 x 1152 12.6 / 13.0.)
    if (need >= 3 && a.M * a.K * 3 <= (256ll << 20) && (a.K >= 1408 || a.M <= 8192))
      return need >= 6 || a.M <= 1024 ? launch_shares<4, ACT, false>(a, s) : launch_shares<2, ACT, false>(a, s);
    // Larger ones are streamed past the cache, and shared where one wavefront would need 128 registers and more (us, one wavefront a
    // row / two / four: 65536 x 4096: 308 / 166 / 159, 65536 x 2560: 115 / 102 / 105).
    if (need == 4 || need == 5) return launch_shares<2, ACT, true>(a, s);
    if (need >= 6 && need <= 8) return launch_shares<4, ACT, true>(a, s);
    // K > 4096: quarters that fill their lanes (K % 1024 == 0), while their stores spread.  K-block major codes of M % 16 == 0 rows have
    // their K blocks a multiple of 1 KB apart, and the four stores meet.  From 11 chunks per lane on one wavefront is short of
    // registers: 16384 x 8192 82 / 77.5; not at more rows: 32768 x 5120 87 / 105 (one / four).
    const bool spread = !a.kb64 || a.M % 16 != 0;
    if (need > 8 && a.M <= 16384 && (need > 12 || (a.K % 1024 == 0 && spread))) return launch_shares<4, ACT, true>(a, s);
  } else {
    if (need == 4) return launch_quant<4, 8, LN, ACT>(a, s);
    if (need > 4 && need <= 6) return launch_quant<6, 8, LN, ACT>(a, s);
    if (need > 6 && need <= 8) return launch_quant<8, 8, LN, ACT>(a, s);
  }
  if (need <= 2) return launch_quant<2, 8, LN, ACT>(a, s);
  if (need <= 3) return launch_quant<3, 8, LN, ACT>(a, s);
  if (need <= 10) return launch_quant<10, 8, LN, ACT>(a, s);
  if (need <= 12) return launch_quant<12, 8, LN, ACT>(a, s);
  return launch_quant<16, 8, LN, ACT>(a, s);
}

static int check_common(const char* who, const void* x, int64_t ldx, const int8_t* xq, const float* sx,
                        int64_t M, int K, int dtype, int layout) {
  SF_REQUIRE(layout == SAMFAST_LAYOUT_ROWMAJOR || (layout == SAMFAST_LAYOUT_KB64 && K % 64 == 0),
             "%s: layout must be row-major, or K-block major with K %% 64 == 0", who);
  SF_REQUIRE(M >= 0 && K > 0, "%s: bad shape M=%lld K=%d", who, (long long)M, K);
  SF_REQUIRE(M == 0 || (x && xq && sx), "%s: null pointer", who);  // no rows: the buffers may be null
  if (dtype != SAMFAST_BF16) SF_FAIL(SAMFAST_E_UNSUPPORTED, "%s: only bf16 input", who);
  SF_REQUIRE(K % 8 == 0 && K <= 8192, "%s: K=%d must be a multiple of 8, <= 8192", who, K);
  SF_REQUIRE(ldx >= K && ldx % 8 == 0, "%s: ldx=%lld must be >= K and a multiple of 8", who,
             (long long)ldx);
  SF_REQUIRE(aligned16(x) && (reinterpret_cast<uintptr_t>(xq) & 7u) == 0,
             "%s: x must be 16-byte and xq 8-byte aligned", who);
  SF_REQUIRE((M + 3) / 4 < (1ll << 31), "%s: M too large", who);
  SF_REQUIRE(M * (int64_t)K < (1ll << 31), "%s: outputs of 2 GiB or more are not supported (the GEMM cannot read them)", who);
  return SAMFAST_OK;
}

}  // namespace samfast

namespace samfast {

template <bool ACT>
static int quant_rowwise(const char* who, const void* x, int64_t ldx, int8_t* xq, float* sx, int64_t M, int K, int dtype, int layout, void* stream) {
  const int rc = check_common(who, x, ldx, xq, sx, M, K, dtype, layout);
  if (rc != SAMFAST_OK) return rc;
  if (M == 0) return SAMFAST_OK;
  QuantArgs a = {};
  a.x = reinterpret_cast<const unsigned short*>(x);
  a.ldx = ldx; a.xq = xq; a.sx = sx; a.M = M; a.K = K;
  a.kb64 = layout == SAMFAST_LAYOUT_KB64;
  return dispatch_quant<false, ACT>(a, reinterpret_cast<hipStream_t>(stream));
}

}  // namespace samfast

extern "C" int samfast_quant_rowwise_i8(const void* x, int64_t ldx, int8_t* xq, float* sx,
                                        int64_t M, int K, int dtype, int layout, void* stream) {
  return samfast::quant_rowwise<false>("quant_rowwise", x, ldx, xq, sx, M, K, dtype, layout, stream);
}

extern "C" int samfast_gelu_quant_rowwise_i8(const void* x, int64_t ldx, int8_t* xq, float* sx,
                                             int64_t M, int K, int dtype, int layout, void* stream) {
  return samfast::quant_rowwise<true>("gelu_quant_rowwise", x, ldx, xq, sx, M, K, dtype, layout, stream);
}

extern "C" int samfast_layernorm_quant_i8(const void* x, int64_t ldx, const void* gamma,
                                          const void* beta, float eps, const int32_t* src_row,
                                          int8_t* xq, float* sx, int64_t M, int K, int dtype,
                                          int layout, void* stream) {
  using namespace samfast;
  const int rc = check_common("layernorm_quant", x, ldx, xq, sx, M, K, dtype, layout);
  if (rc != SAMFAST_OK) return rc;
  SF_REQUIRE(gamma && beta && aligned16(gamma) && aligned16(beta),
             "layernorm_quant: gamma / beta must be non-null and 16-byte aligned");
  SF_REQUIRE(eps > 0.f, "layernorm_quant: eps must be positive");
  if (M == 0) return SAMFAST_OK;
  QuantArgs a = {};
  a.x = reinterpret_cast<const unsigned short*>(x);
  a.ldx = ldx; a.xq = xq; a.sx = sx; a.M = M; a.K = K;
  a.gamma = reinterpret_cast<const unsigned short*>(gamma);
  a.beta = reinterpret_cast<const unsigned short*>(beta);
  a.src_row = src_row; a.eps = eps; a.inv_K = 1.0f / (float)K;
  a.kb64 = layout == SAMFAST_LAYOUT_KB64;
  return dispatch_quant<true, false>(a, reinterpret_cast<hipStream_t>(stream));
}
