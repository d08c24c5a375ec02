// bf16 / fp16 Linears of an encoder block: the turn-taking kernels of gemm_pingpong.hpp with the block's own epilogues, so that GELU and
// the residual add cost no pass over memory of their own.
#include "gemm_pingpong.hpp"
#include "samfast_bench.h"

namespace samfast {

// The kernel for a product: columns / 32 of a tile; 6, 8 and 10 the resident kernel (kHalfTall: with 320 rows and 256 columns), 3 to 5 the
// split one, 0 none (the library's product and a pass of its own for GELU or residual are ahead).  The lines, by the rounds of the
// CUs and the share of their time that makes output (us, library with its pass / here, residuals with the LayerNorm behind them):
//   GELU: from half of the CUs on.  4096 x 768 -> 3072 34.2 / 27.6, 4096 x 1280 -> 5120 77.1 / 50.1, 20480 x 1024 -> 4096 188 / 152,
//     65536 x 1280 -> 5120 856 / 729.
//   plain: from 0.7 on, on loops shorter than 1024 up to 8 rounds.  4096 x 1024 -> 3072 28.5 / 26.6, 8192 x 768 -> 2304 38.8 / 30.8, 20480 x 1024 -> 3072
//     106 / 99.5, 32768 x 768 -> 2304 120 / 101, 57344 x 1024 -> 3072 (11 rounds) 299 / 280, 49152 x 1280 -> 3840 (12) 370 / 361; but 4096 x 768 -> 2304
//     (0.56) 20.1 / 21.0, 65536 x 768 -> 2304 (9 rounds) 196 / 213.
//   residual: 128-row tiles where the CUs hold them all at once.  4096 x 1280 -> 1280 28.6 / 24.9, 4096 x 5120 -> 1280 61 / 53.
//     Else 320 x 256 where that fills its rounds from 0.8 on: 20480 x 4096 -> 1024 (1.0) 164 / 137, 20480 x 1024 -> 1024 74.3 / 52.7, 24576 x 3072
//     -> 768 (0.9) 146 / 102, 40960 x 5120 -> 1280 (three rounds, 0.83) 545 / 450, 57344 x 5120 -> 1280 (four, 0.88) 700 / 622, 57344 x
//     1280 -> 1280 (four, 0.88) 255 / 233.
//     Else 256 x 256, on long loops within one round from 0.7 on (12288 x 5120 -> 1280 140 / 126; 0.62: 8192 x 5120 -> 1280 alone 104 / 104, an
//     encoder of two images 4 % slower; two rounds: 32768 x 4096 -> 1024 231 / 238), on short ones up to four rounds from 0.55 on (0.56: 12288
//     x 768 -> 768 39.8 / 30.5, 0.62: 8192 x 1280 -> 1280 45.2 / 40.2, 16384 x 1280 -> 1280 88.3 / 75.4, 0.75: 12288 x 1024 -> 1024 42.4 / 38.3; 0.5: 8192 x 1024 -> 1024
//     32.2 / 33.6, five rounds: 65536 x 1280 -> 1280 276 / 278).
// The rows decide, so the order in which a product's terms are summed, and with it the last bits of an image's embedding in the half
// types, follows the batch, as it does with the library's kernels (one ViT-H image: 3-5 split K, five ViT-L images: 320-row tiles, the
// library in between; 0.016 and 2e-4 of the embedding's norm).  int8 sums are integers: an image comes out the same in any batch.
constexpr int kHalfTall = 58;  // 320 rows, 256 columns
constexpr int kHalfNarrow = 192;  // the knob's number for 192 columns
static int half_choose(int64_t M, int N, int K, int epi) {
  const int force = knob_or(KNOB_GEMM_HALF, 1);
  if (force <= 0 || K % 64 != 0 || K < 320 || M < 256 || N < 96) return 0;
  if (force == kHalfNarrow) return epi != PP_RESIDUAL && N >= 192 ? 6 : 0;
  if (force == kHalfTall) return epi == PP_RESIDUAL && N >= 256 && M >= 320 ? force : 0;
  if (force >= 3) {
    const bool built = (force <= 5 || force == 8 || (force == 10 && epi != PP_RESIDUAL)) && N >= 32 * force;
    return built ? force : 0;
  }
  if (epi == PP_RESIDUAL)
    for (int tn = 3; tn <= 5; ++tn) {
      const int64_t tiles = ((M + 127) / 128) * ((N + 32 * tn - 1) / (32 * tn));
      if (tiles <= 256 && tiles >= 128 && N >= 32 * tn) return tn;
    }
  const PPChoice c = pp_choose(M, N, K / 64, epi == PP_RESIDUAL);
  if (c.tn == 0) return 0;
  bool pays = c.used >= 0.5;
  if (epi == PP_PLAIN) pays = c.used >= 0.7 && (c.rounds <= 8 || K >= 1024);
  if (epi == PP_RESIDUAL) pays = c.tm == 5 ? c.used >= 0.8 : K >= 2048 ? c.rounds == 1 && c.used >= 0.7 : c.rounds <= 4 && c.used >= 0.55;
  if (!pays) return 0;
  if (c.tm == 5) return kHalfTall;
  // (192 columns are no reason to leave the library's product, whose order of K is another: all of these sum in the same one)
  return epi == PP_RESIDUAL ? c.tn : pp_choose(M, N, K / 64, false, epi == PP_GELU ? 8.4 : 8.1).tn;
}

template <class E>
static int half_launch(PPArgs a, int tn, int epi, hipStream_t stream) {
  a.group_m = 4;
  if (tn == kHalfTall) {
    a.tiles_m = (a.M + 319) / 320;
    a.tiles_n = (a.N + 255) / 256;
    hipLaunchKernelGGL((gemm_pingpong_kernel<E, PP_RESIDUAL, 8, false, 5>), dim3(pp_grid(a)), dim3(512), 0, stream, a);
    return check_launch("gemm_pingpong_kernel");
  }
  a.tiles_n = (a.N + 32 * tn - 1) / (32 * tn);
  if (tn >= 6) {
    a.tiles_m = (a.M + 255) / 256;
    const dim3 grid(pp_grid(a));
#define SF_PP(EPI, TN) hipLaunchKernelGGL((gemm_pingpong_kernel<E, EPI, TN, false>), grid, dim3(512), 0, stream, a)
    if (epi == PP_GELU) { if (tn == 6) SF_PP(PP_GELU, 6); else if (tn == 8) SF_PP(PP_GELU, 8); else SF_PP(PP_GELU, 10); }
    else if (epi == PP_RESIDUAL) SF_PP(PP_RESIDUAL, 8);
    else { if (tn == 6) SF_PP(PP_PLAIN, 6); else if (tn == 8) SF_PP(PP_PLAIN, 8); else SF_PP(PP_PLAIN, 10); }
#undef SF_PP
    return check_launch("gemm_pingpong_kernel");
  }
  a.tiles_m = (a.M + 127) / 128;
  const dim3 grid((unsigned int)(((int64_t)a.tiles_m * a.tiles_n + 7) / 8 * 8));
#define SF_PP(EPI, TN) hipLaunchKernelGGL((gemm_pingpong_split_kernel<E, EPI, TN>), grid, dim3(512), 0, stream, a)
#define SF_PP_ALL(TN) do { if (epi == PP_RESIDUAL) SF_PP(PP_RESIDUAL, TN); else if (epi == PP_GELU) SF_PP(PP_GELU, TN); else SF_PP(PP_PLAIN, TN); } while (0)
  if (tn == 3) SF_PP_ALL(3);
  else if (tn == 4) SF_PP_ALL(4);
  else SF_PP_ALL(5);
#undef SF_PP_ALL
#undef SF_PP
  return check_launch("gemm_pingpong_split_kernel");
}

}  // namespace samfast

extern "C" int samfast_linear_half_pays(int64_t M, int N, int K, int epilogue) {
  using namespace samfast;
  const int epi = epilogue == SAMFAST_EPILOGUE_GELU ? PP_GELU : epilogue == SAMFAST_EPILOGUE_RESIDUAL ? PP_RESIDUAL : PP_PLAIN;
  return N > 0 && N % 8 == 0 && half_choose(M, N, K, epi) != 0;
}

extern "C" int samfast_bench_linear_half(int64_t M, int N, int K, int epilogue) {
  using namespace samfast;
  SF_REQUIRE(M > 0 && N > 0 && K > 0 && N % 8 == 0, "bench_linear_half: bad shape M=%lld N=%d K=%d", (long long)M, N, K);
  const int tn = half_choose(M, N, K, epilogue == SAMFAST_EPILOGUE_GELU ? PP_GELU : epilogue == SAMFAST_EPILOGUE_RESIDUAL ? PP_RESIDUAL : PP_PLAIN);
  return tn == 0 ? 0 : tn == kHalfTall ? 320256 : (tn < 6 ? 128000 : 256000) + 32 * tn;
}

extern "C" int samfast_linear_half(const void* x, int64_t ldx, const void* w, const void* bias, void* y, int64_t ldy,
                                   int64_t M, int N, int K, int dtype, int epilogue, const void* residual, int64_t ld_res, void* stream) {
  using namespace samfast;
  if (dtype != SAMFAST_BF16 && dtype != SAMFAST_F16) SF_FAIL(SAMFAST_E_UNSUPPORTED, "linear_half: element type %d is neither SAMFAST_BF16 nor SAMFAST_F16", dtype);
  int epi;
  switch (epilogue) {
    case SAMFAST_EPILOGUE_NONE: epi = PP_PLAIN; break;
    case SAMFAST_EPILOGUE_GELU: epi = PP_GELU; break;
    case SAMFAST_EPILOGUE_RESIDUAL: epi = PP_RESIDUAL; break;
    default: SF_FAIL(SAMFAST_E_INVALID, "linear_half: unknown epilogue %d", epilogue);
  }
  SF_REQUIRE(M >= 0 && N > 0 && K > 0 && N % 8 == 0, "linear_half: bad shape M=%lld N=%d K=%d (N must be a multiple of 8)", (long long)M, N, K);
  if (M == 0) return SAMFAST_OK;
  SF_REQUIRE(x && w && y && (epi != PP_RESIDUAL || residual), "linear_half: null pointer");
  SF_REQUIRE(aligned16(x) && aligned16(w) && aligned16(y) && aligned16(residual) && (reinterpret_cast<uintptr_t>(bias) & 3u) == 0,
             "linear_half: operands must be 16-byte aligned, the bias 4-byte");
  SF_REQUIRE(ldx >= K && ldx % 8 == 0 && ldy >= N && ldy % 8 == 0 && (epi != PP_RESIDUAL || (ld_res >= N && ld_res % 8 == 0)),
             "linear_half: row strides must be multiples of 8 and hold a row");
  SF_REQUIRE(M < (1ll << 31) - 512 && ldx < (1ll << 22) && K < (1 << 22), "linear_half: too large");
  const int tn = half_choose(M, N, K, epi);
  PPArgs a = {};
  a.x = reinterpret_cast<const unsigned char*>(x);
  a.w = reinterpret_cast<const unsigned char*>(w);
  a.out = reinterpret_cast<unsigned short*>(y);
  a.bias = bias;
  a.residual = reinterpret_cast<const unsigned short*>(residual);
  a.ldo = ldy;
  a.ld_res = epi == PP_RESIDUAL ? ld_res : 0;
  a.x_kstep = a.w_kstep = 64;
  a.x_pitch = (unsigned int)(ldx * 2);
  a.w_pitch = (unsigned int)(K * 2);
  a.M = (int)M;
  a.N = N;
  a.nk = K / 64;
  if (tn == 0 || !pp_addressable(a))
    SF_FAIL(SAMFAST_E_UNSUPPORTED, "linear_half: no kernel for M=%lld N=%d K=%d (samfast_linear_half_pays)", (long long)M, N, K);
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  return dtype == SAMFAST_F16 ? half_launch<PPF16>(a, tn, epi, s) : half_launch<PPBf16>(a, tn, epi, s);
}
