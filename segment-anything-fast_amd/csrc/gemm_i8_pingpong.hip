// int8 GEMM for outputs of whole rounds of wide tiles: the turn-taking kernel of gemm_pingpong.hpp.
#include "gemm_pingpong.hpp"
#include "samfast_bench.h"

namespace samfast {

static PPArgs pp_args(const GemmArgs& g) {
  PPArgs a = {};
  a.x = reinterpret_cast<const unsigned char*>(g.x);
  a.w = reinterpret_cast<const unsigned char*>(g.w);
  a.out = reinterpret_cast<unsigned short*>(g.out);
  a.sx = g.sx;
  a.sw = g.sw;
  a.bias = g.bias;
  a.residual = g.residual;
  a.ldo = g.ldo;
  a.ld_res = g.residual ? g.ld_res : 0;
  a.x_kstep = g.x_kstep;
  a.w_kstep = g.w_kstep;
  a.x_pitch = (unsigned int)g.x_pitch;
  a.w_pitch = (unsigned int)g.w_pitch;
  a.M = g.M;
  a.N = g.N;
  a.nk = g.K / 128;
  return a;
}

// SAMFAST_GEMM_PINGPONG = 1 chooses among all tiles, 6 takes 192 columns wherever they fit, other numbers the wider ones.  With the residual short loops have nothing from 192 columns
// (12288 x 768 -> 768 15.5 / 15.9, 28672 x 768 -> 768 28.6 / 28.8), and below 4096 values two rounds of them are ahead alone (28672 x 3072 -> 768 72.1 / 65.2) but not in an
// encoder (seven images of ViT-B 7.08 / 7.11 ms; one round, three images 3.40 / 3.38; K = 5120, four of ViT-H 16.99 / 16.66).
constexpr double kNarrowPlain = 8.7;
static PPChoice choose(int epi, int64_t M, int N, int K) {
  const int mode = knob_or(KNOB_GEMM_PINGPONG, 1);
  const bool residual = K >= 4096 || (K >= 2048 && (M + 255) / 256 * ((N + 191) / 192) <= 256);
  return pp_choose(M, N, K / 128, epi == EPI_RESIDUAL_BF16, mode == 6 ? 0.1 : mode != 1 ? 0.0 : epi != EPI_RESIDUAL_BF16 ? kNarrowPlain : residual ? 9.0 : 0.0);
}

static bool whole_lines(const void* p, int64_t ld) { return reinterpret_cast<uintptr_t>(p) % 128 == 0 && ld % 64 == 0; }

// lines: rows of the output and the residual are whole cache lines (residual products)
static bool pays(int epi, int K, const PPChoice& c, bool lines) {
  // The lines, by the share of the CUs' time that makes output (us, the other members / this one, K-block major, random codes):
  //   plain, K >= 1280, 0.75: 0.78 (5000 rows -> 5120) 43.1 / 38.1, 0.94 (4096 -> 3840) 26.9 / 21.0, 1.0 (65536 -> 3840) 309 / 263,
  //     K = 5120, 1.0 (65536 -> 3840) 1126 / 994; but 0.59 (5000 -> 3840) 30.0 / 37.6
  //   shorter loops, 0.8: 0.84 (12288 x 768 -> 2304) 31.0 / 26.5, 0.9 (8192 x 768 -> 2304) 23.4 / 20.4, 0.84 in four rounds (24576 x 768 -> 2304) 52.3 /
  //     50.1, 1.0 (4096 x 1024 -> 4096) 23.1 / 20.1; but 0.75 (8192 x 768 -> 3072 in 256 columns) 25.7 / 25.8, (4096 x 768 -> 2304 in 192) 15.8 / 16.2.  Tiles of 192
  //     columns fill rounds that the wider ones leave out: 90 products drawn where they are taken are 0.68 to 0.99 times as long, one of them 1.015 (26317 x 896 -> 1280):
  //     8192 x 768 -> 3072 25.0 / 22.7, 8192 x 1024 -> 3072 29.6 / 26.6, 2820 x 3584 -> 3840 42.4 / 35.4, 11268 x 3456 -> 2080 96.7 / 65.9, 32355 x 3072 -> 768 72.9 / 60.9
  //   plain, one round of 192 columns, K above 768, 0.68: 0.75 (4096 x 1152 -> 2304) 18.6 / 15.8, (12288 x 1024 -> 768) 17.6 / 15.1, 0.69 (2437 x 1024 -> 3584) 16.3 / 14.6, (2200 x 5120 ->
  //     3904) 53.7 / 40.5, row-major 0.68 (2400 x 2432 -> 3552) 35.8 / 23.0, 85 products drawn between 0.68 and 0.8, K 896 to 5120, 0.62 to 1.005 times as long; but 0.67, where
  //     512 tiles of 128 x 128 are two per CU, (8192 x 1024 -> 1024) 15.0 / 15.3, 0.66 (4604 x 1152 -> 1792) 14.6 / 15.2.  From K = 2048 on 0.5: 0.51 (6262 x 4096 -> 1024) 33.9 / 31.9, 0.55 (8270 x 5120 -> 832) 43.6 / 39.8, 0.66 (3313 x
  //     5120 -> 2488) 54.0 / 40.5, row-major 0.58 (1702 x 4096 -> 4280) 45.6 / 32.8, 32 drawn 0.63 to 0.95 times as long; but 0.55 (4025 x 1280 -> 1728) 15.1 / 15.5.  K of 640 and
  //     768 keep 0.8 (0.94 to 1.0 in most there; 4096 x 768 -> 2304 14.5 / 12.9 in later measurements than the one above)
  //   residual, K >= 2048, 0.7, within one round of 256 columns 0.55: 0.56 (12288 x 3072 -> 768) 38.6 / 36.6, 0.62 (8192 x 5120 -> 1280) 59.5 / 54.6, 0.75 (12288 x 4096 ->
  //     1024) 54.1 / 49.8, (192 columns) 0.83 (16384 x 5120 -> 1280) 108 / 96, 0.75 (12288 x 3072 ->
  //     768) 36.5 / 32.6, but 0.66 (10771 x 3200 -> 768) 31.7 / 32.4, 1.0 (20480 x 4096 -> 1024, 320 rows) 86.5 / 64.3, (65536 x 5120 -> 1280) 402 / 336, 0.88 (28672 x 5120 -> 1280, 320 rows) 190 /
  //     149; but 0.5 (8192 x 4096 -> 1024) 40.6 / 45.5, 0.66 in two rounds (28672 x 3072 -> 768) 70.4 / 71.1
  //   residual, shorter loops, 0.85: 0.94 (20480 x 768 -> 768) 22.4 / 19.8, two rounds (40960 x 768 -> 768) 41.3 / 34.4, 0.88 (28672 x 1024 -> 1024) 43.9 / 38.5, 1.0
  //     (20480 x 1024 -> 1024, 320 rows) 31.9 / 28.4, 0.88 in five rounds (57344 x 1280 -> 1280) 124.2 / 117.2; but 0.75 (24576 x 1024 -> 1024) 35.7 / 37.5, 0.83
  //     (32768 x 1280 -> 1280) 63.2 / 66.3; from K = 1280 on 0.77 in up to two rounds: 0.78 (20480 -> 1280) 48.5 / 41.5
  //     Rows that are no whole lines, whose segments each touch two, only within two rounds: 7556 x 1024 -> 1992 31.4 / 28.3, 16384 x 640 -> 1992 47.4 / 44.6; but
  //     four 28672 x 640 -> 1992 72.4 / 78.1, five 14563 x 640 -> 4904 102 / 114, thirteen 40960 x 1024 -> 4904 309 / 321 (28672 x 1280 -> 1992 110 / 101)
  if (epi != EPI_RESIDUAL_BF16) return c.used >= (c.rounds == 1 && c.tn == 6 && K > 768 ? (K >= 2048 ? 0.5 : 0.68) : K >= 1280 ? 0.75 : 0.8);
  if (K >= 2048) return c.used >= (c.rounds == 1 && c.tn != 6 ? 0.55 : 0.7);
  if (K < 1280 && c.rounds > 2 && !lines) return false;
  return c.used >= (K >= 1280 && c.rounds <= 2 ? 0.77 : 0.85);
}

bool gemm_i8_pingpong_reads_rows(int64_t M, int N, int K) {
  if (K % 128 != 0 || K < 640) return false;  // (no knob: a workspace sized by this answer must fit the call that follows)
  const PPChoice c = pp_choose(M, N, K / 128, false, kNarrowPlain);  // choose's without a knob
  return c.tn != 0 && pays(EPI_SCALE_BIAS_BF16, K, c, true);
}

bool gemm_i8_pingpong_covers(int epi, const GemmArgs& g) {
  const int mode = knob_or(KNOB_GEMM_PINGPONG, 1);
  if (mode <= 0 || (epi != EPI_SCALE_BIAS_BF16 && epi != EPI_RESIDUAL_BF16) || g.dst_row || g.tile_counters) return false;
  if (g.K % 128 != 0 || !pp_addressable(pp_args(g))) return false;
  const PPChoice c = choose(epi, g.M, g.N, g.K);
  if (c.tn == 0) return false;
  if (mode >= 2) return true;
  return pays(epi, g.K, c, whole_lines(g.out, g.ldo) && whole_lines(g.residual, g.ld_res));
}

int gemm_i8_pingpong_launch(int epi, const GemmArgs& g, hipStream_t stream) {
  PPArgs a = pp_args(g);
  const PPChoice c = choose(epi, g.M, g.N, g.K);
  const int tn = c.tn;
  a.group_m = 4;
  a.tiles_m = (a.M + 64 * c.tm - 1) / (64 * c.tm);
  a.tiles_n = (a.N + 32 * tn - 1) / (32 * tn);
  // an output larger than the last-level cache that is read once (qkv, lin1) is streamed out; not where rows are no whole cache lines,
  // whose two halves two stores bring (streamed / not, us: 31790 x 640 -> 4904 186 / 128, 55833 x 768 -> 4904 318 / 279, 40000 x 1280 -> 5096 299 / 280)
  const bool nt = g.stream_out != 0 && whole_lines(g.out, g.ldo);
#define SF_PP(E, TN, NT) hipLaunchKernelGGL((gemm_pingpong_kernel<PPInt8, E, TN, NT>), dim3(pp_grid(a)), dim3(512), 0, stream, a)
#define SF_PP_PLAIN(TN) do { if (nt) SF_PP(PP_PLAIN, TN, true); else SF_PP(PP_PLAIN, TN, false); } while (0)
  if (epi == EPI_RESIDUAL_BF16 && c.tm == 5)
    hipLaunchKernelGGL((gemm_pingpong_kernel<PPInt8, PP_RESIDUAL, 8, false, 5>), dim3(pp_grid(a)), dim3(512), 0, stream, a);
  else if (epi == EPI_RESIDUAL_BF16 && tn == 6) SF_PP(PP_RESIDUAL, 6, false);
  else if (epi == EPI_RESIDUAL_BF16) SF_PP(PP_RESIDUAL, 8, false);
  else if (tn == 6) SF_PP_PLAIN(6);
  else if (tn == 8) SF_PP_PLAIN(8);
  else SF_PP_PLAIN(10);
#undef SF_PP_PLAIN
#undef SF_PP
  return check_launch("gemm_pingpong_kernel");
}

}  // namespace samfast

extern "C" int samfast_bench_gemm_i8_turns(int64_t M, int N, int K, int epilogue, int64_t row_stride) {
  using namespace samfast;
  SF_REQUIRE(M > 0 && M < (1ll << 31) - 256 && N > 0 && K > 0 && row_stride >= N, "bench_gemm_i8_turns: bad shape M=%lld N=%d K=%d", (long long)M, N, K);
  GemmArgs g = {};
  g.M = (int)M; g.N = N; g.K = K; g.ldo = g.ld_res = row_stride;
  const int epi = epilogue == SAMFAST_EPILOGUE_NONE ? EPI_SCALE_BIAS_BF16 : epilogue == SAMFAST_EPILOGUE_RESIDUAL ? EPI_RESIDUAL_BF16 : EPI_GELU_BF16;
  return gemm_i8_pingpong_covers(epi, g) ? 32 * choose(epi, M, N, K).tn : 0;
}
