// The middle of an int8 block for an image or two in one launch: the attention output's row quantiser, proj, the residual add, norm2 and
// lin1's row quantiser.
//
// At 4096 rows the three launches of it (5.0, 8.7 and 5.4 us at width 768) are mostly starts, ends and latency.  Here a workgroup
// owns 16 whole rows (32 from 4097 rows on), so nothing between the quantisers leaves the CU: eight wavefronts quantise the rows into LDS,
// multiply them by all of W - each its own eighth of the columns, through a ring of 14 to 16 KB of its own in LDS that is requested before the
// rows are there - and finish whole rows again, one wavefront each, with the quantiser's own code.  What bounds it is W through
// the load path of every CU, 0.6 MB at 56 bytes a cycle: 4.7 us of the 13.6 at width 768 (fragments straight into registers, 16 bytes of each
// of 16 rows to a quarter of the lanes, came at 33 bytes a cycle: 16.3 us).  Width 1280, 1.6 MB, is no faster than the three
// launches (4096 rows 26.6 / 26.8) and not built.
//
// Codes, sums, roundings and scales are those of the separate launches: the same bits.
#include "attn_relpos_shared.hpp"
#include "gemm_i8_shared.hpp"
#include "quant_row.hpp"

#pragma clang fp contract(off)

namespace samfast {

struct ProjBlockArgs {
  const unsigned short* x;         // attention output, (M, C), row stride ldx
  const int8_t* w;                 // (C/64, C, 64)
  const float* sw;
  const float* bias;               // may be null
  const unsigned short* residual;  // (M, C) contiguous
  unsigned short* tokens;          // (M, C) contiguous; may be the residual
  int64_t ldx;
  QuantArgs q;                     // x unused; gamma, beta, eps, xq (K-block major), sx of the output
};

// at most n vector memory operations of this wavefront outstanding (n constant at every use)
SF_DEVICE void proj_wait(int n) {
  switch (n) {
#define SF_CASE(H) case H: __builtin_amdgcn_s_waitcnt(0x0F70 | (H)); break
    SF_CASE(0); SF_CASE(1); SF_CASE(2); SF_CASE(3); SF_CASE(4); SF_CASE(5); SF_CASE(6); SF_CASE(7);
    SF_CASE(8); SF_CASE(9); SF_CASE(10); SF_CASE(11); SF_CASE(12); SF_CASE(13); SF_CASE(14); SF_CASE(15);
#undef SF_CASE
  }
  __builtin_amdgcn_sched_barrier(0);
}

template <int C, int RT>
__global__ __launch_bounds__(512) void proj_block_i8_kernel(ProjBlockArgs a) {
  constexpr int EPC = quant_epc_for(C), NCH = quant_nch_for(C), NCHUNK = C / EPC;
  using In = RowQuantizer<NCH, EPC, false>;
  using Ln = RowQuantizer<NCH, EPC, true>;
  typedef typename In::in_t in_t;
  constexpr int R = 16 * RT, RPW = 2 * RT;      // rows of the workgroup, of a wavefront
  constexpr int NF = C / 128, NK = C / 64;      // column fragments of a wavefront (16 columns x 64 bytes, 1 KB), k steps
  constexpr int RING = RT == 1 ? 16 : 14;       // fragments of a wavefront in LDS
  constexpr int CP = C + 16, OP = 2 * C + 16;   // LDS row pitches: codes, Linear output
  static_assert(RING >= NF && RING - NF < 16, "wait thresholds");
  static_assert(R * OP <= 8 * RING * 1024, "the output rows take the ring's place");
  __shared__ __attribute__((aligned(16))) unsigned char lds[8 * RING * 1024 + R * CP];
  __shared__ float scales[R];
  unsigned char* rows = lds;                    // R rows of bf16, behind the products
  unsigned char* codes = lds + 8 * RING * 1024; // R rows

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lq = lane >> 4;
  const int64_t row0 = (int64_t)blockIdx.x * R;
  const int64_t last = a.q.M - 1;

  // ---- loads that wait for nothing: the rows to quantise, then everything that is needed behind the products, then W ----------------
  in_t xw[RPW][NCH], res[RPW][NCH], gw[NCH], bw[NCH];
#pragma unroll
  for (int r = 0; r < RPW; ++r) In::template load_row<false>(a.x + min(row0 + wave * RPW + r, last) * a.ldx, NCHUNK, lane, xw[r]);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int r = 0; r < RPW; ++r) Ln::template load_row<false>(a.residual + min(row0 + wave * RPW + r, last) * C, NCHUNK, lane, res[r]);
  Ln::load_affine(a.q.gamma, a.q.beta, NCHUNK, lane, gw, bw);
  f32x4 sw[NF], bias[NF];
  const float* bias_or_sw = a.bias ? a.bias : a.sw;  // (a load under a branch would make the compiler wait here)
#pragma unroll
  for (int j = 0; j < NF; ++j) {
    const int n = wave * (C / 8) + 16 * j + 4 * lq;
    sw[j] = *reinterpret_cast<const f32x4*>(a.sw + n);
    bias[j] = *reinterpret_cast<const f32x4*>(bias_or_sw + n);
  }
  __builtin_amdgcn_sched_barrier(0);
  // Through LDS, although no other wavefront reads these columns: a fragment as the instruction takes it is 16 bytes of each of 16
  // rows to a quarter of the lanes, which the load path serves at 33 bytes a cycle, in the order of memory at 56.
  const unsigned int w_lane = (unsigned int)((lane >> 2) * 64 + (((lane & 3) ^ (-(lane >> 4) & 3)) * 16));
  unsigned char* ring = lds + wave * RING * 1024;
  const unsigned int ring_at = (unsigned int)(uintptr_t)((__attribute__((address_space(3))) unsigned char*)ring);
  const unsigned char* wbase = reinterpret_cast<const unsigned char*>(a.w) + (int64_t)wave * (C / 8) * 64;
  auto load_w = [&](int f) __attribute__((always_inline)) {
    lds_dma16(wbase + (int64_t)(f / NF) * C * 64 + (f % NF) * 1024, w_lane, ring_at + f % RING * 1024);
  };
#pragma unroll
  for (int f = 0; f < RING; ++f) load_w(f);
  __builtin_amdgcn_sched_barrier(0);

  // LDS written by all is visible to all; loads stay in flight (a __syncthreads would wait for them)
  auto meet = [] __device__ () __attribute__((always_inline)) {
    __builtin_amdgcn_s_waitcnt(0xC07F);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };

  // ---- the attention output's codes into LDS --------------------------------------------------------------------------------------
#pragma unroll
  for (int r = 0; r < RPW; ++r) {
    const int row = wave * RPW + r;
    const float scale = In::finish(a.q, NCHUNK, lane, xw[r], gw, bw, [&](int i, const unsigned int (&v)[EPC / 4]) {
#pragma unroll
      for (int e = 0; e < EPC / 4; ++e) reinterpret_cast<unsigned int*>(codes + row * CP + (64 * i + lane) * EPC)[e] = v[e];
    });
    if (lane == 0) scales[row] = scale;
  }
  meet();

  // ---- products: W rows are the instruction's rows, a lane ends with four adjacent channels of token lr ------------------------------
  i32x4 acc[RT][NF];
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int j = 0; j < NF; ++j) acc[t][j] = i32x4{0, 0, 0, 0};
  const unsigned char* wfrag = ring + lr * 64 + ((lq ^ (-(lr >> 2) & 3)) * 16);
#pragma unroll
  for (int k = 0; k < NK; ++k) {
    proj_wait((k * NF + RING < NK * NF ? k * NF + RING : NK * NF) - (k + 1) * NF);
    i32x4 f[RT], w[NF];
#pragma unroll
    for (int t = 0; t < RT; ++t) f[t] = *reinterpret_cast<const i32x4*>(codes + (16 * t + lr) * CP + k * 64 + lq * 16);
#pragma unroll
    for (int j = 0; j < NF; ++j) w[j] = *reinterpret_cast<const i32x4*>(wfrag + (k * NF + j) % RING * 1024);
    __builtin_amdgcn_s_waitcnt(0xC07F);  // the fragments are in registers: their places are requested anew
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < NF; ++j)
      if (k * NF + j + RING < NK * NF) load_w(k * NF + j + RING);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < NF; ++j)
#pragma unroll
      for (int t = 0; t < RT; ++t) acc[t][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w[j], f[t], acc[t][j], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
  }
  meet();  // nobody reads the ring any more
  if (!a.bias)  // uniform
#pragma unroll
    for (int j = 0; j < NF; ++j) bias[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    const float sx = scales[16 * t + lr];
#pragma unroll
    for (int j = 0; j < NF; ++j) {
      const int n = wave * (C / 8) + 16 * j + 4 * lq;
      float y[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        // three separately rounded fp32 operations (no fused multiply-add)
        float v = (float)acc[t][j][e] * sx;
        v = v * sw[j][e];
        y[e] = v + bias[j][e];
      }
      *reinterpret_cast<u32x2*>(rows + (16 * t + lr) * OP + n * 2) = u32x2{pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3])};
    }
  }
  meet();

  // ---- whole rows again: residual add, norm2, quantiser ---------------------------------------------------------------------------
#pragma unroll
  for (int r = 0; r < RPW; ++r) {
    const int row = wave * RPW + r;
    if (row0 + row > last) continue;  // uniform over the wavefront
    in_t v[NCH];
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int c = lane + 64 * i;
      const in_t z = {};
      v[i] = z;
      if (c < NCHUNK) {
        const in_t y = *reinterpret_cast<const in_t*>(rows + row * OP + c * EPC * 2);
#pragma unroll
        for (int e = 0; e < In::W; ++e)
          v[i][e] = pack_bf16x2(bf16_lo_to_f32(y[e]) + bf16_lo_to_f32(res[r][i][e]), bf16_hi_to_f32(y[e]) + bf16_hi_to_f32(res[r][i][e]));
        reinterpret_cast<in_t*>(a.tokens + (row0 + row) * C)[c] = v[i];
      }
    }
    Ln::finish_row(a.q, row0 + row, NCHUNK, lane, v, gw, bw);
  }
}

}  // namespace samfast

// While one workgroup per CU does it; the time hardly depends on the rows, so the wider W needs enough of them to be ahead.  us, three launches /
// one (medians of nine recordings of twenty, which spread by 1 %): width 768, 16 rows 11.1 / 11.0, 1024 12.5 / 11.8, 2048 14.5 / 12.3, 4096 19.7 / 13.3, 4097 19.8 / 17.8,
// 6144 23.8 / 19.4, 8192 25.3 / 20.6, two rounds from 8193 on (8200 26.5 / 33.0); width 1024, 1024 rows 15.3 / 17.0, 1536 17.1 / 17.2, 1664 17.3 / 17.4, 1792 18.2 / 17.4, 3072 22.2 /
// 18.5, 4096 24.2 / 20.3, 4100 26.0 / 26.0, 4224 26.3 / 25.5, 4608 26.9 / 26.3, 5120 26.7 / 25.6, 6144 28.5 / 27.3, 8192 32.7 / 30.2 (8200 35.4 / 48.3).
extern "C" int samfast_proj_block_pays(int64_t M, int C) {
  return (C == 768 || (C == 1024 && M > 1664)) && M <= 8192;
}

extern "C" int samfast_proj_block_i8(const void* x, int64_t ldx, const int8_t* wq, const float* sw, const float* bias,
                                     const void* residual, void* tokens, const void* gamma, const void* beta, float eps,
                                     int8_t* xq, float* sx, int64_t M, int C, int dtype, void* stream) {
  using namespace samfast;
  if (dtype != SAMFAST_BF16) SF_FAIL(SAMFAST_E_UNSUPPORTED, "proj_block: only bf16");
  if (C != 768 && C != 1024) SF_FAIL(SAMFAST_E_UNSUPPORTED, "proj_block: width %d, 768 and 1024 are built", C);
  SF_REQUIRE(M >= 0 && M * (int64_t)C < (1ll << 31), "proj_block: bad M=%lld", (long long)M);
  if (M == 0) return SAMFAST_OK;
  SF_REQUIRE(x && wq && sw && residual && tokens && gamma && beta && xq && sx, "proj_block: null pointer");
  SF_REQUIRE(aligned16(x) && aligned16(wq) && aligned16(sw) && aligned16(bias) && aligned16(residual) && aligned16(tokens) && aligned16(gamma) &&
             aligned16(beta) && aligned16(xq), "proj_block: operands must be 16-byte aligned");
  SF_REQUIRE(ldx >= C && ldx % 8 == 0 && eps > 0.f, "proj_block: ldx=%lld must be >= C and a multiple of 8, eps positive", (long long)ldx);
  ProjBlockArgs a = {};
  a.x = reinterpret_cast<const unsigned short*>(x);
  a.ldx = ldx;
  a.w = wq;
  a.sw = sw;
  a.bias = bias;
  a.residual = reinterpret_cast<const unsigned short*>(residual);
  a.tokens = reinterpret_cast<unsigned short*>(tokens);
  a.q.gamma = reinterpret_cast<const unsigned short*>(gamma);
  a.q.beta = reinterpret_cast<const unsigned short*>(beta);
  a.q.xq = xq;
  a.q.sx = sx;
  a.q.M = M;
  a.q.K = C;
  a.q.eps = eps;
  a.q.inv_K = 1.0f / (float)C;
  a.q.kb64 = 1;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const int rt = M <= 4096 ? 1 : 2;
  const dim3 grid((unsigned int)((M + 16 * rt - 1) / (16 * rt)));
#define SF_PROJ(W) do { if (rt == 1) hipLaunchKernelGGL((proj_block_i8_kernel<W, 1>), grid, dim3(512), 0, s, a); \
                        else hipLaunchKernelGGL((proj_block_i8_kernel<W, 2>), grid, dim3(512), 0, s, a); } while (0)
  if (C == 768) SF_PROJ(768);
  else SF_PROJ(1024);
#undef SF_PROJ
  return check_launch("proj_block_i8_kernel");
}
