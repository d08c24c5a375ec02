// The middle of an int8 block for an image or two in one launch: the attention output's row quantiser, proj, the residual add, norm2 and
// lin1's row quantiser.
//
// At 4096 rows the three launches of it (5.0, 8.7 and 5.4 us at width 768) are mostly starts, ends and latency.  Here a workgroup
// owns 16 whole rows (32 from 4097 rows on), so nothing between the quantisers leaves the CU: eight wavefronts quantise the rows into LDS,
// multiply them by all of W - each its own eighth of the columns, fragments straight from the K-block-major weight into
// registers, 1 KB a load, requested before the rows are there - and finish whole rows again, one wavefront each, with the quantiser's
// own code.  What bounds it is W through the load path of every CU, 0.6 MB at 56 bytes a cycle: 4.5 us of the 16 (1.6 MB and 12 us at width
// 1280, where the three launches stay ahead, 27.5 / 35.3 us at 4096 rows; 24.7 / 25.0 at width 1024: only 768 is built).
//
// Codes, sums, roundings and scales are those of the separate launches: the same bits.
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

template <int C, int RT>
__global__ __launch_bounds__(512) void proj_block_i8_kernel(ProjBlockArgs a) {
  constexpr int EPC = quant_epc_for(C), NCH = quant_nch_for(C), NCHUNK = C / EPC;
  using In = RowQuantizer<NCH, EPC, false>;
  using Ln = RowQuantizer<NCH, EPC, true>;
  typedef typename In::in_t in_t;
  constexpr int R = 16 * RT, RPW = 2 * RT;      // rows of the workgroup, of a wavefront
  constexpr int NF = C / 128, NK = C / 64;      // column fragments of a wavefront, k steps
  constexpr int AHEAD = 7;                      // k steps of W in registers
  constexpr int CP = C + 16, OP = 2 * C + 16;   // LDS row pitches: codes, Linear output
  __shared__ __attribute__((aligned(16))) unsigned char lds[R * (CP > OP ? CP : OP) + R * CP];
  __shared__ float scales[R];
  unsigned char* codes = lds;                   // R rows
  unsigned char* rows = lds + R * CP;           // R rows of bf16
  static_assert(R * CP + R * OP <= (int)sizeof(lds), "codes and rows side by side");

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lq = lane >> 4;
  const int64_t row0 = (int64_t)blockIdx.x * R;
  const int64_t last = a.q.M - 1;

  // ---- loads that wait for nothing: the rows to quantise, W's first k steps, the residual rows, gamma and beta ----------------------
  in_t xw[RPW][NCH], res[RPW][NCH], gw[NCH], bw[NCH];
#pragma unroll
  for (int r = 0; r < RPW; ++r) In::template load_row<false>(a.x + min(row0 + wave * RPW + r, last) * a.ldx, NCHUNK, lane, xw[r]);
  const int8_t* wlane = a.w + (int64_t)(wave * (C / 8) + lr) * 64 + lq * 16;
  i32x4 wf[AHEAD][NF];
  auto load_w = [&](int k, i32x4 (&f)[NF]) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < NF; ++j) f[j] = *reinterpret_cast<const i32x4*>(wlane + (int64_t)k * C * 64 + j * 1024);
  };
#pragma unroll
  for (int k = 0; k < AHEAD; ++k) {
    load_w(k, wf[k]);
    __builtin_amdgcn_sched_barrier(0);
  }

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
    const float scale = In::finish(a.q, NCHUNK, lane, xw[r], gw, bw, [&](int c, const unsigned int (&v)[EPC / 4]) {
#pragma unroll
      for (int e = 0; e < EPC / 4; ++e) reinterpret_cast<unsigned int*>(codes + row * CP + c * EPC)[e] = v[e];
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
#pragma unroll
  for (int k = 0; k < NK; ++k) {
    i32x4 f[RT];
#pragma unroll
    for (int t = 0; t < RT; ++t) f[t] = *reinterpret_cast<const i32x4*>(codes + (16 * t + lr) * CP + k * 64 + lq * 16);
#pragma unroll
    for (int j = 0; j < NF; ++j)
#pragma unroll
      for (int t = 0; t < RT; ++t) acc[t][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wf[k % AHEAD][j], f[t], acc[t][j], 0, 0, 0);
    if (k + AHEAD < NK) load_w(k + AHEAD, wf[k % AHEAD]);
    __builtin_amdgcn_sched_barrier(0);  // (products and loads in this order: gathered, the loads behind would wait for all in front)
    if (k == NK - AHEAD) {
      // the residual rows and norm2's parameters travel under the last products
#pragma unroll
      for (int r = 0; r < RPW; ++r) Ln::template load_row<false>(a.residual + min(row0 + wave * RPW + r, last) * C, NCHUNK, lane, res[r]);
      Ln::load_affine(a.q.gamma, a.q.beta, NCHUNK, lane, gw, bw);
    }
  }
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    const float sx = scales[16 * t + lr];
#pragma unroll
    for (int j = 0; j < NF; ++j) {
      const int n = wave * (C / 8) + 16 * j + 4 * lq;
      const f32x4 sw = *reinterpret_cast<const f32x4*>(a.sw + n);
      f32x4 bias = {0.f, 0.f, 0.f, 0.f};
      if (a.bias) bias = *reinterpret_cast<const f32x4*>(a.bias + n);
      float y[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        // three separately rounded fp32 operations (no fused multiply-add)
        float v = (float)acc[t][j][e] * sx;
        v = v * sw[e];
        y[e] = v + bias[e];
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

// A workgroup's time is the same for one row and for sixteen, so the three launches are ahead while they leave CUs idle and the one where its
// grid is most of a round of 256 workgroups, of 16 rows up to 4096 and of 32 up to 8192.  us, three launches / one: 16 rows
// 11.6 / 14.3, 2048 15.2 / 15.7, 2560 16.5 / 15.8, 4096 20.2 / 16.3, 4100 20.2 / 20.9, 5000 22.1 / 21.5, 6144 23.9 / 22.1, 8192
// 25.7 / 23.0.
extern "C" int samfast_proj_block_pays(int64_t M, int C) {
  return C == 768 && ((M > 2304 && M <= 4096) || (M > 5120 && M <= 8192));
}

extern "C" int samfast_proj_block_i8(const void* x, int64_t ldx, const int8_t* wq, const float* sw, const float* bias,
                                     const void* residual, void* tokens, const void* gamma, const void* beta, float eps,
                                     int8_t* xq, float* sx, int64_t M, int C, int dtype, void* stream) {
  using namespace samfast;
  if (dtype != SAMFAST_BF16) SF_FAIL(SAMFAST_E_UNSUPPORTED, "proj_block: only bf16");
  if (C != 768) SF_FAIL(SAMFAST_E_UNSUPPORTED, "proj_block: width %d, only 768 is built", C);
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
  if (rt == 1) hipLaunchKernelGGL((proj_block_i8_kernel<768, 1>), grid, dim3(512), 0, s, a);
  else hipLaunchKernelGGL((proj_block_i8_kernel<768, 2>), grid, dim3(512), 0, s, a);
  return check_launch("proj_block_i8_kernel");
}
