// int8 GEMM with GELU for K = 768 whose output the GPU holds once (lin1 of an image at width 768): one workgroup per CU, 128 rows
// whose codes lie in LDS for the whole of K, by 384 columns, 48 to a wavefront.
//
// What bounds such a product (4096 x 768 -> 3072: 19 GOP, 4.5 us of matrix pipe) is its ends - launching 256 workgroups 1.9 us, first operands
// 1, output 3, with GELU 5 of vector work - and operand delivery, so a tile is as large as one per CU can be and nothing in its loop
// meets: after two barriers for X every wavefront runs on W alone, through a ring of its own in LDS (in the order of memory the load path
// gives 56 bytes a cycle; fragments straight into registers, 16 bytes of each of 16 rows to a quarter of the lanes, 33).
// The columns of a fragment pair are dealt so that a lane ends with eight adjacent ones: stores without a turn through LDS.
// us, 64 x 128 tiles / this one, K-block-major operands: 4096 x 768 -> 3072 18.9 / 16.8, 4900 x 768 -> 2304 17.8 / 16.4, 8192 x 768 -> 1536 18.6 /
// 16.7; one image of ViT-B, twelve of these launches, 1474 / 1466 (medians of fifteen turns).  Without GELU the other members are level (15.4 / 15.2, 13.9 / 14.1, 14.9 / 14.6): not built.
// Integer sums and the epilogue's arithmetic are those of the other members: the same bits.
#include "attn_relpos_shared.hpp"
#include "gemm_i8_shared.hpp"

// every fp32 step below is rounded on its own (no fused multiply-add), as in the other forms
#pragma clang fp contract(off)

namespace samfast {

// at most n vector memory operations of this wavefront outstanding (n constant at every use)
SF_DEVICE void strip_wait(int n) {
  switch (n) {
#define SF_CASE(H) case H: __builtin_amdgcn_s_waitcnt(0x0F70 | (H)); break
    SF_CASE(0); SF_CASE(1); SF_CASE(2); SF_CASE(3); SF_CASE(4); SF_CASE(5); SF_CASE(6); SF_CASE(7);
    SF_CASE(8); SF_CASE(9); SF_CASE(10); SF_CASE(11); SF_CASE(12); SF_CASE(13); SF_CASE(14); SF_CASE(15);
#undef SF_CASE
  }
  __builtin_amdgcn_sched_barrier(0);
}

__global__ __launch_bounds__(512, 2) void gemm_i8_strip_kernel(GemmArgs a) {
  constexpr int NK = 12, NF = 3, RF = 8;        // k steps of 64, fragments of 16 columns and of 16 rows
  constexpr int BM = 16 * RF, BN = 8 * 16 * NF;
  constexpr int BLOCK = BM * GLD;               // LDS bytes of 64 bytes of every row
  constexpr int RING = 7;                       // fragments (1 KB) of W of a wavefront in LDS
  constexpr int FRAGS = NK * NF, FIRST = NK + RING;  // requests in front of the loop
  __shared__ __attribute__((aligned(16))) unsigned char lds[NK * BLOCK + 8 * RING * 1024];
  static_assert(sizeof(lds) <= 160 * 1024, "LDS of a CU");

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lq = lane >> 4;

  const unsigned int total = (unsigned int)a.tiles_m * (unsigned int)a.tiles_n;
  const unsigned int pid = xcd_contiguous_id(blockIdx.x, total);
  if (pid >= total) return;  // uniform over the workgroup
  const unsigned int per_group = (unsigned int)a.group_m * a.tiles_n;
  const unsigned int first_m = (pid / per_group) * a.group_m;
  const unsigned int gsz = min((unsigned int)a.tiles_m - first_m, (unsigned int)a.group_m);
  const unsigned int in_group = pid % per_group;
  // the last tiles are moved back inside (M >= BM, N >= BN): rows and columns of two tiles get the same bits twice
  const int m0 = min((int)(first_m + in_group % gsz) * BM, a.M - BM);
  const int n0 = min((int)(in_group / gsz) * BN, a.N - BN) + wave * 16 * NF;

  // ---- scales and bias: row 16 t + lr; columns 8 lq + 4 j of the first 32, 32 + 4 lq --------------------------------------------------
  float sx[RF];
#pragma unroll
  for (int t = 0; t < RF; ++t) sx[t] = a.sx[m0 + 16 * t + lr];
  f32x4 sw[NF], bias[NF];
  const float* bias_or_sw = a.bias ? a.bias : a.sw;
#pragma unroll
  for (int j = 0; j < NF; ++j) {
    const int n = n0 + (j < 2 ? 8 * lq + 4 * j : 32 + 4 * lq);
    sw[j] = *reinterpret_cast<const f32x4*>(a.sw + n);
    bias[j] = *reinterpret_cast<const f32x4*>(bias_or_sw + n);
  }
  __builtin_amdgcn_sched_barrier(0);

  // ---- requests.  Row r of a fragment is 64 bytes at 64 r in LDS, its 16-byte chunk c at position c ^ (-(r / 4) & 3); row r of W
  // fragment j is column 8 (r / 4) + 4 j + r % 4, or 32 + r -------------------------------------------------------------------------------
  const int r = lane >> 2, chunk = ((lane & 3) ^ (-(r >> 2) & 3)) * 16;
  const unsigned int x_off = (unsigned int)((wave * 16 + r) * a.x_pitch + chunk);
  unsigned int w_off[NF];
#pragma unroll
  for (int j = 0; j < NF; ++j) w_off[j] = (unsigned int)((j < 2 ? (r >> 2) * 8 + 4 * j + (r & 3) : 32 + r) * a.w_pitch + chunk);
  const unsigned int lds_at = (unsigned int)(uintptr_t)((__attribute__((address_space(3))) unsigned char*)lds);
  const unsigned int ring_at = lds_at + NK * BLOCK + wave * RING * 1024;
  const unsigned char* xb = reinterpret_cast<const unsigned char*>(a.x) + (int64_t)m0 * a.x_pitch;
  const unsigned char* wb = reinterpret_cast<const unsigned char*>(a.w) + (int64_t)n0 * a.w_pitch;
  auto load_x = [&](int k) __attribute__((always_inline)) { lds_dma16(xb + k * a.x_kstep, x_off, lds_at + k * BLOCK + wave * 1024); };
  auto load_w = [&](int f) __attribute__((always_inline)) { lds_dma16(wb + f / NF * a.w_kstep, w_off[f % NF], ring_at + f % RING * 1024); };
#pragma unroll
  for (int k = 0; k < NK; ++k) {
    load_x(k);
#pragma unroll
    for (int f = k * NF; f < (k + 1) * NF; ++f)
      if (f < RING) load_w(f);
  }
  __builtin_amdgcn_sched_barrier(0);

  i32x4 acc[RF][NF];
#pragma unroll
  for (int t = 0; t < RF; ++t)
#pragma unroll
    for (int j = 0; j < NF; ++j) acc[t][j] = i32x4{0, 0, 0, 0};
  const int frag = lr * 64 + ((lq ^ (-(lr >> 2) & 3)) * 16);
  const unsigned char* xfrag = lds + frag;
  const unsigned char* wfrag = lds + NK * BLOCK + wave * RING * 1024 + frag;
  // of a SIMD's two wavefronts one multiplies ahead of the other and runs its GELU under the other's products (4096 x 768 -> 3072 19.4 / 19.1 us)
  if (wave < 4) __builtin_amdgcn_s_setprio(3);
  else __builtin_amdgcn_s_setprio(2);
#pragma unroll
  for (int k = 0; k < NK; ++k) {
    // outstanding behind what step k reads, of X 0, W 0-2, X 1, W 3-5, X 2, W 6, X 3, .. X 11, W 7, ..: in step 0 X 0 and 1 (and W 0-2), in step 1 W 3-5, from
    // step 2 on W 3 k + 2, in front of which every X has come
    const int issued = min(FIRST + k * NF, NK + FRAGS);
    const int needed = k == 0 ? 5 : k == 1 ? 8 : NK + (k + 1) * NF;
    strip_wait(min(issued - needed, 15));
    if (k == 0 || k == 2) {  // X is everybody's
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
    }
    i32x4 xf[RF], wf[NF];
#pragma unroll
    for (int t = 0; t < RF; ++t) xf[t] = *reinterpret_cast<const i32x4*>(xfrag + k * BLOCK + t * 1024);
#pragma unroll
    for (int j = 0; j < NF; ++j) wf[j] = *reinterpret_cast<const i32x4*>(wfrag + (k * NF + j) % RING * 1024);
    __builtin_amdgcn_s_waitcnt(0xC07F);  // the fragments are in registers: their places are requested anew
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int f = k * NF + RING; f < (k + 1) * NF + RING; ++f)
      if (f < FRAGS) load_w(f);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < RF; ++t)
#pragma unroll
      for (int j = 0; j < NF; ++j) acc[t][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wf[j], xf[t], acc[t][j], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
  }

  __builtin_amdgcn_s_setprio(0);
  if (!a.bias)  // uniform
#pragma unroll
    for (int j = 0; j < NF; ++j) bias[j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const unsigned int out_off = (unsigned int)(lr * a.ldo) * 2u;
  unsigned char* out = reinterpret_cast<unsigned char*>(reinterpret_cast<unsigned short*>(a.out) + (int64_t)m0 * a.ldo + n0);
#pragma unroll
  for (int t = 0; t < RF; ++t) {
    unsigned int o[NF][2];
#pragma unroll
    for (int j = 0; j < NF; ++j)
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        float y[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          // three separately rounded fp32 operations (no fused multiply-add)
          float v = (float)acc[t][j][2 * c + e] * sx[t];
          v = v * sw[j][2 * c + e];
          y[e] = v + bias[j][2 * c + e];
        }
        o[j][c] = pack_bf16x2(y[0], y[1]);
        // activation of the bf16-rounded Linear output, as a separate GELU would see it
        o[j][c] = pack_bf16x2(gelu_erf(bf16_lo_to_f32(o[j][c])), gelu_erf(bf16_hi_to_f32(o[j][c])));
      }
    unsigned char* row = out + (int64_t)(16 * t) * a.ldo * 2 + out_off;
    *reinterpret_cast<u32x4*>(row + 16 * lq) = u32x4{o[0][0], o[0][1], o[1][0], o[1][1]};
    *reinterpret_cast<u32x2*>(row + 64 + 8 * lq) = u32x2{o[2][0], o[2][1]};
  }
}

// From seven eighths of the CUs on; below, the smaller tiles (4096 x 768 -> 2304, 192 tiles: 15.5 / 15.9, 3000 x 768 -> 3072 15.5 / 15.8).
bool gemm_i8_strip_covers(int epi, const GemmArgs& a) {
  const int mode = knob_or(KNOB_GEMM_STRIP, 1);
  if (mode <= 0 || epi != EPI_GELU_BF16 || a.dst_row || a.tile_counters) return false;
  if (a.K != 768 || a.M < 128 || a.N < 384 || a.ldo >= (1ll << 24)) return false;
  const int64_t tiles = (int64_t)((a.M + 127) / 128) * ((a.N + 383) / 384);
  return mode >= 2 || (tiles <= 256 && tiles >= 224);
}

int gemm_i8_strip_launch(const GemmArgs& a0, hipStream_t stream) {
  GemmArgs a = a0;
  a.tiles_m = (a.M + 127) / 128;
  a.tiles_n = (a.N + 383) / 384;
  a.group_m = 8;  // an XCD's 32 tiles: 8 row tiles x 4 column tiles
  const dim3 grid((unsigned int)((a.tiles_m * a.tiles_n + 7) / 8 * 8));
  hipLaunchKernelGGL(gemm_i8_strip_kernel, grid, dim3(512), 0, stream, a);
  return check_launch("gemm_i8_strip_kernel");
}

}  // namespace samfast
