// 2:4-sparse product with scale + bias epilogue over few rows: the K range dealt out over the eight
// wavefronts of a workgroup (see gemm_i8_skinny_kernel in linear_i8_small.hip), for launches whose
// 256 x 128 tiles would leave most CUs empty and walk K serially.
//
// v_smfmac_i32_32x32x64_i8 with W as the sparse operand: a lane (row lane % 32, half h) takes 16 stored
// bytes and one index word of a packed row and 32 consecutive k (32h ..) of an X row (operand order:
// gemm_i8_sparse24.hip).  Both operands go from memory straight into registers,
// DEPTH k steps ahead; the packed weight is K-block major, so its loads are whole 1 KB runs.
#include "gemm_i8_sparse24_shared.hpp"

// every fp32 step below is rounded on its own (no fused multiply-add)
#pragma clang fp contract(off)

namespace samfast {

constexpr int kSpWaves = 8;

// a workgroup's tile: 32 tokens x 32 channels
__global__ __launch_bounds__(64 * kSpWaves, 2) void gemm_i8_sp24_skinny_kernel(SparseArgs a) {
  __shared__ __attribute__((aligned(16))) int red[kSpWaves * 1024];
  constexpr int DEPTH = 4;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 31, lh = lane >> 5;
  // (tiles_x / tiles_w count this kernel's tiles) token tiles of one channel panel side by side on an XCD
  const unsigned int total = (unsigned int)(a.tiles_x * a.tiles_w);
  const unsigned int pid = xcd_contiguous_id(blockIdx.x, total);
  if (pid >= total) return;  // uniform
  const int m0 = (int)(pid % a.tiles_x) * 32, n0 = (int)(pid / a.tiles_x) * 32;
  const int nc = min(n0 + lr, a.N - 1);
  const int8_t* xrow = a.x + (int64_t)min(m0 + lr, a.M - 1) * a.x_row_pitch + 32 * lh;
  const int8_t* wrow = a.wc + (int64_t)nc * 32 + 16 * lh;
  const int32_t* irow = a.widx + (int64_t)nc * 2 + lh;
  const int nk = a.K / SBK;
  const int steps = (nk - wave + kSpWaves - 1) / kSpWaves;  // 0 for the last wavefronts of a short K

  i32x4 wf[DEPTH];
  int ix[DEPTH];
  i32x8 xf[DEPTH];
  auto request = [&](int i, int d) {
    const int64_t step = wave + kSpWaves * i;
    wf[d] = *reinterpret_cast<const i32x4*>(wrow + step * a.N * 32);
    ix[d] = irow[step * a.N * 2];
    const i32x4 lo = *reinterpret_cast<const i32x4*>(xrow + step * a.x_kstep);
    const i32x4 hi = *reinterpret_cast<const i32x4*>(xrow + step * a.x_kstep + 16);
    xf[d] = i32x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  };
#pragma unroll
  for (int d = 0; d < DEPTH; ++d)
    if (d < steps) request(d, d);
  i32x16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0;
  for (int i = 0; i < steps; i += DEPTH) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d)
      if (i + d < steps) {
        acc = __builtin_amdgcn_smfmac_i32_32x32x64_i8(wf[d], xf[d], acc, ix[d], 0, 0);
        if (i + d + DEPTH < steps) request(i + d + DEPTH, d);
      }
  }

  // partial sums [wave][register][lane]: lane = token lane % 32, channels 8 (r/4) + 4 (lane/32) + r%4
#pragma unroll
  for (int r = 0; r < 16; ++r) red[wave * 1024 + r * 64 + lane] = acc[r];
  __syncthreads();
  // a thread finishes two adjacent channels of one token; 16 consecutive threads: one token row
  const int tok = tid >> 4, c = 2 * (tid & 15);
  const int row = m0 + tok, n = n0 + c;
  if (row >= a.M || n >= a.N) return;  // N % 8 == 0: a pair is in or out together
  const int at = (4 * (c >> 3) + (c & 3)) * 64 + 32 * ((c >> 2) & 1) + tok;
  int s0 = 0, s1 = 0;
#pragma unroll
  for (int w = 0; w < kSpWaves; ++w) {
    s0 += red[w * 1024 + at];
    s1 += red[w * 1024 + at + 64];
  }
  const float s = a.sx[row];
  float b0 = 0.f, b1 = 0.f;
  if (a.bias) { b0 = a.bias[n]; b1 = a.bias[n + 1]; }
  float t0 = (float)s0 * s, t1 = (float)s1 * s;
  t0 = t0 * a.sw[n];
  t1 = t1 * a.sw[n + 1];
  *reinterpret_cast<unsigned int*>(reinterpret_cast<unsigned short*>(a.out) + (int64_t)row * a.ldo + n) = pack_bf16x2(t0 + b0, t1 + b1);
}

static int64_t skinny_tiles(const SparseArgs& a) { return (int64_t)((a.M + 31) / 32) * ((a.N + 31) / 32); }

bool gemm_i8_sp24_skinny_covers(int epi, const SparseArgs& a) {
  if (knob_or(KNOB_GEMM_SKINNY, 1) <= 0 || epi != SEPI_SCALE_BIAS) return false;
  // up to two tiles per CU, three on a long K loop: beyond that the operand reads (64 bytes per
  // multiply-add tile row, no reuse between workgroups but through the caches) cost more than the serial
  // loop of the 256 x 128 tiles.  256 x 1280 x 1280: 320 tiles 6.9 us against 10.0; 512 x 768 x 3072: 384
  // tiles 8.8 against 16.9; 256 x 3840 x 1280: 960 tiles 11.3 against 10.2
  return skinny_tiles(a) <= (a.K >= 2048 ? 768 : 512);
}

int gemm_i8_sp24_skinny_launch(const SparseArgs& a0, hipStream_t stream) {
  SparseArgs a = a0;
  a.tiles_x = (a.M + 31) / 32;
  a.tiles_w = (a.N + 31) / 32;
  const unsigned int grid = (unsigned int)((a.tiles_x * a.tiles_w + 7) / 8 * 8);
  hipLaunchKernelGGL(gemm_i8_sp24_skinny_kernel, dim3(grid), dim3(64 * kSpWaves), 0, stream, a);
  return check_launch("gemm_i8_sp24_skinny_kernel");
}

}  // namespace samfast
