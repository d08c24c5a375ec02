// A whole quantised Linear over few rows in one launch: row quantiser, int8 product and
// the scale + bias epilogue (what quant_rowwise.hip + gemm_i8.hip do in two).
//
// Such a call is latency: the two launches and their gap, a row's way through memory twice, and a
// K loop that a 64 x 128 tile walks serially on a GPU it leaves empty.  Here a 512-thread workgroup
// owns 16 * NT output columns (2:4: 32) of 8 or 16 rows:
//   * every wavefront first requests its share of the weight columns straight into registers (the K
//     range is dealt out to the eight wavefronts in steps of 64, at most NCH each), so that the
//     weights travel while the rows are quantised;
//   * the workgroup quantises the rows itself - each workgroup repeats that for its own columns, which
//     is why the form ends at a few hundred rows - and leaves the codes in LDS; one row to a wavefront: what bounds it is that
//     chain of 50 to 200 vector instructions per 512 values (blocks of 32 rows took 1-3 us more throughout);
//   * v_mfma_i32_16x16x64_i8, codes as A and weights as B (both take 16 consecutive k bytes of one
//     row per lane; 2:4: v_smfmac_i32_32x32x64_i8), then the eight partial sums meet in LDS: integer sums, so the order is free
//     and the results have the bits of the two-launch form.
#include "gemm_i8_shared.hpp"
#include "linear_i8_small.hpp"
#include "quant_row.hpp"
#include "samfast_bench.h"

// every fp32 step below is rounded on its own (no fused multiply-add), as in the other forms
#pragma clang fp contract(off)

namespace samfast {

struct SmallArgs {
  const unsigned short* x;  // one launch: bf16 rows
  int64_t ldx;
  const int8_t* xq;         // product alone: codes, and their row scales
  const float* sx;
  const int8_t* w;
  const float* sw;
  const float* bias;
  unsigned short* y;
  int64_t ldy;
  int M, N, K;
  int x_pitch, w_pitch;      // bytes between consecutive code / weight rows: K, or 64 (K-block major)
  int64_t x_kstep, w_kstep;  // bytes between consecutive 64-byte k steps: 64, or rows * 64
  int tiles_m, tiles;  // row blocks or row tiles, all tiles
  const int32_t* widx;  // 2:4 weights: `w` holds (K/64, N, 32) bytes, this (K/64, N, 2) words
};

constexpr int kSmallWaves = 8;

// The eight wavefronts' partial sums of a 16 MT x 16 NT tile meet in LDS ([wave][m][t][register][lane]; a
// lane holds column lane % 16, rows 4 (lane / 16) + register of its 16 x 16 tiles) and leave through the
// scale + bias epilogue, two adjacent columns of one row per thread.
template <int MT, int NT, typename RowScale>
SF_DEVICE void finish_tile(const SmallArgs& a, const i32x4 (&acc)[MT][NT], unsigned char* lds, int m0, int n0, int tid, RowScale row_scale) {
  const int lane = tid & 63, wave = tid >> 6;
  int* red = reinterpret_cast<int*>(lds);
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) red[((wave * MT + m) * NT + t) * 256 + r * 64 + lane] = acc[m][t][r];
  __syncthreads();
  for (int p = tid; p < MT * NT * 128; p += 64 * kSmallWaves) {
    // consecutive threads: the column pairs of one row, then the next row
    const int pair = p % (8 * NT), r = p / (8 * NT);
    const int t = pair / 8, c = 2 * (pair % 8), m = r / 16, row16 = r % 16;
    const int row = m0 + r, n = n0 + 16 * t + c;
    if (row >= a.M || n >= a.N) continue;  // N % 8 == 0: a pair is in or out together
    const int at = (m * NT + t) * 256 + (row16 & 3) * 64 + (row16 >> 2) * 16 + c;
    int s0 = 0, s1 = 0;
#pragma unroll
    for (int w = 0; w < kSmallWaves; ++w) {
      const u32x2 v = *reinterpret_cast<const u32x2*>(red + w * (MT * NT * 256) + at);
      s0 += (int)v[0];
      s1 += (int)v[1];
    }
    const float s = row_scale(row);
    float b0 = 0.f, b1 = 0.f;
    if (a.bias) { b0 = a.bias[n]; b1 = a.bias[n + 1]; }
    float t0 = (float)s0 * s, t1 = (float)s1 * s;
    t0 = t0 * a.sw[n];
    t1 = t1 * a.sw[n + 1];
    *reinterpret_cast<unsigned int*>(a.y + (int64_t)row * a.ldy + n) = pack_bf16x2(t0 + b0, t1 + b1);
  }
}

// The eight wavefronts quantise rows m0 .. m0 + 8 RPW - 1 (wave + 8 j of them is a wavefront's) into `codes`, their scales into `sx`.
template <int NCH, int RPW>
SF_DEVICE void quantize_rows(const SmallArgs& a, int m0, float* sx, unsigned char* codes, int pitch, int wave, int lane) {
  // the arithmetic of RowQuantizer::finish_row
  const int nchunk = a.K / 8;
  u32x4 xw[RPW][NCH];
#pragma unroll
  for (int j = 0; j < RPW; ++j) {
    const int row = m0 + wave + kSmallWaves * j;
    const u32x4* src = reinterpret_cast<const u32x4*>(a.x + row * a.ldx);
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const u32x4 z = {0u, 0u, 0u, 0u};
      xw[j][i] = z;
      if (row < a.M && lane + 64 * i < nchunk) xw[j][i] = src[lane + 64 * i];
    }
  }
  // (rows at or past M hold zeros: they are quantised along, which keeps the rows' serial chains -
  // maximum, lane reduction, two divisions - independent and in flight together)
#pragma unroll
  for (int j = 0; j < RPW; ++j) {
    const int row = wave + kSmallWaves * j;
    float f[NCH][8], amax;
#pragma unroll
    for (int i = 0; i < NCH; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        f[i][2 * e] = bf16_lo_to_f32(xw[j][i][e]);
        f[i][2 * e + 1] = bf16_hi_to_f32(xw[j][i][e]);
      }
    const bool row_nan = wave_absmax(f, amax);
    const QuantScale q(amax);
#pragma unroll
    for (int i = 0; i < NCH; ++i)
      if (lane + 64 * i < nchunk) {
        unsigned int c[2];
        quantize_chunk<8>(f[i], q, c);
        const u32x2 o = {c[0], c[1]};
        *reinterpret_cast<u32x2*>(codes + row * pitch + (lane + 64 * i) * 8) = o;
      }
    if (lane == 0) sx[row] = row_nan ? __uint_as_float(0x7fc00000u) : q.scale;
  }
}

template <int NCH, int RPW, int NT>  // RPW: rows per wavefront, so blocks of 8 or 16 rows
__global__ __launch_bounds__(64 * kSmallWaves, 2) void linear_i8_small_kernel(SmallArgs a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  constexpr int ROWS = 16;
  float* sx = reinterpret_cast<float*>(lds);          // ROWS scales
  unsigned char* codes = lds + ROWS * 4;              // ROWS x (K + 16) bytes; later the partial sums
  const int pitch = a.K + 16;                         // an odd number of 16-byte pieces: operand reads spread over the banks
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // row blocks of one column panel next to each other on an XCD
  const unsigned int pid = xcd_contiguous_id(blockIdx.x, a.tiles);
  if (pid >= (unsigned int)a.tiles) return;  // uniform
  const int m0 = (int)(pid % a.tiles_m) * 8 * RPW, n0 = (int)(pid / a.tiles_m) * 16 * NT;
  const int nk = a.K / 64;
  const int lr = lane & 15, lq = lane >> 4;

  // weights first: step wave + 8 i, columns n0 + 16 t + lr, k bytes 16 lq .. +15
  i32x4 wf[NCH][NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int8_t* wrow = a.w + (int64_t)min(n0 + 16 * t + lr, a.N - 1) * a.w_pitch + 16 * lq;
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int step = wave + kSmallWaves * i;
      if (step < nk) wf[i][t] = *reinterpret_cast<const i32x4*>(wrow + step * a.w_kstep);  // uniform
    }
  }
  quantize_rows<NCH, RPW>(a, m0, sx, codes, pitch, wave, lane);
  __syncthreads();

  i32x4 acc[1][NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[0][t] = i32x4{0, 0, 0, 0};
#pragma unroll
  for (int i = 0; i < NCH; ++i) {
    const int step = wave + kSmallWaves * i;
    if (step < nk) {
      const i32x4 xf = *reinterpret_cast<const i32x4*>(codes + lr * pitch + step * 64 + 16 * lq);
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[0][t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(xf, wf[i][t], acc[0][t], 0, 0, 0);
    }
  }

  __syncthreads();  // nobody reads the codes any more
  // (of a block of 8 rows the upper half of the product's 16 is whatever stood in LDS, and nobody's)
  SmallArgs b = a;
  b.M = min(a.M, m0 + 8 * RPW);
  finish_tile<1, NT>(b, acc, codes, m0, n0, tid, [&](int row) { return sx[row - m0]; });
}

// The same with 2:4 weights, in the packed order of gemm_i8_sparse24.hip: v_smfmac_i32_32x32x64_i8, weights (the sparse operand)
// as the rows, tokens as the columns.  A workgroup owns 32 channels of 8 rows.
template <int NCH>
__global__ __launch_bounds__(64 * kSmallWaves, 2) void linear_i8_sp24_small_kernel(SmallArgs a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  typedef int i32x8 __attribute__((ext_vector_type(8)));
  constexpr int ROWS = 8;
  float* sx = reinterpret_cast<float*>(lds);          // ROWS scales, in the first 64 bytes
  unsigned char* codes = lds + 64;
  const int pitch = a.K + 16;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const unsigned int pid = xcd_contiguous_id(blockIdx.x, a.tiles);
  if (pid >= (unsigned int)a.tiles) return;  // uniform
  const int m0 = (int)(pid % a.tiles_m) * ROWS, n0 = (int)(pid / a.tiles_m) * 32;
  const int nk = a.K / 64;
  const int lr = lane & 31, lh = lane >> 5;

  i32x4 wf[NCH];
  int ix[NCH];
  {
    const int nc = min(n0 + lr, a.N - 1);
    const int8_t* wrow = a.w + (int64_t)nc * 32 + 16 * lh;
    const int32_t* irow = a.widx + (int64_t)nc * 2 + lh;
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int64_t step = wave + kSmallWaves * i;
      if (step < nk) {  // uniform
        wf[i] = *reinterpret_cast<const i32x4*>(wrow + step * a.N * 32);
        ix[i] = irow[step * a.N * 2];
      }
    }
  }
  quantize_rows<NCH, 1>(a, m0, sx, codes, pitch, wave, lane);
  __syncthreads();

  i32x16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0;
#pragma unroll
  for (int i = 0; i < NCH; ++i) {
    const int step = wave + kSmallWaves * i;
    if (step < nk) {
      // (the columns beyond the eight tokens repeat the last one; nobody reads them)
      const unsigned char* p = codes + min(lr, ROWS - 1) * pitch + step * 64 + 32 * lh;
      const i32x4 lo = *reinterpret_cast<const i32x4*>(p), hi = *reinterpret_cast<const i32x4*>(p + 16);
      const i32x8 xf = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      acc = __builtin_amdgcn_smfmac_i32_32x32x64_i8(wf[i], xf, acc, ix[i], 0, 0);
    }
  }
  __syncthreads();  // nobody reads the codes any more

  // partial sums [wave][register][token], two runs of eight tokens a register: lane = token + 32 h, channels 8 (r/4) + 4 h + r%4
  int* red = reinterpret_cast<int*>(codes);
  if (lr < ROWS) {
#pragma unroll
    for (int r = 0; r < 16; ++r) red[wave * 256 + r * 16 + 8 * lh + lr] = acc[r];
  }
  __syncthreads();
  // a thread finishes two adjacent channels of one token; 16 consecutive threads: one token row
  if (tid >= 16 * ROWS) return;
  const int tok = tid >> 4, c = 2 * (tid & 15);
  const int row = m0 + tok, n = n0 + c;
  if (row >= a.M || n >= a.N) return;  // N % 8 == 0: a pair is in or out together
  const int at = (4 * (c >> 3) + (c & 3)) * 16 + 8 * ((c >> 2) & 1) + tok;
  int s0 = 0, s1 = 0;
#pragma unroll
  for (int w = 0; w < kSmallWaves; ++w) {
    s0 += red[w * 256 + at];
    s1 += red[w * 256 + at + 16];
  }
  const float s = sx[tok];
  float b0 = 0.f, b1 = 0.f;
  if (a.bias) { b0 = a.bias[n]; b1 = a.bias[n + 1]; }
  float t0 = (float)s0 * s, t1 = (float)s1 * s;
  t0 = t0 * a.sw[n];
  t1 = t1 * a.sw[n + 1];
  *reinterpret_cast<unsigned int*>(a.y + (int64_t)row * a.ldy + n) = pack_bf16x2(t0 + b0, t1 + b1);
}

// The product alone, on codes that a quantiser launch has written: the same dealing of the K range over
// eight wavefronts for launches whose 64 x 128 tiles would leave most CUs empty and walk K serially.
// A workgroup owns 16 MT rows x 16 NT columns; both operands go from memory into registers (K-block major:
// 1 KB of whole lines per load), DEPTH steps ahead.
template <int MT, int NT>
__global__ __launch_bounds__(64 * kSmallWaves, 2) void gemm_i8_skinny_kernel(SmallArgs a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  constexpr int DEPTH = MT + NT <= 4 ? 4 : 3;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lq = lane >> 4;
  // row tiles of one column panel next to each other on an XCD: the weights are the larger operand
  const unsigned int pid = xcd_contiguous_id(blockIdx.x, a.tiles);
  if (pid >= (unsigned int)a.tiles) return;  // uniform
  const int m0 = (int)(pid % a.tiles_m) * 16 * MT, n0 = (int)(pid / a.tiles_m) * 16 * NT;
  const int8_t* xrow[MT];
  const int8_t* wrow[NT];
#pragma unroll
  for (int m = 0; m < MT; ++m) xrow[m] = a.xq + (int64_t)min(m0 + 16 * m + lr, a.M - 1) * a.x_pitch + 16 * lq;
#pragma unroll
  for (int t = 0; t < NT; ++t) wrow[t] = a.w + (int64_t)min(n0 + 16 * t + lr, a.N - 1) * a.w_pitch + 16 * lq;
  const int nk = a.K / 64;
  const int steps = (nk - wave + kSmallWaves - 1) / kSmallWaves;  // 0 for the last wavefronts of a short K

  i32x4 xf[DEPTH][MT], wf[DEPTH][NT];
  auto request = [&](int i, int d) {
    const int64_t step = wave + kSmallWaves * i;
#pragma unroll
    for (int t = 0; t < NT; ++t) wf[d][t] = *reinterpret_cast<const i32x4*>(wrow[t] + step * a.w_kstep);
#pragma unroll
    for (int m = 0; m < MT; ++m) xf[d][m] = *reinterpret_cast<const i32x4*>(xrow[m] + step * a.x_kstep);
  };
#pragma unroll
  for (int d = 0; d < DEPTH; ++d)
    if (d < steps) request(d, d);
  i32x4 acc[MT][NT];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[m][t] = i32x4{0, 0, 0, 0};
  for (int i = 0; i < steps; i += DEPTH) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d)
      if (i + d < steps) {
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
          for (int t = 0; t < NT; ++t) acc[m][t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(xf[d][m], wf[d][t], acc[m][t], 0, 0, 0);
        if (i + d + DEPTH < steps) request(i + d + DEPTH, d);
      }
  }
  finish_tile<MT, NT>(a, acc, lds, m0, n0, tid, [&](int row) { return a.sx[row]; });
}

bool linear_i8_small_any_alignment(int64_t M, int K) { return M <= 8 || (M <= 16 && K <= 2048) || (M <= 32 && K <= 768); }

// Rows per wavefront * 8 + column tiles (16 columns each; 2:4: 32) of a workgroup; 0 = not this form.
// A call of one launch costs the host 4.5 to 6.3 us, of two 7.3 to 9.7, whatever the GPU does meanwhile; on the GPU every workgroup quantises its
// rows, so the form ends where that repetition, or another workgroup on a CU, makes it longer than the quantiser and the small-tile
// product.  GPU time in us, two launches / one (shape), at the last calls of each line and beyond:
//   int8, one column tile  up to 256 tiles, at any length 9 x 5120 -> 1280 8.2 / 6.5, 22 x 5120 -> 1280 8.4 / 6.6, 40 x 3072 -> 768 7.1 / 5.3, 58 x 2560 -> 264 6.6 / 5.0,
//         12 x 3072 -> 768 6.6 / 5.0; with rows of up to 1024 values three on a CU are ahead of wider ones (four column tiles / one: 168 x 1024 -> 488 5.0 / 4.7, 203 x 768 -> 424 4.6 / 4.4,
//         259 x 384 -> 288 3.9 / 3.65; 780 tiles: 158 x 1024 -> 624 5.10 / 5.13, 200 x 768 -> 512 4.6 / 4.8; at 1152 to 1536 values level).  Nine k steps, of which one
//         wavefront has two: not three workgroups on a CU (four column tiles / one: 829 x 576 -> 104, 728 tiles, 3.79 / 4.00, 66 x 576 -> 1280 3.80 / 3.99; on two 60 x 576 -> 1024 3.38 / 3.32)
//   two column tiles  up to 256 tiles and 4096 values 254 x 2304 -> 240 7.0 / 5.7, 124 x 2816 -> 496 7.0 / 6.3, 120 x 3072 -> 512 7.2 / 6.5, 144 x 3584 -> 432 7.8 / 7.2, 51 x
//         4096 -> 840 7.75 / 7.7; beyond: 67 x 2816 -> 1048 (297) 8.1 / 8.9, 32 x 5120 -> 1280 8.3 / 8.7; up to 512 short rows 223 x 256 -> 520 3.8 / 3.65 (four column tiles / two)
//   others  128 x 1024 -> 1024 6.6 / 5.5 (4 tiles), 256 x 1024 -> 1024 6.9 / 6.9 (16 rows, 4)
//   2:4   to 2048 values up to 1024 tiles 117 x 1024 -> 2064 6.95 / 5.6, 165 x 1280 -> 1504 7.9 / 6.5, 174 x 1536 -> 1000 7.6 / 6.2, 318 x 1792 -> 776 8.3 / 7.5, 258 x 2048 -> 976 10.2 / 7.6;
//         but 256 values and more than 768 tiles are the band kernel's where it takes them, unless the columns are whole 128s, which it reads slower (it / this:
//         480 -> 520 4.41 / 4.75, 241 -> 936 4.50 / 4.71; 60 -> 4096 4.94 / 4.68, 186 -> 1280 4.87 / 4.65); beyond: 109 x 768 -> 2992 (1316) 6.15 / 6.6, 251 x 1280 -> 1304 (1312) 7.9 / 8.5; to 3072 up to 512 290 x 2560 -> 352 9.1 / 6.7, 90 x 3072 -> 1304 9.0 / 7.4; beyond: 42 x 2304 -> 2984
//         (564) 8.2 / 8.8; else up to 256 31 x 5120 -> 1280 10.4 / 6.3, 48 x 4096 -> 1024 9.0 / 6.6; beyond: 119 x 3328 -> 680 (330) 9.1 / 11.4
//   Up to four short rows are quantised in no time, and two column tiles on more workgroups than CUs are ahead of four: 1 x 256 -> 8200 3.07 / 3.64 (two / four),
//         4 x 128 -> 10240 3.2 / 3.5, 1 x 512 -> 16384 3.83 / 3.98, 1 x 1024 -> 8200 4.46 / 4.75; but 8 x 256 -> 10240 3.8 / 3.6, 4 x 768 -> 12288 4.8 / 4.5.
// A call, launches included: 64 x 1024 -> 1024 9.8 / 6.4, 12 x 3072 -> 768 7.5 / 5.6, 2:4 48 x 5120 -> 1280 10.8 / 6.3, 16 x 4096 -> 1024 8.7 / 6.8.
// (A forced tile of the band kernel turns this form off.)
static int small_shape(int64_t M, int N, int K, bool sparse) {
  if (knob_or(KNOB_LINEAR_SMALL, 1) <= 0 || knob_or(KNOB_LINEAR_BAND, 1) > 1 || K % 64 != 0 || N % 8 != 0 || N <= 0 || K <= 0 || K > 5120 || M <= 0 || M > 4096) return 0;
  const int64_t eights = (M + 7) / 8;
  if (sparse) {
    const int64_t tiles = eights * ((N + 31) / 32);
    if (K <= 256 && tiles > 768 && N % 128 != 0 && linear_i8_band_covers(M, N, K, true)) return 0;
    return K % 128 == 0 && K >= 256 && tiles <= (K <= 2048 ? 1024 : K <= 3072 ? 512 : 256) ? 8 + 1 : 0;
  }
  auto tiles = [&](int nt) { return eights * ((N + 16 * nt - 1) / (16 * nt)); };
  if (tiles(1) <= 256) return 8 + 1;
  if (M <= 8 || K <= 4096) {
    if (tiles(2) <= 256) return 8 + 2;
    if (M <= 4 && (K <= 512 || tiles(2) <= 288)) return 8 + 2;
    if (M > 8 && K <= 1024 && tiles(1) <= (K == 576 ? 512 : 768)) return 8 + 1;
    if (M > 8 && K <= 512 && tiles(2) <= 512) return 8 + 2;
    if (K <= 1536 && tiles(4) <= 256) return 8 + 4;
    if (M <= 8) return 8 + 2;
  }
  if (K <= 1536 && ((M + 15) / 16) * ((N + 63) / 64) <= 256) return 16 + 4;
  if (K <= 768 && tiles(4) <= 512) return 8 + 4;
  return linear_i8_small_any_alignment(M, K) ? (K <= 1536 ? 16 + 4 : 8 + 2) : 0;
}

bool linear_i8_small_covers(int64_t M, int N, int K, bool sparse) { return small_shape(M, N, K, sparse) != 0; }

template <typename Kernel>
static int launch_small(Kernel kernel, SmallArgs a, int rows, int cols, int lds, hipStream_t stream) {
  a.tiles_m = (a.M + rows - 1) / rows;
  a.tiles = a.tiles_m * ((a.N + cols - 1) / cols);
  hipLaunchKernelGGL(kernel, dim3((unsigned int)((a.tiles + 7) / 8 * 8)), dim3(64 * kSmallWaves), (size_t)lds, stream, a);
  return check_launch("linear_i8_small_kernel");
}

template <int NCH>
static int launch_shape(const SmallArgs& a, int shape, hipStream_t stream) {
  auto lds = [&](int scales, int rows, int sums) { return scales + max(rows * (a.K + 16), sums); };
  if (a.widx) {
    if (shape == 8 + 1) return launch_small(linear_i8_sp24_small_kernel<NCH>, a, 8, 32, lds(64, 8, kSmallWaves * 1024), stream);
  } else {
    if (shape == 8 + 1) return launch_small(linear_i8_small_kernel<NCH, 1, 1>, a, 8, 16, lds(64, 16, kSmallWaves * 1024), stream);
    if (shape == 8 + 2) return launch_small(linear_i8_small_kernel<NCH, 1, 2>, a, 8, 32, lds(64, 16, kSmallWaves * 2048), stream);
    if constexpr (NCH <= 3) {
      if (shape == 8 + 4) return launch_small(linear_i8_small_kernel<NCH, 1, 4>, a, 8, 64, lds(64, 16, kSmallWaves * 4096), stream);
      if (shape == 16 + 4) return launch_small(linear_i8_small_kernel<NCH, 2, 4>, a, 16, 64, lds(64, 16, kSmallWaves * 4096), stream);
    }
  }
  set_error("linear_i8_small: %d rows of %d values are not covered", a.M, a.K);
  return SAMFAST_E_UNSUPPORTED;
}

int linear_i8_small_launch(const unsigned short* x, int64_t ldx, const int8_t* w, const int32_t* widx, const float* sw, const float* bias,
                           unsigned short* y, int64_t ldy, int M, int N, int K, int layout, hipStream_t stream) {
  SmallArgs a = {};
  a.x = x; a.ldx = ldx; a.w = w; a.widx = widx; a.sw = sw; a.bias = bias; a.y = y; a.ldy = ldy; a.M = M; a.N = N; a.K = K;
  const bool kb = layout == SAMFAST_LAYOUT_KB64;
  a.w_pitch = kb ? 64 : K;
  a.w_kstep = kb ? (int64_t)N * 64 : 64;
  const int shape = small_shape(M, N, K, widx != nullptr);
  if (K <= 512) return launch_shape<1>(a, shape, stream);
  if (K <= 1024) return launch_shape<2>(a, shape, stream);
  if (K <= 1536) return launch_shape<3>(a, shape, stream);
  if (K <= 2048) return launch_shape<4>(a, shape, stream);
  if (K <= 3072) return launch_shape<6>(a, shape, stream);
  if (K <= 4096) return launch_shape<8>(a, shape, stream);
  return launch_shape<10>(a, shape, stream);
}

// The smallest tile whose tiles still fit the GPU's CUs once: a smaller tile means a shorter chain, a second
// round costs more than that gains.  Measured on K-block major codes, us, against the tiled kernels:
// 128 x 3840 x 1280 in 64 x 32 tiles 4.7 (6.3), 64 x 1280 x 5120 in 16 x 32 5.6 (14.6).  From 2304 values on 64 x 32 tiles are slower than
// 64 x 64 ones whose operands come through LDS (gemm_i8_once.hip; 278 x 1280 x 3072 8.3 / 7.6, 0.96 times as long over 70 shapes, below 2240 1.04 to 1.07), and
// 64 x 64 tiles straight into registers were at any length (512 x 1280 x 3072 10.6 / 8.4).  `w_splits_lines`: K-block-major codes beside row-major weights of an
// odd multiple of 64 bytes, whose pieces of 64 bytes share cache lines with their neighbours: there 64 x 32 tiles stay ahead, each wavefront reading
// its own part of a row (a Linear, 64 x 64 through LDS / 64 x 32, us: 39 x 3776 -> 5120 10.4 / 9.65, 194 x 3648 -> 1600 11.6 / 10.9, 331 x 5056 -> 1280 15.2 / 14.5; 1.03 times as long over
// 170 shapes, over 360 of whole lines 0.89; with row-major codes as well 0.83, with both K-block major 0.94).
// Returns 16-row tiles * 8 + 16-column tiles, 0 = none.
static int skinny_shape(int M, int N, int K, bool w_splits_lines) {
  auto fits = [&](int mt, int nt) { return (int64_t)((M + 16 * mt - 1) / (16 * mt)) * ((N + 16 * nt - 1) / (16 * nt)) <= 256; };
  if (fits(1, 1)) return 1 * 8 + 1;
  if (fits(1, 2)) return 1 * 8 + 2;
  if (fits(2, 2)) return 2 * 8 + 2;
  if ((K < 2304 || w_splits_lines) && fits(4, 2)) return 4 * 8 + 2;
  return 0;
}
static int skinny_shape(const GemmArgs& a) { return skinny_shape(a.M, a.N, a.K, a.x_pitch == GBK && a.w_pitch != GBK && a.K % 128 != 0); }

bool gemm_i8_skinny_covers(const GemmArgs& a) {
  return knob_or(KNOB_GEMM_SKINNY, 1) > 0 && skinny_shape(a) != 0;
}

template <int MT, int NT>
static int launch_skinny(SmallArgs a, hipStream_t stream) {
  a.tiles_m = (a.M + 16 * MT - 1) / (16 * MT);
  a.tiles = a.tiles_m * ((a.N + 16 * NT - 1) / (16 * NT));
  const unsigned int grid = (unsigned int)((a.tiles + 7) / 8 * 8);
  hipLaunchKernelGGL((gemm_i8_skinny_kernel<MT, NT>), dim3(grid), dim3(64 * kSmallWaves), kSmallWaves * MT * NT * 1024, stream, a);
  return check_launch("gemm_i8_skinny_kernel");
}

int gemm_i8_skinny_launch(const GemmArgs& g, hipStream_t stream) {
  SmallArgs a = {};
  a.xq = g.x; a.sx = g.sx; a.w = g.w; a.sw = g.sw; a.bias = g.bias;
  a.y = reinterpret_cast<unsigned short*>(g.out);
  a.ldy = g.ldo; a.M = g.M; a.N = g.N; a.K = g.K;
  a.x_pitch = g.x_pitch; a.w_pitch = g.w_pitch; a.x_kstep = g.x_kstep; a.w_kstep = g.w_kstep;
  switch (skinny_shape(g)) {
    case 1 * 8 + 1: return launch_skinny<1, 1>(a, stream);
    case 1 * 8 + 2: return launch_skinny<1, 2>(a, stream);
    case 2 * 8 + 2: return launch_skinny<2, 2>(a, stream);
    default: return launch_skinny<4, 2>(a, stream);
  }
}

}  // namespace samfast

extern "C" int samfast_bench_gemm_i8_few_rows(int64_t M, int N, int K, int x_layout, int w_layout) {
  using namespace samfast;
  SF_REQUIRE(M > 0 && M < (1ll << 31) && N > 0 && K > 0, "bench_gemm_i8_few_rows: bad shape M=%lld N=%d K=%d", (long long)M, N, K);
  GemmArgs g = {};
  g.M = (int)M; g.N = N; g.K = K;
  g.x_pitch = x_layout == SAMFAST_LAYOUT_KB64 ? GBK : K;
  g.w_pitch = w_layout == SAMFAST_LAYOUT_KB64 ? GBK : K;
  const int s = gemm_i8_skinny_covers(g) ? skinny_shape(g) : 0;
  return 16 * (s / 8) * 1000 + 16 * (s % 8);
}

extern "C" int samfast_bench_linear_i8_few_rows(int64_t M, int N, int K, int layout) {
  using namespace samfast;
  SF_REQUIRE(M > 0 && N > 0 && K > 0 && layout >= SAMFAST_LAYOUT_ROWMAJOR && layout <= SAMFAST_LAYOUT_SPARSE24,
             "bench_linear_i8_few_rows: bad shape M=%lld N=%d K=%d or layout %d", (long long)M, N, K, layout);
  const bool sparse = layout == SAMFAST_LAYOUT_SPARSE24;
  const int s = small_shape(M, N, K, sparse);
  return s / 8 * 8 * 1000 + s % 8 * (sparse ? 32 : 16);
}
