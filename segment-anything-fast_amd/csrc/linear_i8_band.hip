// A whole quantised Linear, 2:4 ones too, over a band of rows and a range of columns per workgroup: row quantiser, int8 product and the scale +
// bias epilogue in one launch, for the row counts between linear_i8_small.hip's and those whose products fill the GPU in rounds.
//
// Two launches of such a call are mostly starts and ends (4096 x 768 -> 3072: 5 and 15 us for 4.5 us of matrix pipe), the codes go through
// memory between them, and the host pays for both.  Here every workgroup quantises its 32 or 64 rows itself - once per range of columns,
// at the encoders' widths 2 to 14 times in all, at N = 32000 up to 84, which is why ranges are wide, at 64 rows 640 or 768 columns, and why sixteen
// lanes take a row (one reduction and one division serve four rows) - keeps the codes in LDS for the whole of K and runs on W alone: a ring per wavefront in LDS, a
// 16-column x 128-byte fragment at a time, whole lines of row-major weights as well as of K-block-major ones.  Wavefronts meet in front of the
// products and never again: the row scales are in registers by then, so that one that is through converts and stores under the others'
// products (with the scales fetched behind a barrier at the end 28900 cycles instead of 26500).  Bound (4096 x 768 -> 3072, cycles of a workgroup's
// 26500, by a cycle counter in probes that are not kept, with four instructions per code; with one, quant_row.hpp, 0.7 us less): rows and first W through the load path
// 4000, codes 6000 of vector work, products 12700 (9200 of matrix pipe), output 3700; little of it overlaps, 160 KB of LDS being one workgroup per CU.
// us on the GPU, two launches / this one: 4096 x 768 -> 3072 21.9 / 17.6, 4096 x 768 -> 768 12.2 / 8.7, 2048 x 768 -> 3072 15.6 / 12.2, 16384 x 768 -> 768 26.9 / 19.5, 1024 x 1024
// -> 3072 12.8 / 9.3, 512 x 1280 -> 5120 12.3 / 9.9.  Integer sums and the epilogue's arithmetic are those of the other forms: the same bits.
#include "attn_relpos_shared.hpp"
#include "gemm_i8_shared.hpp"
#include "linear_i8_small.hpp"
#include "quant_row.hpp"

// every fp32 step below is rounded on its own (no fused multiply-add), as in the other forms
#pragma clang fp contract(off)

namespace samfast {

typedef int i32x8 __attribute__((ext_vector_type(8)));

struct BandArgs {
  const unsigned short* x;
  int64_t ldx;
  const int8_t* w;
  const int32_t* widx;  // 2:4 weights: `w` holds (K/64, N, 32) bytes, this (K/64, N, 2) words
  const float* sw;
  const float* bias;
  unsigned short* y;
  int64_t ldy;
  int M, N, K;
  int tiles_m, tiles_n, tiles;
  int group_m;  // row tiles per scheduling group
  unsigned int w_pitch, w_kstep;  // bytes between weight rows / between 64-byte k steps: K and 64, or 64 and 64 N (K-block major)
};

// at most n vector memory operations of this wavefront outstanding (n constant at every use)
SF_DEVICE void band_wait(int n) {
  switch (n) {
#define SF_CASE(H) case H: __builtin_amdgcn_s_waitcnt(0x0F70 | (H)); break
    SF_CASE(0); SF_CASE(1); SF_CASE(2); SF_CASE(3); SF_CASE(4); SF_CASE(5); SF_CASE(6); SF_CASE(7);
    SF_CASE(8); SF_CASE(9); SF_CASE(10); SF_CASE(11); SF_CASE(12); SF_CASE(13); SF_CASE(14); SF_CASE(15);
#undef SF_CASE
  }
  __builtin_amdgcn_sched_barrier(0);
}

// KMAX: 128 * the chunks of 8 values a lane holds of a row; RF: fragments of 16 rows; NF: fragments of 16 columns of a wavefront;
// DEPTH: k steps of 128 in a wavefront's ring; SPARSE: packed 2:4 weights (gemm_i8_sparse24.hip), v_smfmac_i32_16x16x128_i8.  K % 128 == 0, 128 * DEPTH <= K <= KMAX, M >= 16 RF, N >= 128 NF.
template <int KMAX, int RF, int NF, int DEPTH, bool SPARSE>
__global__ __launch_bounds__(512, 2) void linear_i8_band_kernel(BandArgs a) {
  constexpr int R = 16 * RF, BN = 128 * NF, RPW = 2 * RF, NB = RPW / 4;  // rows, columns; rows of a wavefront, quantised four at a time
  constexpr int NCH = KMAX / 128;
  // a column fragment: 16 columns x 128 bytes; SPARSE: 16 x 64 and their index words.  Requested in two parts
  constexpr int PART = SPARSE ? 256 : 1024, SLOT = 1024 + PART, RING = NF * DEPTH * SLOT;
  constexpr int CODES = R * KMAX;
  static_assert(CODES + 8 * RING <= 160 * 1024, "LDS of a CU");
  static_assert(2 * (NF * DEPTH - 1) <= 15, "wait thresholds");
  constexpr bool ROOM = CODES + 8 * RING + R * 4 <= 160 * 1024;  // for the row scales beside codes and rings
  __shared__ __attribute__((aligned(16))) unsigned char lds[CODES + 8 * RING + (ROOM ? R * 4 : 0)];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lq = lane >> 4;
  const unsigned int pid = xcd_contiguous_id(blockIdx.x, (unsigned int)a.tiles);
  if (pid >= (unsigned int)a.tiles) return;  // uniform over the workgroup
  const unsigned int per_group = (unsigned int)(a.group_m * a.tiles_n);
  const unsigned int first_m = pid / per_group * a.group_m, in_group = pid % per_group;
  const unsigned int gsz = min((unsigned int)a.tiles_m - first_m, (unsigned int)a.group_m);
  // the last tiles are moved back inside (M >= R, N >= BN): rows and columns of two tiles get the same bits twice
  const int m0 = min((int)(first_m + in_group % gsz) * R, a.M - R);
  const int n0 = min((int)(in_group / gsz) * BN, a.N - BN) + wave * 16 * NF;
  const int steps = a.K / 128;

  // ---- the rows: sixteen lanes to a row, chunks lr, lr + 16, .. of eight values (past the row's end: its last ones once more) -----------
  u32x4 xw[NB][NCH];
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    const unsigned short* src = a.x + (int64_t)(m0 + wave * RPW + 4 * b + lq) * a.ldx + 8 * lr;
#pragma unroll
    for (int i = 0; i < NCH; ++i) xw[b][i] = *reinterpret_cast<const u32x4*>(src + 128 * min(i, steps - 1));
  }
  __builtin_amdgcn_sched_barrier(0);

  // (column scales and bias, needed last, stand between the rows and W: the compiler's waits for the rows, which do not count the
  // requests of W, then leave those in flight)
  f32x4 sw[NF], bias[NF];
  const float* bias_or_sw = a.bias ? a.bias : a.sw;  // (a load under a branch would make the compiler wait here)
#pragma unroll
  for (int j = 0; j < NF; ++j) {
    const int n = n0 + (NF % 2 == 1 && j == NF - 1 ? 16 * j + 4 * lq : 32 * (j / 2) + 8 * lq + 4 * (j & 1));
    sw[j] = *reinterpret_cast<const f32x4*>(a.sw + n);
    bias[j] = *reinterpret_cast<const f32x4*>(bias_or_sw + n);
  }
  __builtin_amdgcn_sched_barrier(0);

  // ---- W: row r of fragment j is 128 bytes at 128 r in its slot, 16-byte chunk c at position c ^ (r / 2 % 8).  Of a pair of fragments
  // row r is column 8 (r / 4) + 4 (j % 2) + r % 4, so that a lane ends with eight adjacent columns; of a last one alone column r ------------
  unsigned int w_off[NF][2];
#pragma unroll
  for (int j = 0; j < NF; ++j)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      // SPARSE: 64-k block by block, the 32 bytes of every row; then, sixteen lanes, the 8 bytes of indices of two rows each
      const int r = SPARSE ? (h == 0 ? (lane & 31) >> 1 : 2 * (lane & 7)) : 8 * h + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
      const int col = NF % 2 == 1 && j == NF - 1 ? 16 * j + r : 32 * (j / 2) + 8 * (r >> 2) + 4 * (j & 1) + (r & 3);
      if (!SPARSE) w_off[j][h] = (unsigned int)col * a.w_pitch + (unsigned int)(c >> 2) * a.w_kstep + (unsigned int)(c & 3) * 16u;
      else if (h == 0) w_off[j][h] = (unsigned int)((lane >> 5) * a.N + col) * 32u + (lane & 1) * 16u;
      else w_off[j][h] = (unsigned int)((lane >> 3 & 1) * a.N + col) * 8u;
    }
  unsigned char* ring = lds + CODES + wave * RING;
  const unsigned int ring_at = (unsigned int)(uintptr_t)((__attribute__((address_space(3))) unsigned char*)ring);
  const unsigned char* wbase = reinterpret_cast<const unsigned char*>(a.w) + (int64_t)n0 * (SPARSE ? 32 : a.w_pitch);
  const unsigned char* ibase = reinterpret_cast<const unsigned char*>(a.widx) + (int64_t)n0 * 8;
  const int64_t w_step = SPARSE ? (int64_t)a.N * 64 : 2 * (int64_t)a.w_kstep, i_step = (int64_t)a.N * 16;
  // part h of fragment j of k step k
  auto load_w = [&](int k, int j, int h, unsigned int slot) __attribute__((always_inline)) {
    if (!SPARSE || h == 0) lds_dma16(wbase + k * w_step, w_off[j][h], ring_at + slot + h * 1024);
    else if (lane < 16) lds_dma16(ibase + k * i_step, w_off[j][h], ring_at + slot + 1024);
  };
  // request i of the first DEPTH k steps' 2 NF DEPTH, between the rows' chunks
  auto first_w = [&](int i) __attribute__((always_inline)) { load_w(i / (2 * NF), i / 2 % NF, i % 2, i / 2 * SLOT); };

  // ---- codes: 128 bytes of every row to a block, chunks at the same positions as W's. -------------------------------------------------
  // Row scales: beside the rings, or, where LDS is full, in the place of each ring's last part, whose request then waits for them to be read
  auto scale_of = [&](int row) __attribute__((always_inline)) {
    return reinterpret_cast<float*>(ROOM ? lds + CODES + 8 * RING + row * 4 : lds + CODES + row / RPW * RING + RING - PART + row % RPW * 4);
  };
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    float f[NCH][8];
    float amax = 0.f;
#pragma unroll
    for (int i = 0; i < NCH; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        f[i][2 * e] = bf16_lo_to_f32(xw[b][i][e]);
        f[i][2 * e + 1] = bf16_hi_to_f32(xw[b][i][e]);
        amax = __builtin_elementwise_maximum(amax, __builtin_elementwise_maximum(fabsf(f[i][2 * e]), fabsf(f[i][2 * e + 1])));
      }
    // over the row's sixteen lanes; a NaN has the largest pattern
    auto row_max = [](float v) __attribute__((always_inline)) {
      auto larger = [](float p, float q) { return __uint_as_float(max(__float_as_uint(p), __float_as_uint(q))); };
      v = larger(v, dpp_f32<0xB1>(v));
      v = larger(v, dpp_f32<0x4E>(v));
      v = larger(v, dpp_f32<0x141>(v));
      return larger(v, dpp_f32<0x140>(v));
    };
    amax = row_max(fabsf(amax));
    const bool row_nan = __float_as_uint(amax) > 0x7f800000u;
    if (__any(row_nan)) {  // the maximum without them
      float m = 0.f;
#pragma unroll
      for (int i = 0; i < NCH; ++i)
#pragma unroll
        for (int e = 0; e < 8; ++e) m = fmaxf(m, fabsf(f[i][e]));
      amax = row_max(m);
    }
    const QuantScale q(amax);
    const int row = wave * RPW + 4 * b + lq;
    unsigned char* at = lds + row * 128 + (((lr >> 1) ^ ((row >> 1) & 7)) * 16) + (lr & 1) * 8;
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      constexpr int FIRST = 2 * NF * DEPTH, CHUNKS = NB * NCH;
#pragma unroll
      for (int w = FIRST * (b * NCH + i) / CHUNKS; w < FIRST * (b * NCH + i + 1) / CHUNKS; ++w)
        if (ROOM || w < FIRST - 1) first_w(w);
      if (i < steps) {  // uniform
        unsigned int c[2];
        quantize_chunk<8>(f[i], q, c);
        *reinterpret_cast<u32x2*>(at + i * (R * 128)) = u32x2{c[0], c[1]};
      }
    }
    if (lr == 0) *scale_of(row) = row_nan ? __uint_as_float(0x7fc00000u) : q.scale;
  }
  // LDS written by all is visible to all; W stays in flight (a __syncthreads would wait for it)
  auto meet = [] __device__ () __attribute__((always_inline)) {
    __builtin_amdgcn_s_waitcnt(0xC07F);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };
  meet();
  float sx[RF];
#pragma unroll
  for (int t = 0; t < RF; ++t) sx[t] = *scale_of(16 * t + lr);
  if constexpr (!ROOM) {
    meet();
    first_w(2 * NF * DEPTH - 1);
  }

  // ---- products: every wavefront runs on its own ring, a column fragment at a time -----------------------------------------------------
  i32x4 acc[RF][NF];
#pragma unroll
  for (int t = 0; t < RF; ++t)
#pragma unroll
    for (int j = 0; j < NF; ++j) acc[t][j] = i32x4{0, 0, 0, 0};
  // Of a 128-byte row of codes the two 16-byte chunks of the lane, of a fragment its bytes.  SPARSE: lane (i, q) holds the stored half q % 2 of
  // 64-k block q / 2 of weight row i, so that lane (j, Q) of the codes wants chunks 2 (Q % 2) + Q / 2 and four more (gemm_i8_sp24_turns.hip)
  int frag[2], wfrag[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    frag[h] = lr * 128 + (((4 * h + (SPARSE ? 2 * (lq & 1) + (lq >> 1) : lq)) ^ ((lr >> 1) & 7)) * 16);
    wfrag[h] = !SPARSE ? frag[h] : h == 0 ? (lq >> 1) * 512 + lr * 32 + (lq & 1) * 16 : 1024 + (lq >> 1) * 128 + lr * 8 + (lq & 1) * 4;
  }
  // k step k out of the slots at `slots`; LEFT: k steps behind it whose W has been requested
  auto step = [&](int k, unsigned int slots, auto left_c) __attribute__((always_inline)) {
    constexpr int LEFT = decltype(left_c)::value;
    constexpr bool REQUEST = LEFT == DEPTH;
    i32x4 xf[RF][2];
#pragma unroll
    for (int t = 0; t < RF; ++t)
#pragma unroll
      for (int h = 0; h < 2; ++h) xf[t][h] = *reinterpret_cast<const i32x4*>(lds + k * (R * 128) + t * 2048 + frag[h]);
#pragma unroll
    for (int j = 0; j < NF; ++j) {
      band_wait(REQUEST ? 2 * (NF * DEPTH - 1) : 2 * (NF * (LEFT + 1) - 1 - j));
      const unsigned char* f = ring + slots + j * SLOT;
      i32x4 wf[2];
      int index = 0;
      wf[0] = *reinterpret_cast<const i32x4*>(f + wfrag[0]);
      if (SPARSE) index = *reinterpret_cast<const int*>(f + wfrag[1]);
      else wf[1] = *reinterpret_cast<const i32x4*>(f + wfrag[1]);
      __builtin_amdgcn_s_waitcnt(0xC07F);  // the fragment is in registers: its slot is requested anew
      __builtin_amdgcn_sched_barrier(0);
      if (REQUEST) {
        load_w(k + DEPTH, j, 0, slots + j * SLOT);
        load_w(k + DEPTH, j, 1, slots + j * SLOT);
      }
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (SPARSE) {
#pragma unroll
        for (int t = 0; t < RF; ++t) {
          const i32x8 x8 = {xf[t][0][0], xf[t][0][1], xf[t][0][2], xf[t][0][3], xf[t][1][0], xf[t][1][1], xf[t][1][2], xf[t][1][3]};
          acc[t][j] = __builtin_amdgcn_smfmac_i32_16x16x128_i8(wf[0], x8, acc[t][j], index, 0, 0);
        }
      } else {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int t = 0; t < RF; ++t) acc[t][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wf[h], xf[t][h], acc[t][j], 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  unsigned int slots = 0;
  int k = 0;
  // Of a SIMD's two wavefronts one multiplies ahead of the other and converts and stores under its products: priorities 3 and 2 here, 0 behind (64-row
  // tiles, us, all alike / so: 4096 x 768 -> 3072 19.7 / 19.1, 4096 x 768 -> 2304 17.4 / 16.7, 4096 x 1280 -> 1280 18.2 / 17.7; with 32 rows nothing)
  if (RF == 4) {
    if (wave < 4) __builtin_amdgcn_s_setprio(3);
    else __builtin_amdgcn_s_setprio(2);
  }
  for (; k + DEPTH < steps; ++k) {
    step(k, slots, std::integral_constant<int, DEPTH>{});
    slots = DEPTH == 1 || slots == (DEPTH - 1) * NF * SLOT ? 0 : slots + NF * SLOT;
  }
  if (DEPTH == 2) {
    step(k++, slots, std::integral_constant<int, DEPTH - 1>{});
    slots = slots == 0 ? NF * SLOT : 0;
  }
  step(k, slots, std::integral_constant<int, 0>{});
  if (RF == 4) __builtin_amdgcn_s_setprio(0);

  // ---- (float(acc) * sx) * sw + bias; a wavefront that is through finishes under the others' products ------------------------------------
  if (!a.bias)  // uniform
#pragma unroll
    for (int j = 0; j < NF; ++j) bias[j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int64_t out_off = lr * a.ldy * 2;
  unsigned char* out = reinterpret_cast<unsigned char*>(a.y + (int64_t)m0 * a.ldy + n0);
#pragma unroll
  for (int t = 0; t < RF; ++t) {
    unsigned int o[NF][2];
#pragma unroll
    for (int j = 0; j < NF; ++j)
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        float v[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          // three separately rounded fp32 operations (no fused multiply-add)
          v[e] = (float)acc[t][j][2 * c + e] * sx[t];
          v[e] = v[e] * sw[j][2 * c + e];
          v[e] = v[e] + bias[j][2 * c + e];
        }
        o[j][c] = pack_bf16x2(v[0], v[1]);
      }
    unsigned char* to = out + (int64_t)(16 * t) * a.ldy * 2 + out_off;
#pragma unroll
    for (int j = 0; j + 1 < NF; j += 2) *reinterpret_cast<u32x4*>(to + 32 * j + 16 * lq) = u32x4{o[j][0], o[j][1], o[j + 1][0], o[j + 1][1]};
    if (NF % 2 == 1) *reinterpret_cast<u32x2*>(to + 32 * (NF - 1) + 8 * lq) = u32x2{o[NF - 1][0], o[NF - 1][1]};
  }
}

// Row fragments * 8 + column fragments of a wavefront in the tile; 0 = not this form.
// The smallest tile whose tiles fit the CUs once; a second round costs more than the smaller tile gains (4096 x 768 -> 2304: 32 x 384 tiles, three
// rounds, 20.7 us, 64 x 384, two, 19.6, 64 x 768 16.9), and beyond one round of the largest the two launches are ahead (6000 x 768 -> 2304 26.6 / 29.3,
// 2700 x 1024 -> 4096 27.2 / 34.5).  On longer rows the quantiser's share grows with the rows a workgroup has: 64 x 384 tiles only from about 180 of
// them on (us, two launches / one: 1024 x 1280 -> 3840, 160 tiles, 14.1 / 14.8, 1200 x 1280 -> 3840, 190, 17.2 / 15.2, 900 x 1024 -> 4096, 165, 13.0 / 12.5, a call 12.6 / 12.1), and
// behind 1280 values the small-tile product's rows stay with it (300 x 1280 -> 1280 8.0 / 8.4, 400, beyond them, 11.9 / 9.0).
// 2:4 weights: the two launches take longer (the quantiser is the same, the products are bound by what they load) and win nowhere below one round,
// but for the wide tiles below: us, two / one, 4096 x 768 -> 3072 20.5 / 16.2, 4096 x 768 -> 768 13.3 / 8.7, 1024 x 768 -> 3072 11.9 / 8.2, 1024 x 1024 -> 1024
// 11.6 / 7.8, 512 x 1280 -> 5120 13.9 / 10.3, 700 x 1280 -> 5120 14.9 / 13.8, 2048 x 1280 -> 5120 (256 tiles) 22.7 / 19.3.  (On rows of 1152 and 1280 and up to 24
// tiles of 32 x 384 the two are the shorter ones on the GPU by up to half a microsecond, and no shorter as calls: 48 x 1280 -> 3840 7.95 / 8.4, a call 8.75 / 8.5.)
// Wide tiles (us, two / one).  A workgroup takes as long however few there are, so that they pay from 181 of 64 x 768 on: 200 x 1024 -> 32000 (168) 17.8 / 19.0, 481 x
// 1024 -> 16384 (176) 1.06 times as long, 761 x 512 -> 10880 (180) 13.9 / 14.6, 2:4 1024 x 1024 -> 8192 (176) 16.6 / 18.1.  The more rows, the longer the quantiser that is
// saved: over more than 2048 at any number (2256 x 1024 -> 3072, 144, 0.96, 2:4 2980 x 512 -> 2048, 141, 0.92 times), over more than 1024 on rows up to 768 at any
// number (2:4: 152), up to 1024 from 156 on (1497 x 1024 -> 4096, 144, 19.1 / 20.0; 1933 x 896 -> 3584, 155, 18.5 / 19.2), 2:4 not (1540 x 1024 -> 4096, 150, 16.8 / 17.5);
// up to 3072 rows of 256 from 168 on (1451 x 256 -> 5120, 161, 11.3 / 11.9, 2616 x 256 -> 3072, 164, 11.8 / 12.3; 3490 x 256 -> 2048, 165, 0.98 times).
// 64 x 640 over more than 1024 rows at any number, else from 205 on (351 x 1280 -> 16384, 156, 1.06 times; 229 x 1280 -> 32000, 200, 1.03 times); 2:4 from 212
// on (492 x 1280 -> 16384, 208, 1.08 times), on rows up to 1152 sooner: over more than 2048 at any number, more than 1024 from 176 on (331 x 1152 -> 20680, 198, 15.7 / 17.2).
static bool wide_pays(int64_t M, int K, bool sparse, int64_t tiles) {
  if (tiles >= (K <= 1024 ? 181 : sparse ? 212 : 205)) return true;
  if (sparse && K > 1152) return false;
  if (!sparse && K <= 256 && M <= 3072) return M > 1024 && tiles >= 168;
  if (M > 2048) return true;
  if (M <= 1024) return false;
  if (K <= 768) return !sparse || tiles >= 152;
  if (K <= 1024) return !sparse && tiles >= 156;
  return !sparse || tiles >= 176;
}

static int band_shape(int64_t M, int N, int K, bool sparse) {
  const int mode = knob_or(KNOB_LINEAR_BAND, 1);
  if (mode <= 0 || knob_or(KNOB_LINEAR_SMALL, 1) <= 0 || K % 128 != 0 || K < 256 || K > 1280 || N % 8 != 0 || M < 32 || N < 384 || M > (1 << 20) || (int64_t)N * K >= (1ll << 31)) return 0;
  auto tiles = [&](int rf, int nf) { return (M + 16 * rf - 1) / (16 * rf) * ((N + 128 * nf - 1) / (128 * nf)); };
  auto fits = [&](int rf, int nf) { return M >= 16 * rf && N >= 128 * nf && tiles(rf, nf) <= 256; };
  const int wide = K <= 1024 ? 6 : 5;
  if (mode > 1) return (mode == 2 * 8 + 3 || mode == 4 * 8 + 3 || mode == 4 * 8 + wide) && M >= 16 * (mode / 8) && N >= 128 * (mode % 8) ? mode : 0;
  if (!sparse && K > 1024 && (M + 63) / 64 * ((N + 31) / 32) <= 256) return 0;
  if (fits(2, 3)) return 2 * 8 + 3;
  if (fits(4, 3)) return sparse || K <= 768 || tiles(4, 3) >= 176 ? 4 * 8 + 3 : 0;
  return fits(4, wide) && wide_pays(M, K, sparse, tiles(4, wide)) ? 4 * 8 + wide : 0;
}

bool linear_i8_band_covers(int64_t M, int N, int K, bool sparse) { return band_shape(M, N, K, sparse) != 0; }

template <int KMAX, int RF, int NF, int DEPTH>
static int launch_band(BandArgs a, hipStream_t stream) {
  a.tiles_n = (a.N + 128 * NF - 1) / (128 * NF);
  a.tiles_m = (a.M + 16 * RF - 1) / (16 * RF);
  a.tiles = a.tiles_m * a.tiles_n;
  // An XCD's eighth of the tiles is to be g row tiles by t / g column tiles with g * R rows of two bytes about as many bytes as the
  // columns' weights: what its L2 fetches is least there
  // (256 x 1280 -> 5120, whose 6.5 MB of weights every XCD would read otherwise, 12.8 -> 9.8 us).
  const int t = (a.tiles + 7) / 8;
  int g = 1;
  while (g < a.tiles_m && (g + 1) * (g + 1) * 2 * 16 * RF <= t * 128 * NF) ++g;
  a.group_m = g;
  const dim3 grid((unsigned int)((a.tiles + 7) / 8 * 8));
  if (a.widx) hipLaunchKernelGGL((linear_i8_band_kernel<KMAX, RF, NF, DEPTH, true>), grid, dim3(512), 0, stream, a);
  else hipLaunchKernelGGL((linear_i8_band_kernel<KMAX, RF, NF, DEPTH, false>), grid, dim3(512), 0, stream, a);
  return check_launch("linear_i8_band_kernel");
}

template <int KMAX>
static int launch_band_shape(const BandArgs& a, int shape, hipStream_t stream) {
  if (shape == 2 * 8 + 3) return launch_band<KMAX, 2, 3, 2>(a, stream);
  if constexpr (KMAX <= 1024) {
    if (shape == 4 * 8 + 3) return launch_band<KMAX, 4, 3, 2>(a, stream);
    if (shape == 4 * 8 + 6) return launch_band<KMAX, 4, 6, 1>(a, stream);
  } else {
    if (shape == 4 * 8 + 3) return launch_band<KMAX, 4, 3, 1>(a, stream);
    if (shape == 4 * 8 + 5) return launch_band<KMAX, 4, 5, 1>(a, stream);
  }
  set_error("linear_i8_band: %d x %d values to %d are not covered", a.M, a.K, a.N);
  return SAMFAST_E_UNSUPPORTED;
}

int linear_i8_band_launch(const unsigned short* x, int64_t ldx, const int8_t* w, const int32_t* widx, const float* sw, const float* bias, unsigned short* y,
                          int64_t ldy, int M, int N, int K, int layout, hipStream_t stream) {
  BandArgs a = {};
  a.x = x; a.ldx = ldx; a.w = w; a.widx = widx; a.sw = sw; a.bias = bias; a.y = y; a.ldy = ldy; a.M = M; a.N = N; a.K = K;
  const bool kb = layout == SAMFAST_LAYOUT_KB64;
  a.w_pitch = kb ? 64 : (unsigned int)K;
  a.w_kstep = kb ? (unsigned int)N * 64u : 64u;
  const int shape = band_shape(M, N, K, widx != nullptr);
  if (K <= 768) return launch_band_shape<768>(a, shape, stream);
  if (K <= 1024) return launch_band_shape<1024>(a, shape, stream);
  return launch_band_shape<1280>(a, shape, stream);
}

}  // namespace samfast
