// Global attention (64-wide key grid) with caller-computed bias factors.
//
// The mathematics of attn_global_kernel (attn_relpos.hip) - S^T = K Q^T by 32x32x16 MFMAs with rel_w as the initial
// accumulator, rel_h one scalar per (query, key row), base-2 softmax, O^T = V^T P^T on transposing LDS reads -
// on a loop that is pipelined inside a wavefront: between the exponentials of one half row of keys stand the
// matrix instructions of the next half row's scores and of the previous one's P V, and the LDS reads that feed
// them.  No running maximum is taken in the common case, LDS reads meet no bank twice (GridRow), and the
// workgroups of a head touch its K and V ahead, so that the rows come out of their XCD's L2.
//   Bound: at 8 x 16 x 4096 x 80 (fp16 738 us, 931 TFLOP/s, bf16 691; attn_global_kernel 803 and 763) first the instructions of the two pipes, then the power
//   limit: the same launch on zeros takes 600 us in bf16 and 620 in fp16, on values 707 and 749 (one machine; of the 42 between the types half is fp16's test of the packed pairs, half its values' power).  On the
//   256 workgroups of 1 x 8 heads, where a SIMD has one wavefront, zeros are 2 to 5 % ahead (54.9 / 56.1, 54.9 / 57.9).  At one image of 12 heads of 64 channels
//   (63.8 us against 82) the last, half-empty round and the prologue.
//   (The encoder, which hands over tables, keeps attn_global_kernel: its int8 Linears turn any other order of these
//   roundings into other codes.)
//
// Four kernels.  attn_global_bias16_kernel (hd 80, on the smaller matrix instruction): a wavefront owns 32 queries and walks whole key rows; workgroups of 8 (one
// per CU: every row staged once for 256 queries) or 4 wavefronts (two per CU).  attn_global_bias_kernel: the same at hd 64, on the larger
// instruction, where it is asked for.  attn_global_split16_kernel (hd 64, on the smaller matrix
// instruction): the keys of every row are split between two wavefronts, whose results (maximum reference, denominator, output) meet in
// LDS once, at the end; workgroups of two query tiles x two key halves (64 queries, under 54 KB of LDS), three per CU, so that one image's 12 heads are
// 768 workgroups: three on each of the 256 CUs, where 128-query workgroups leave half of the CUs with one and half with two.  attn_global_split_kernel:
// the same at hd 80, on the larger instruction, where it is asked for.  bias_form picks, by head_dim: the kernels round
// differently, and a slice's bits are not to depend on the batch.
#include "attn_relpos_shared.hpp"

namespace samfast {

constexpr float kCeiling = 256.0f;  // of a lane's share of a half row's sum (16 of 32 keys, on the smaller instruction 8): each probability stays far inside both types

template <int WAVES>
struct BiasCfg : GridRow<64> {
  using R = GridRow<64>;
  static constexpr int BM = 32 * WAVES;       // queries per workgroup
  static constexpr int KDPW = (R::KP + WAVES - 1) / WAVES, VDPW = (R::VP + WAVES - 1) / WAVES;  // wave instructions per tile a wave issues at most
  // LDS: two K tiles, three V tiles (a row's V is still read while the next row's has to be there), rel_h
  static constexpr int V_OFF = 2 * R::KTILE;
  static constexpr int RH = 32;               // key rows whose rel_h is at hand
  static constexpr int RELH_OFF = V_OFF + 3 * R::VTILE;
  static constexpr int LDS_BYTES = RELH_OFF + RH * BM * 4;
  static_assert(LDS_BYTES <= (WAVES == 4 ? 80 : 160) * 1024, "workgroups per CU");
};

template <typename T, int WAVES>
__global__ __launch_bounds__(64 * WAVES, 2) void attn_global_bias_kernel(AttnArgs a) {
  using C = BiasCfg<WAVES>;
  constexpr int HD = 64;
  __shared__ __attribute__((aligned(16))) unsigned char lds[C::LDS_BYTES];
  float* relhT = reinterpret_cast<float*>(lds + C::RELH_OFF);  // [kh % RH][BM], * log2(e); a wave reads only its own columns

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 31, lh = lane >> 5;

  const unsigned int nqb = a.N / C::BM;
  const unsigned int total = (unsigned int)(a.B * a.nH) * nqb;
  const unsigned int pid = xcd_contiguous_id(blockIdx.x, total);
  if (pid >= total) return;
  const int bh = pid / nqb, qb = pid % nqb;
  const int b = bh / a.nH, h = bh % a.nH;
  const int q0 = qb * C::BM + 32 * wave;  // the wavefront's first query: half of one grid row

  const unsigned short* kbase = a.k + b * a.k_sb + h * a.k_sh;
  const unsigned short* vbase = a.v + b * a.v_sb + h * a.v_sh;

  // ---- K / V rows: global memory -> LDS directly, wave instruction i of a tile fills pieces 64 i .. 64 i + 63 ----
  unsigned int koff[C::KDPW], voff[C::VDPW];  // bytes, from the tile's first key row; unsigned: scalar-base load form
#pragma unroll
  for (int m = 0; m < C::KDPW; ++m) {
    int row;
    const int at = C::k_source(64 * (wave + WAVES * m) + lane, row);
    koff[m] = (unsigned int)(row * (int)a.k_sn) * 2u + at;
  }
#pragma unroll
  for (int m = 0; m < C::VDPW; ++m) {
    int row;
    const int at = C::v_source(64 * (wave + WAVES * m) + lane, row);
    voff[m] = (unsigned int)(row * (int)a.v_sn) * 2u + at;
  }
  const unsigned int lds_base = (unsigned int)(uintptr_t)((__attribute__((address_space(3))) unsigned char*)lds);
  auto k_dma = [&](int kt, int buf) __attribute__((always_inline)) {
    const unsigned char* src = reinterpret_cast<const unsigned char*>(kbase + (int64_t)kt * 64 * a.k_sn);
#pragma unroll
    for (int m = 0; m < C::KDPW; ++m)
      if (wave + WAVES * m < C::KP) lds_dma16(src, koff[m], lds_base + buf * C::KTILE + (wave + WAVES * m) * 1024);
  };
  auto v_dma = [&](int kt, unsigned int buf_off) __attribute__((always_inline)) {
    const unsigned char* src = reinterpret_cast<const unsigned char*>(vbase + (int64_t)kt * 64 * a.v_sn);
#pragma unroll
    for (int m = 0; m < C::VDPW; ++m)
      if (wave + WAVES * m < C::VP) lds_dma16(src, voff[m], lds_base + C::V_OFF + buf_off + (wave + WAVES * m) * 1024);
  };
  k_dma(0, 0);
  v_dma(0, 0);
  k_dma(1, 1);  // N % 128 == 0: at least two key rows
  v_dma(1, C::VTILE);

  // ---- Q^T operand: query lr, channels 16s + 8lh .. +7 ----
  u32x4 qf[C::KS];
  {
    const unsigned short* qp = a.q + b * a.q_sb + h * a.q_sh + (int64_t)(q0 + lr) * a.q_sn + 8 * lh;
#pragma unroll
    for (int s = 0; s < C::KS; ++s) qf[s] = load_x8_global(qp + 16 * s);
  }
  // The workgroups of a head walk its key rows in step, so every row would be waited for at the latency of
  // the Infinity Cache or HBM.  Each of them touches its own share of the head's K and V first: together
  // they have the head in their XCD's L2 by the time they get to it.
  constexpr int NTOUCH = 2 * C::BM * (HD / 8) / (64 * WAVES);
  unsigned int touched[NTOUCH];
#pragma unroll
  for (int i = 0; i < NTOUCH; ++i) {
    const int P = (tid + 64 * WAVES * i) % (C::BM * (HD / 8)), row = P / (HD / 8), col = P % (HD / 8);
    const bool is_v = 2 * i >= NTOUCH;
    touched[i] = *reinterpret_cast<const unsigned int*>((is_v ? vbase : kbase) + (int64_t)(qb * C::BM + row) * (is_v ? a.v_sn : a.k_sn) + col * 8);
  }

  // V^T operand of the P V product through transposing LDS reads (ds_read_b64_tr_b16): in
  // each group of 16 lanes, lane l receives as element j the l%4-th 16-bit value of the 8
  // bytes addressed by lane 4j + l/4 of the group.  Source lane 4j + i therefore points at
  // key j of the lane half's four keys, channels 4i .. 4i+3 of the group's 16 channels, and
  // lane l ends up with channel l of four consecutive keys: the MFMA A operand.
  int vrd[C::DT], krd[C::KS];
#pragma unroll
  for (int dt = 0; dt < C::DT; ++dt) vrd[dt] = C::V_OFF + C::v_read(lane, dt);
#pragma unroll
  for (int ks = 0; ks < C::KS; ++ks) krd[ks] = C::k_read(lr, lh, ks);

  // ---- bias: rel_w / sm_scale of the lane's query is the initial accumulator of the score tiles of the two
  //      half rows; rel_h * log2(e) stands in LDS, 32 key rows at a time ----
  auto fill_relh = [&](int kh0) __attribute__((always_inline)) {
    // lane: query lr, key rows kh0 + 16 lh .. +15
    const unsigned short* src = a.rh + b * a.rh_sb + h * a.rh_sh + (int64_t)(q0 + lr) * a.rh_sn + kh0 + 16 * lh;
    unsigned short v[16];
    if (a.relh_x8) {
      *reinterpret_cast<u32x4*>(v) = load_x8_global(src);
      *reinterpret_cast<u32x4*>(v + 8) = load_x8_global(src + 8);
    } else {
#pragma unroll
      for (int e = 0; e < 16; ++e) v[e] = kh0 + 16 * lh + e < a.gh ? src[e] : (unsigned short)0;
    }
#pragma unroll
    for (int e = 0; e < 16; ++e) relhT[(16 * lh + e) * C::BM + 32 * wave + lr] = T::from_bits(v[e]) * kLog2e;
  };
  f32x16 b1[2];
  fill_relh(0);
  {
    const unsigned short* rwp = a.rw + b * a.rw_sb + h * a.rw_sh + (int64_t)(q0 + lr) * a.rw_sn + 4 * lh;
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const u32x2 w = *reinterpret_cast<const u32x2*>(rwp + 32 * half + 8 * j);
        b1[half][4 * j + 0] = T::lo(w[0]) * a.inv_scale;
        b1[half][4 * j + 1] = T::hi(w[0]) * a.inv_scale;
        b1[half][4 * j + 2] = T::lo(w[1]) * a.inv_scale;
        b1[half][4 * j + 3] = T::hi(w[1]) * a.inv_scale;
      }
  }
#pragma unroll
  for (int i = 0; i < NTOUCH; ++i) asm volatile("" : : "v"(touched[i]));
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's share of the first two rows has landed
  __syncthreads();

  // ---- main loop over half rows of 32 keys ----
  f32x16 oacc[C::DT];
#pragma unroll
  for (int dt = 0; dt < C::DT; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) oacc[dt][r] = 0.f;
  float m_i = T::kLowest, l_i = 0.f;
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) s16x4* trptr_t;

  // The loop is pipelined inside a wavefront, instruction by instruction: between the exponentials of half row
  // i stand the matrix instructions of the scores of half row i + 1 and of P V of half row i - 1, and the
  // LDS reads that feed them, so that none of the three pipes waits for another's burst.
  u32x4 kf[C::KS], vf[2][C::DT], pkA[2], pkB[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    pkA[j] = pkB[j] = u32x4{0u, 0u, 0u, 0u};
#pragma unroll
    for (int dt = 0; dt < C::DT; ++dt) vf[j][dt] = u32x4{0u, 0u, 0u, 0u};
  }
  auto read_v = [&](int j, int dt, unsigned int v_off) __attribute__((always_inline)) {
    const unsigned char* p = lds + v_off + vrd[dt] + 16 * j * (C::VP * 16);
    const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((trptr_t)p));
    const u32x2 hi = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((trptr_t)(p + 8 * C::VP * 16)));
    vf[j][dt] = u32x4{lo[0], lo[1], hi[0], hi[1]};
  };
  // s, pk: scores and probabilities of this half row, its V at v_off, rel_h of its row b0; s_next: scores of the
  // next one, from K at k_off with the initial accumulator b_next; pk_prev, v_prev: the one before
  auto half_row = [&](f32x16& s, f32x16& s_next, u32x4 (&pk)[2], u32x4 (&pk_prev)[2], const f32x16& b_next, int k_off, unsigned int v_off,
                      unsigned int v_prev, float b0, bool has_prev) __attribute__((always_inline)) {
#pragma unroll
    for (int ks = 0; ks < C::KS; ++ks) kf[ks] = *reinterpret_cast<const u32x4*>(lds + krd[ks] + k_off);
    if (has_prev) {  // (before the first half row: the zeros above, with probabilities of zero)
#pragma unroll
      for (int dt = 0; dt < C::DT; ++dt) read_v(1, dt, v_prev);
    }
    __builtin_amdgcn_sched_barrier(0);

    // online softmax, one query per lane.  The exponent offset m_i is a reference, not the running
    // maximum (the final division by the denominator, accumulated with the same offsets, makes the
    // result independent of it): probabilities may sit anywhere below a ceiling, so no maximum of the scores is
    // taken in the common case.  Whether one has grown too large shows in the half row's sum (in the kernels whose denominators are
    // products, in the packed pairs: T::note, T::outgrown).  Then - always where the first keys are met, m_i being T::kLowest - the maximum is found, the accumulators are
    // rescaled and the probabilities formed once more.  m_i is finite throughout: keys that a factor of -inf, or of
    // the type's lowest value, has taken away have probabilities of zero whatever stands before or behind them.
    float l0 = 0.f, l1 = 0.f;  // this half row's share of the denominator, unrounded (two chains)
    auto pair = [&](int w, float neg_mrow) __attribute__((always_inline)) {  // packed pair w of 8
      const float p0 = fast_exp2(fmaf(s[2 * w], a.c, neg_mrow)), p1 = fast_exp2(fmaf(s[2 * w + 1], a.c, neg_mrow));
      pk[w >> 2][w & 3] = T::pack2(p0, p1);
      l0 += p0 + p1;
    };
    auto score = [&](int ks) __attribute__((always_inline)) { s_next = T::mfma(kf[ks], qf[ks], ks == 0 ? b_next : s_next); };
    auto pv = [&](int j, int dt) __attribute__((always_inline)) { oacc[dt] = T::mfma(vf[j][dt], pk_prev[j], oacc[dt]); };
    const float neg_mrow = b0 - m_i;
    float e0, e1;  // a pair is packed one step after its exponentials were issued
#pragma unroll
    for (int g = 0; g < 8; ++g) {
      const float x0 = fmaf(s[2 * g], a.c, neg_mrow), x1 = fmaf(s[2 * g + 1], a.c, neg_mrow);
      if (g > 0) {
        pk[(g - 1) >> 2][(g - 1) & 3] = T::pack2(e0, e1);
        l0 += e0, l1 += e1;
      }
      e0 = fast_exp2(x0);
      e1 = fast_exp2(x1);
      __builtin_amdgcn_sched_barrier(0);
      if (g == 0) pv(0, 0);
      if (g == 1) {
#pragma unroll
        for (int dt = 1; dt < C::DT; ++dt) pv(0, dt);
      }
      if (g >= 2 && g < 2 + C::KS) score(g - 2);
      if (g >= 2 && g < 2 + C::DT) read_v(0, g - 2, v_off);
      if (g == 6) pv(1, 0);
      if (g == 7) {
#pragma unroll
        for (int dt = 1; dt < C::DT; ++dt) pv(1, dt);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    pk[1][3] = T::pack2(e0, e1);
    l0 = (l0 + e0) + (l1 + e1);
    if (__any(l0 > kCeiling)) {  // uniform; an infinity included
      float mx = s[0];
#pragma unroll
      for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[r]);
      mx = max_with_lane_xor32(mx);
      const float m_new = fmaxf(m_i, fmaf(mx, a.c, b0 + T::kMargin));
      const float alpha = fast_exp2(m_i - m_new);  // first keys: 0; none yet: 1, on accumulators of zero
      m_i = m_new;
      l_i *= alpha;
      l0 = 0.f;
#pragma unroll
      for (int dt = 0; dt < C::DT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[dt][r] *= alpha;
#pragma unroll
      for (int w = 0; w < 8; ++w) pair(w, b0 - m_i);
    }
    l_i += l0;
  };

  const int nkt = a.N / 64;
  // V tiles rotate: row kt's, and the one row kt + 2 goes to (row kt - 1's)
  unsigned int v_cur = 0, v_free = 2 * C::VTILE;
  constexpr unsigned int VHALF = 32 * C::VP * 16;
  f32x16 sA, sB;
#pragma unroll
  for (int ks = 0; ks < C::KS; ++ks) sA = T::mfma(*reinterpret_cast<const u32x4*>(lds + krd[ks]), qf[ks], ks == 0 ? b1[0] : sA);
  auto key_row = [&](int kt, auto buf_c) __attribute__((always_inline)) {
    constexpr int BUF = decltype(buf_c)::value;  // kt & 1, for constant LDS offsets
    if (kt == C::RH) {  // the wavefront's own columns: no barrier
      fill_relh(kt);
    }
    const float b0 = relhT[(kt % C::RH) * C::BM + 32 * wave + lr];
    half_row(sA, sB, pkA, pkB, b1[1], BUF * C::KTILE + 32 * (C::KP * 16), v_cur, v_free + VHALF, b0, kt > 0);
    // row kt + 1 has landed (own share) and everybody has left K row kt and V row kt - 1: refill them
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (kt + 2 < nkt) {
      k_dma(kt + 2, BUF);
      v_dma(kt + 2, v_free);
    }
    // (after the last row kf is whatever the buffer holds: that product is not used)
    half_row(sB, sA, pkB, pkA, b1[0], (BUF ^ 1) * C::KTILE, v_cur + VHALF, v_cur, b0, true);
    v_free = v_cur;
    v_cur = v_cur == 2 * C::VTILE ? 0 : v_cur + C::VTILE;
  };
  for (int kt = 0; kt < nkt; kt += 2) {  // nkt is even
    key_row(kt, std::integral_constant<int, 0>{});
    key_row(kt + 1, std::integral_constant<int, 1>{});
  }
  // P V of the last half row
#pragma unroll
  for (int dt = 0; dt < C::DT; ++dt) read_v(1, dt, v_free + VHALF);
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int dt = 0; dt < C::DT; ++dt) oacc[dt] = T::mfma(vf[j][dt], pkB[j], oacc[dt]);

  // ---- epilogue: O = acc / l, 4 adjacent channels per store ----
  const float inv = 1.0f / (l_i + xor32(l_i));
  unsigned short* op = a.out + b * a.o_sb + h * a.o_sh + (int64_t)(q0 + lr) * a.o_sn;
#pragma unroll
  for (int dt = 0; dt < C::DT; ++dt)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const u32x2 o = {T::pack2(oacc[dt][4 * j] * inv, oacc[dt][4 * j + 1] * inv),
                       T::pack2(oacc[dt][4 * j + 2] * inv, oacc[dt][4 * j + 3] * inv)};
      *reinterpret_cast<u32x2*>(op + 32 * dt + 8 * j + 4 * lh) = o;
    }
}

// Split keys at hd 80 (SAMFAST_ATTN_SPLIT=2; hd 64 has a form of its own below).
struct SplitCfg : GridRow<80> {
  using R = GridRow<80>;
  static constexpr int QW = 2;                  // query tiles of 32 per workgroup
  static constexpr int WAVES = 2 * QW;
  static constexpr int BM = 32 * QW;
  static constexpr int KDPW = (R::KP + WAVES - 1) / WAVES, VDPW = (R::VP + WAVES - 1) / WAVES;
  static constexpr int V_OFF = 2 * R::KTILE;    // LDS: K tiles of both stages, V tiles of both stages, rel_h
  static constexpr int RELH_OFF = V_OFF + 2 * R::VTILE;
  static constexpr int RH = 32;                 // key rows whose rel_h is at hand
  static constexpr int LDS_BYTES = RELH_OFF + RH * BM * 4;
  static_assert(2 * LDS_BYTES <= 160 * 1024, "two workgroups per CU");
  static_assert(QW * 64 * (16 * R::DT + 1) * 4 <= RELH_OFF, "the second halves' results");
};

template <typename T>
__global__ __launch_bounds__(64 * SplitCfg::WAVES, 2) void attn_global_split_kernel(AttnArgs a) {
  using C = SplitCfg;
  constexpr int HD = 80;
  __shared__ __attribute__((aligned(16))) unsigned char lds[C::LDS_BYTES];
  float* relhT = reinterpret_cast<float*>(lds + C::RELH_OFF);  // [kh % RH][BM], * log2(e)

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 31, lh = lane >> 5;
  const int qt = wave & (C::QW - 1), kg = wave / C::QW;  // query tile, key half

  const unsigned int nqb = a.N / C::BM;
  const unsigned int total = (unsigned int)(a.B * a.nH) * nqb;
  const unsigned int pid = xcd_contiguous_id(blockIdx.x, total);
  if (pid >= total) return;
  const int bh = pid / nqb, qb = pid % nqb;
  const int b = bh / a.nH, h = bh % a.nH;
  const int q0 = qb * C::BM + 32 * qt;  // the wavefront's first query: half of one grid row

  const unsigned short* kbase = a.k + b * a.k_sb + h * a.k_sh;
  const unsigned short* vbase = a.v + b * a.v_sb + h * a.v_sh;

  // ---- K / V rows: global memory -> LDS directly, wave instruction i of a tile fills pieces 64 i .. 64 i + 63 ----
  unsigned int koff[C::KDPW];  // bytes, from the tile's first key row; unsigned: scalar-base load form
  int voff[C::VDPW];           // negative: a spare piece, the lane loads nothing
#pragma unroll
  for (int m = 0; m < C::KDPW; ++m) {
    int row;
    const int at = C::k_source(64 * (wave + C::WAVES * m) + lane, row);
    koff[m] = (unsigned int)(row * (int)a.k_sn) * 2u + at;
  }
#pragma unroll
  for (int m = 0; m < C::VDPW; ++m) {
    int row;
    const int at = C::v_source(64 * (wave + C::WAVES * m) + lane, row);
    voff[m] = at < 0 ? -1 : row * (int)a.v_sn * 2 + at;
  }
  const unsigned int lds_base = (unsigned int)(uintptr_t)((__attribute__((address_space(3))) unsigned char*)lds);
  auto k_dma = [&](int kt, int buf) __attribute__((always_inline)) {
    const unsigned char* src = reinterpret_cast<const unsigned char*>(kbase + (int64_t)kt * 64 * a.k_sn);
#pragma unroll
    for (int m = 0; m < C::KDPW; ++m)
      if (wave + C::WAVES * m < C::KP) lds_dma16(src, koff[m], lds_base + buf * C::KTILE + (wave + C::WAVES * m) * 1024);
  };
  auto v_dma = [&](int kt, int buf) __attribute__((always_inline)) {
    const unsigned char* src = reinterpret_cast<const unsigned char*>(vbase + (int64_t)kt * 64 * a.v_sn);
#pragma unroll
    for (int m = 0; m < C::VDPW; ++m)
      if (wave + C::WAVES * m < C::VP && voff[m] >= 0)
        lds_dma16(src, (unsigned int)voff[m], lds_base + C::V_OFF + buf * C::VTILE + (wave + C::WAVES * m) * 1024);
  };
  k_dma(0, 0);
  v_dma(0, 0);
  k_dma(1, 1);  // N % 128 == 0: at least two key rows
  v_dma(1, 1);
  // operand reads of this wavefront's key half
  int vrd[C::DT], krd[C::KS];
#pragma unroll
  for (int dt = 0; dt < C::DT; ++dt) vrd[dt] = C::V_OFF + 32 * kg * (C::VP * 16) + C::v_read(lane, dt);
#pragma unroll
  for (int ks = 0; ks < C::KS; ++ks) krd[ks] = 32 * kg * (C::KP * 16) + C::k_read(lr, lh, ks);

  // The workgroups of a head walk its key rows in step, so every row would be waited for at the latency of the
  // Infinity Cache or HBM.  Each of them touches its own share of the head's K and V first: together they
  // have the head in their XCD's L2 by the time they get to it.
  constexpr int NTOUCH = 2 * C::BM * (HD / 8) / (64 * C::WAVES);
  unsigned int touched[NTOUCH];
#pragma unroll
  for (int i = 0; i < NTOUCH; ++i) {
    const int P = (tid + 64 * C::WAVES * i) % (C::BM * (HD / 8)), row = P / (HD / 8), col = P % (HD / 8);
    const bool is_v = 2 * i >= NTOUCH;
    touched[i] = *reinterpret_cast<const unsigned int*>((is_v ? vbase : kbase) + (int64_t)(qb * C::BM + row) * (is_v ? a.v_sn : a.k_sn) + col * 8);
  }

  // ---- Q^T operand: query lr, channels 16s + 8lh .. +7 ----
  u32x4 qf[C::KS];
  {
    const unsigned short* qp = a.q + b * a.q_sb + h * a.q_sh + (int64_t)(q0 + lr) * a.q_sn + 8 * lh;
#pragma unroll
    for (int s = 0; s < C::KS; ++s) qf[s] = load_x8_global(qp + 16 * s);
  }

  // the spare pieces of V tile `buf`: (1, 0, ..) and zeros
  auto ones = [&](int buf) __attribute__((always_inline)) {
    if (tid < 64) {
      u32x4* p = reinterpret_cast<u32x4*>(lds + C::V_OFF + buf * C::VTILE + tid * (C::VP * 16) + HD * 2);
      p[0] = u32x4{T::kOne, 0u, 0u, 0u};
      p[1] = u32x4{0u, 0u, 0u, 0u};
    }
  };
  ones(0);
  ones(1);
  // rel_h of key rows kh0 .. kh0 + 31, shared by the two key halves
  auto fill_relh = [&](int kh0) __attribute__((always_inline)) {
    const unsigned short* rhb = a.rh + b * a.rh_sb + h * a.rh_sh + (int64_t)(qb * C::BM) * a.rh_sn;
    const int ql = tid / 4, part = tid % 4;  // 64 queries x 4 pieces of 8 key rows
    static_assert(C::BM * 4 == 64 * C::WAVES, "one piece per thread");
    unsigned short v8[8];
    const unsigned short* src = rhb + (int64_t)ql * a.rh_sn + kh0 + 8 * part;
    if (a.relh_x8) {
      *reinterpret_cast<u32x4*>(v8) = load_x8_global(src);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) v8[e] = kh0 + 8 * part + e < a.gh ? src[e] : (unsigned short)0;
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) relhT[(8 * part + e) * C::BM + ql] = T::from_bits(v8[e]) * kLog2e;
  };

  // ---- rel_w / sm_scale of this wavefront's keys, the initial accumulator of every score tile ----
  f32x16 b1;
  {
    const unsigned short* rwp = a.rw + b * a.rw_sb + h * a.rw_sh + (int64_t)(q0 + lr) * a.rw_sn + 32 * kg + 4 * lh;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const u32x2 w = *reinterpret_cast<const u32x2*>(rwp + 8 * j);
      b1[4 * j + 0] = T::lo(w[0]) * a.inv_scale;
      b1[4 * j + 1] = T::hi(w[0]) * a.inv_scale;
      b1[4 * j + 2] = T::lo(w[1]) * a.inv_scale;
      b1[4 * j + 3] = T::hi(w[1]) * a.inv_scale;
    }
  }
  fill_relh(0);
#pragma unroll
  for (int i = 0; i < NTOUCH; ++i) asm volatile("" : : "v"(touched[i]));
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's share of tile 0 has landed
  __syncthreads();

  // ---- main loop over key grid rows ----
  f32x16 oacc[C::DT];
#pragma unroll
  for (int dt = 0; dt < C::DT; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) oacc[dt][r] = 0.f;
  float m_i = T::kLowest;

  const int nkt = a.N / 64;
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) s16x4* trptr_t;
  // The loop is pipelined inside a wavefront as attn_global_kernel's is: between the exponentials of row kt stand
  // the matrix instructions of the scores of row kt + 1 and of P V of row kt - 1.
  u32x4 kf[C::KS], vf[2][C::DT], pkA[2], pkB[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    pkA[j] = pkB[j] = u32x4{0u, 0u, 0u, 0u};
#pragma unroll
    for (int dt = 0; dt < C::DT; ++dt) vf[j][dt] = u32x4{0u, 0u, 0u, 0u};
  }
  auto read_v = [&](int j, int dt, int buf) __attribute__((always_inline)) {
    const unsigned char* p = lds + vrd[dt] + buf * C::VTILE + 16 * j * (C::VP * 16);
    const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((trptr_t)p));
    const u32x2 hi = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((trptr_t)(p + 8 * C::VP * 16)));
    vf[j][dt] = u32x4{lo[0], lo[1], hi[0], hi[1]};
  };
  auto row = [&](int kt, auto buf_c, f32x16& s, f32x16& s_next, u32x4 (&pk)[2], u32x4 (&pk_prev)[2]) __attribute__((always_inline)) {
    constexpr int BUF = decltype(buf_c)::value;  // kt & 1, for constant LDS offsets
    if (kt == C::RH) {  // uniform; everybody has left row kt - 1 (the barrier at its end)
      fill_relh(kt);
      __syncthreads();
    }
    const float b0 = relhT[(kt % C::RH) * C::BM + 32 * qt + lr];
#pragma unroll
    for (int ks = 0; ks < C::KS; ++ks) kf[ks] = *reinterpret_cast<const u32x4*>(lds + krd[ks] + (BUF ^ 1) * C::KTILE);
    __builtin_amdgcn_sched_barrier(0);
    if (kt + 2 < nkt) k_dma(kt + 2, BUF);  // row kt's scores are made: its K buffer is free
    __builtin_amdgcn_sched_barrier(0);

    unsigned int seen = 0u;
    auto pair = [&](int w, float neg_mrow) __attribute__((always_inline)) {  // packed pair w of 8
      const float p0 = fast_exp2(fmaf(s[2 * w], a.c, neg_mrow)), p1 = fast_exp2(fmaf(s[2 * w + 1], a.c, neg_mrow));
      pk[w >> 2][w & 3] = T::pack2(p0, p1);
    };
    auto score = [&](int ks) __attribute__((always_inline)) { s_next = T::mfma(kf[ks], qf[ks], ks == 0 ? b1 : s_next); };
    auto pv = [&](int j, int dt) __attribute__((always_inline)) { oacc[dt] = T::mfma(vf[j][dt], pk_prev[j], oacc[dt]); };
    const float neg_mrow = b0 - m_i;
    // (the last row's kf is whatever the buffer holds: its product is not used)
    float e0, e1;  // a pair is packed one step after its exponentials were issued
#pragma unroll
    for (int g = 0; g < 8; ++g) {
      const float x0 = fmaf(s[2 * g], a.c, neg_mrow), x1 = fmaf(s[2 * g + 1], a.c, neg_mrow);
      if (g > 0) pk[(g - 1) >> 2][(g - 1) & 3] = T::pack2(e0, e1);
      e0 = fast_exp2(x0);
      e1 = fast_exp2(x1);
      if (g > 0 && !(g & 1)) seen = T::note(seen, pk[(g - 1) >> 2][(g - 2) & 3], pk[(g - 1) >> 2][(g - 1) & 3]);
      __builtin_amdgcn_sched_barrier(0);
      if (g == 0) pv(0, 0);
      if (g == 1) {
#pragma unroll
        for (int dt = 1; dt < C::DT; ++dt) pv(0, dt);
      }
      if (g >= 2 && g < 2 + C::KS) score(g - 2);
      if (g == 6) pv(1, 0);
      if (g == 7) {
#pragma unroll
        for (int dt = 1; dt < C::DT; ++dt) pv(1, dt);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    // this row's V for the next round
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int dt = 0; dt < C::DT; ++dt) read_v(j, dt, BUF);
    pk[1][3] = T::pack2(e0, e1);
    seen = T::note(seen, pk[1][2], pk[1][3]);
    if (__any(T::outgrown(seen))) {  // move the reference, as above
      float mx = s[0];
#pragma unroll
      for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[r]);
      mx = max_with_lane_xor32(mx);
      const float m_new = fmaxf(m_i, fmaf(mx, a.c, b0 + T::kMargin));
      const float alpha = fast_exp2(m_i - m_new);
      m_i = m_new;
#pragma unroll
      for (int dt = 0; dt < C::DT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[dt][r] *= alpha;
#pragma unroll
      for (int w = 0; w < 8; ++w) pair(w, b0 - m_i);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's share of K row kt + 2 and V row kt + 1 has landed
    __syncthreads();
    if (kt + 2 < nkt) v_dma(kt + 2, BUF);  // row kt's V is in registers
  };
  f32x16 sA, sB;
#pragma unroll
  for (int ks = 0; ks < C::KS; ++ks)
    sA = T::mfma(*reinterpret_cast<const u32x4*>(lds + krd[ks]), qf[ks], ks == 0 ? b1 : sA);
  __syncthreads();  // K row 0 has been read by everyone: its buffer may be refilled
  for (int kt = 0; kt < nkt; kt += 2) {  // nkt is even
    row(kt, std::integral_constant<int, 0>{}, sA, sB, pkA, pkB);
    row(kt + 1, std::integral_constant<int, 1>{}, sB, sA, pkB, pkA);
  }
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int dt = 0; dt < C::DT; ++dt) oacc[dt] = T::mfma(vf[j][dt], pkB[j], oacc[dt]);  // P V of the last row

  // ---- the two key halves meet: reference and accumulators (the denominator among them) of half 1 through LDS ----
  float* other = reinterpret_cast<float*>(lds) + qt * 64 * (16 * C::DT + 1) + lane;  // word w of lane: 64 w + lane
  if (kg == 1) {
#pragma unroll
    for (int dt = 0; dt < C::DT; ++dt)
#pragma unroll
      for (int r = 0; r < 16; ++r) other[64 * (16 * dt + r)] = oacc[dt][r];
    other[64 * 16 * C::DT] = m_i;
  }
  __syncthreads();
  if (kg == 1) return;
  {
    // (a half all of whose keys are taken away: its reference is T::kLowest, its sums are zero)
    const float m1 = other[64 * 16 * C::DT];
    const float m = fmaxf(m_i, m1);
    const float f0 = fast_exp2(m_i - m), f1 = fast_exp2(m1 - m);
#pragma unroll
    for (int dt = 0; dt < C::DT; ++dt)
#pragma unroll
      for (int r = 0; r < 16; ++r) oacc[dt][r] = oacc[dt][r] * f0 + other[64 * (16 * dt + r)] * f1;
  }
  constexpr int orow = HD % 32;  // the denominator's row of the last channel tile
  constexpr int oreg = 4 * (orow / 8) + orow % 4, olh = (orow / 4) % 2;
  const float own = oacc[C::DT - 1][oreg], partner = xor32(own);
  const float inv = 1.0f / (lh == olh ? own : partner);
  unsigned short* op = a.out + b * a.o_sb + h * a.o_sh + (int64_t)(q0 + lr) * a.o_sn;
#pragma unroll
  for (int dt = 0; dt < C::DT; ++dt)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int d = 32 * dt + 8 * j + 4 * lh;
      if (d < HD) {
        const u32x2 o = {T::pack2(oacc[dt][4 * j] * inv, oacc[dt][4 * j + 1] * inv),
                         T::pack2(oacc[dt][4 * j + 2] * inv, oacc[dt][4 * j + 3] * inv)};
        *reinterpret_cast<u32x2*>(op + d) = o;
      }
    }
}

// The split form at hd 64 on 16 x 16 x 32 matrix instructions: half the accumulator bytes per product cross the register file, which counts because the
// power limit is what a SIMD's matrix pipe and vector unit share (bare loops on N(0, 0.5) values 1.94 PFLOP/s for 1.77 of the 32 x 32 form).  A lane holds
// two queries, lane % 16 and 16 more, and of every 16 keys the four from 4 (lane / 16) on; the packed pairs of a half row are the P V
// operand as they stand, its k slots 8 q .. 8 q + 7 being the keys 4 q .. + 3 and 16 + 4 q .. + 3, and two transposing reads bring V in that order.
// us, 32 x 32 x 16 / so (bf16; fp16): 1 x 8 heads 51.5 / 49.7; 50.9 / 47.9, 1 x 12 66.0 / 63.8; 69.3 / 66.3, 4 x 12 242 / 232; 259 / 244, 8 x 16 645 / 636; 675 / 658, 9 x 16 x 6 rows
// of 64 19.2 / 18.1; 18.7 / 18.2.  The error against 64 bits is the same to three digits (2.35e-3, 2.94e-4 of the norm).
// Up to 256 workgroups are one wavefront a SIMD, which waits for the matrix pipe between a step's two instructions if they stand side by side: there
// they stand apart, one on either side of the exponentials (the same operations: the same bits.  us, 32 x 32 x 16 / side by side / apart, bf16; fp16: 2 x 1 heads 30.3 / 32.4 / 30.9;
// 31.2 / 32.6 / 31.0, 2 x 3 x 40 rows 21.4 / 22.8 / 21.9, 4 x 1 x 40 fp16 21.8 / 22.8 / 21.8; over 61 calls 1.045 and 1.01 times as long as the 32 x 32 form, whose half as many
// instructions that wavefront issues sooner).  From 257 to 448, where other wavefronts fill the wait, side by side is up to 2 % ahead, beyond the two are level.
// What the smaller instruction does not gain in bf16: one wavefront a SIMD on some CUs and two on others (1 x 5 heads 41.7 / 42.6, 1 x 6 42.6 / 42.8; fp16 42.7 / 42.4, 43.7 / 42.7), and
// single calls on an idle GPU, which the power limit does not reach (1 x 5 51.5 / 53.0, 1 x 12 73.4 / 73.3, 8 x 16 665 / 670; fp16 53.0 / 53.2, 77.2 / 75.2, 704 / 685).
struct Split16Cfg {
  using R = GridRow<64>;
  static constexpr int QW = 2, WAVES = 2 * QW, BM = 32 * QW;  // query tiles of 32 and two key halves
  static constexpr int KTILE = R::KTILE, VTILE = R::VTILE, PW = R::KP / WAVES;  // PW: wave instructions of a tile
  static constexpr int V_OFF = 2 * KTILE;       // LDS: K tiles of both stages, V tiles of both stages, rel_h
  static constexpr int RELH_OFF = V_OFF + 2 * VTILE;
  static constexpr int RH = 32;                 // key rows whose rel_h is at hand
  static constexpr int LDS_BYTES = RELH_OFF + RH * BM * 4;
  // V rows are 128 bytes; a transposing read takes 32 of them from each of 16 rows, eight rows at a time: 16-byte piece c of row r stands at c ^ v_swizzle(r)
  static SF_DEVICE int v_swizzle(int row) { return 2 * ((row >> 1) & 3); }
  static_assert(R::KP % WAVES == 0 && R::VP == R::KP, "whole wave instructions");
  static_assert(3 * LDS_BYTES <= 160 * 1024, "three workgroups per CU");
  static_assert(QW * 64 * 36 * 4 <= RELH_OFF, "the second halves' results");
};

// SPREAD: a step's two matrix instructions stand apart in its vector work (see above)
template <typename T, bool SPREAD>
__global__ __launch_bounds__(64 * Split16Cfg::WAVES, 3) void attn_global_split16_kernel(AttnArgs a) {
  using C = Split16Cfg;
  constexpr int HD = 64;
  __shared__ __attribute__((aligned(16))) unsigned char lds[C::LDS_BYTES];
  float* relhT = reinterpret_cast<float*>(lds + C::RELH_OFF);  // [kh % RH][BM], * log2(e)

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lq = lane >> 4;
  const int qt = wave & (C::QW - 1), kg = wave / C::QW;  // query tile, key half

  const unsigned int nqb = a.N / C::BM;
  const unsigned int total = (unsigned int)(a.B * a.nH) * nqb;
  const unsigned int pid = xcd_contiguous_id(blockIdx.x, total);
  if (pid >= total) return;
  const int bh = pid / nqb, qb = pid % nqb;
  const int b = bh / a.nH, h = bh % a.nH;
  const int q0 = qb * C::BM + 32 * qt;  // the wavefront's first query: half of one grid row

  const unsigned short* kbase = a.k + b * a.k_sb + h * a.k_sh;
  const unsigned short* vbase = a.v + b * a.v_sb + h * a.v_sh;

  // ---- K / V rows: global memory -> LDS directly, wave instruction i of a tile fills pieces 64 i .. 64 i + 63 ----
  unsigned int koff[C::PW], voff[C::PW];  // bytes, from the tile's first key row; unsigned: scalar-base load form
#pragma unroll
  for (int m = 0; m < C::PW; ++m) {
    int row;
    const int P = 64 * (wave + C::WAVES * m) + lane, at = C::R::k_source(P, row);
    koff[m] = (unsigned int)(row * (int)a.k_sn) * 2u + at;
    voff[m] = (unsigned int)(row * (int)a.v_sn) * 2u + ((P % 8) ^ C::v_swizzle(row)) * 16;
  }
  const unsigned int lds_base = (unsigned int)(uintptr_t)((__attribute__((address_space(3))) unsigned char*)lds);
  auto k_dma = [&](int kt, int buf) __attribute__((always_inline)) {
    const unsigned char* src = reinterpret_cast<const unsigned char*>(kbase + (int64_t)kt * 64 * a.k_sn);
#pragma unroll
    for (int m = 0; m < C::PW; ++m) lds_dma16(src, koff[m], lds_base + buf * C::KTILE + (wave + C::WAVES * m) * 1024);
  };
  auto v_dma = [&](int kt, int buf) __attribute__((always_inline)) {
    const unsigned char* src = reinterpret_cast<const unsigned char*>(vbase + (int64_t)kt * 64 * a.v_sn);
#pragma unroll
    for (int m = 0; m < C::PW; ++m) lds_dma16(src, voff[m], lds_base + C::V_OFF + buf * C::VTILE + (wave + C::WAVES * m) * 1024);
  };
  k_dma(0, 0);
  v_dma(0, 0);
  k_dma(1, 1);  // N % 128 == 0: at least two key rows
  v_dma(1, 1);
  // operand reads of this wavefront's key half: K row lr, channels 32 s + 8 lq .. +7; V keys 4 lq + lr / 4, channels 16 ct + 4 (lr % 4) .. +3
  int krd[2], vrd[4];
#pragma unroll
  for (int s = 0; s < 2; ++s) krd[s] = (32 * kg + lr) * 128 + ((4 * s + lq) ^ C::R::k_swizzle(lr)) * 16;
  {
    const int key = 4 * lq + (lr >> 2);
#pragma unroll
    for (int ct = 0; ct < 4; ++ct)
      vrd[ct] = C::V_OFF + (32 * kg + key) * 128 + ((2 * ct + ((lr & 3) >> 1)) ^ C::v_swizzle(key)) * 16 + 8 * (lr & 1);
  }

  // Each workgroup touches its own share of the head's K and V first (see above).
  constexpr int NTOUCH = 2 * C::BM * (HD / 8) / (64 * C::WAVES);
  unsigned int touched[NTOUCH];
#pragma unroll
  for (int i = 0; i < NTOUCH; ++i) {
    const int P = (tid + 64 * C::WAVES * i) % (C::BM * (HD / 8)), row = P / (HD / 8), col = P % (HD / 8);
    const bool is_v = 2 * i >= NTOUCH;
    touched[i] = *reinterpret_cast<const unsigned int*>((is_v ? vbase : kbase) + (int64_t)(qb * C::BM + row) * (is_v ? a.v_sn : a.k_sn) + col * 8);
  }

  // ---- Q^T operands: queries lr and 16 + lr, channels 32 s + 8 lq .. +7 ----
  u32x4 qf[2][2];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const unsigned short* qp = a.q + b * a.q_sb + h * a.q_sh + (int64_t)(q0 + 16 * t + lr) * a.q_sn + 8 * lq;
#pragma unroll
    for (int s = 0; s < 2; ++s) qf[t][s] = load_x8_global(qp + 32 * s);
  }
  // rel_h of key rows kh0 .. kh0 + 31, shared by the two key halves
  auto fill_relh = [&](int kh0) __attribute__((always_inline)) {
    const unsigned short* rhb = a.rh + b * a.rh_sb + h * a.rh_sh + (int64_t)(qb * C::BM) * a.rh_sn;
    const int ql = tid / 4, part = tid % 4;  // 64 queries x 4 pieces of 8 key rows
    static_assert(C::BM * 4 == 64 * C::WAVES, "one piece per thread");
    unsigned short v8[8];
    const unsigned short* src = rhb + (int64_t)ql * a.rh_sn + kh0 + 8 * part;
    if (a.relh_x8) {
      *reinterpret_cast<u32x4*>(v8) = load_x8_global(src);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) v8[e] = kh0 + 8 * part + e < a.gh ? src[e] : (unsigned short)0;
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) relhT[(8 * part + e) * C::BM + ql] = T::from_bits(v8[e]) * kLog2e;
  };

  // ---- rel_w / sm_scale of this wavefront's keys, the initial accumulator of every score tile: [16 keys][16 queries] ----
  f32x4 b1[2][2];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const unsigned short* rwp = a.rw + b * a.rw_sb + h * a.rw_sh + (int64_t)(q0 + 16 * t + lr) * a.rw_sn + 32 * kg + 4 * lq;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const u32x2 w = *reinterpret_cast<const u32x2*>(rwp + 16 * k);
      b1[k][t] = f32x4{T::lo(w[0]) * a.inv_scale, T::hi(w[0]) * a.inv_scale, T::lo(w[1]) * a.inv_scale, T::hi(w[1]) * a.inv_scale};
    }
  }
  fill_relh(0);
#pragma unroll
  for (int i = 0; i < NTOUCH; ++i) asm volatile("" : : "v"(touched[i]));
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's share of tile 0 has landed
  __syncthreads();

  // ---- main loop over key grid rows, pipelined inside a wavefront as attn_global_split_kernel's ----
  f32x4 oacc[4][2];
#pragma unroll
  for (int ct = 0; ct < 4; ++ct)
#pragma unroll
    for (int t = 0; t < 2; ++t) oacc[ct][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m_i[2] = {T::kLowest, T::kLowest}, l_i[2] = {0.f, 0.f};

  const int nkt = a.N / 64;
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) s16x4* trptr_t;
  struct Scores { f32x4 v[2][2]; };  // [16 keys][16 queries]
  u32x4 kf[2][2], vf[4], pkA[2], pkB[2];
#pragma unroll
  for (int t = 0; t < 2; ++t) pkA[t] = pkB[t] = u32x4{0u, 0u, 0u, 0u};
#pragma unroll
  for (int ct = 0; ct < 4; ++ct) vf[ct] = u32x4{0u, 0u, 0u, 0u};
  auto read_k = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int s = 0; s < 2; ++s) kf[k][s] = *reinterpret_cast<const u32x4*>(lds + krd[s] + buf * C::KTILE + k * 16 * 128);
  };
  auto read_v = [&](int ct, int buf) __attribute__((always_inline)) {
    const unsigned char* p = lds + vrd[ct] + buf * C::VTILE;
    const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((trptr_t)p));
    const u32x2 hi = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((trptr_t)(p + 16 * 128)));
    vf[ct] = u32x4{lo[0], lo[1], hi[0], hi[1]};
  };
  // instruction n of the eight of a half row's scores (both of a k step's key tiles before the next step) / of its P V
  auto score = [&](Scores& s, int n) __attribute__((always_inline)) {
    const int ks = n >> 2, k = (n >> 1) & 1, t = n & 1;
    s.v[k][t] = T::mfma16(kf[k][ks], qf[t][ks], ks == 0 ? b1[k][t] : s.v[k][t]);
  };
  auto pv = [&](const u32x4 (&pk)[2], int n) __attribute__((always_inline)) { oacc[n >> 1][n & 1] = T::mfma16(vf[n >> 1], pk[n & 1], oacc[n >> 1][n & 1]); };
  auto row = [&](int kt, auto buf_c, Scores& s, Scores& s_next, u32x4 (&pk)[2], u32x4 (&pk_prev)[2]) __attribute__((always_inline)) {
    constexpr int BUF = decltype(buf_c)::value;  // kt & 1, for constant LDS offsets
    if (kt == C::RH) {  // uniform; everybody has left row kt - 1 (the barrier at its end)
      fill_relh(kt);
      __syncthreads();
    }
    const float* rh = relhT + (kt % C::RH) * C::BM + 32 * qt + lr;
    const float b0[2] = {rh[0], rh[16]};
    read_k(BUF ^ 1);
    __builtin_amdgcn_sched_barrier(0);
    if (kt + 2 < nkt) k_dma(kt + 2, BUF);  // row kt's scores are made: its K buffer is free
    __builtin_amdgcn_sched_barrier(0);

    float neg_mrow[2] = {b0[0] - m_i[0], b0[1] - m_i[1]};
    float l0[2] = {0.f, 0.f}, l1[2] = {0.f, 0.f};  // this row's share of the denominators, unrounded (two chains each)
    float e0, e1;  // a pair is packed one step after its exponentials were issued
    auto gather = [&](int w) __attribute__((always_inline)) {  // pair w: query w / 4, keys 16 (w / 2 % 2) + 4 lq + 2 (w % 2) and one more
      pk[w >> 2][w & 3] = T::pack2(e0, e1);
      l0[w >> 2] += e0;
      l1[w >> 2] += e1;
    };
    // (the last row's kf is whatever the buffer holds: its product is not used)
#pragma unroll
    for (int g = 0; g < 8; ++g) {
      const int t = g >> 2, k = (g >> 1) & 1, r = 2 * (g & 1);
      const float x0 = fmaf(s.v[k][t][r], a.c, neg_mrow[t]), x1 = fmaf(s.v[k][t][r + 1], a.c, neg_mrow[t]);
      auto product = [&](int n) __attribute__((always_inline)) {
        if (g < 2) pv(pk_prev, 2 * g + n);
        else if (g < 6) score(s_next, 2 * (g - 2) + n);
        else pv(pk_prev, 2 * (g - 4) + n);
      };
      if (g > 0) gather(g - 1);
      if constexpr (SPREAD) {
        __builtin_amdgcn_sched_barrier(0);
        product(0);
        __builtin_amdgcn_sched_barrier(0);
      }
      e0 = fast_exp2(x0);
      e1 = fast_exp2(x1);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (!SPREAD) product(0);
      product(1);
      __builtin_amdgcn_sched_barrier(0);
    }
    // this row's V for the next round
#pragma unroll
    for (int ct = 0; ct < 4; ++ct) read_v(ct, BUF);
    gather(7);
#pragma unroll
    for (int t = 0; t < 2; ++t) l0[t] += l1[t];
    if (__any(l0[0] > kCeiling || l0[1] > kCeiling)) {  // move the references, as above
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        float mx = s.v[0][t][0];
#pragma unroll
        for (int w = 1; w < 8; ++w) mx = fmaxf(mx, s.v[w >> 2][t][w & 3]);
        mx = max_with_lane_xor32(fmaxf(mx, __shfl_xor(mx, 16, 64)));
        const float m_new = fmaxf(m_i[t], fmaf(mx, a.c, b0[t] + T::kMargin));
        const float alpha = fast_exp2(m_i[t] - m_new);
        m_i[t] = m_new;
        l_i[t] *= alpha;
        neg_mrow[t] = b0[t] - m_new;
        l0[t] = 0.f;
#pragma unroll
        for (int ct = 0; ct < 4; ++ct) oacc[ct][t] *= alpha;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          const f32x4 v = s.v[w >> 1][t];
          const float p0 = fast_exp2(fmaf(v[2 * (w & 1)], a.c, neg_mrow[t])), p1 = fast_exp2(fmaf(v[2 * (w & 1) + 1], a.c, neg_mrow[t]));
          pk[t][w] = T::pack2(p0, p1);
          l0[t] += p0 + p1;
        }
      }
    }
#pragma unroll
    for (int t = 0; t < 2; ++t) l_i[t] += l0[t];
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's share of K row kt + 2 and V row kt + 1 has landed
    __syncthreads();
    if (kt + 2 < nkt) v_dma(kt + 2, BUF);  // row kt's V is in registers
  };
  Scores sA, sB;
  read_k(0);
#pragma unroll
  for (int n = 0; n < 8; ++n) score(sA, n);
  __syncthreads();  // K row 0 has been read by everyone: its buffer may be refilled
  for (int kt = 0; kt < nkt; kt += 2) {  // nkt is even
    row(kt, std::integral_constant<int, 0>{}, sA, sB, pkA, pkB);
    row(kt + 1, std::integral_constant<int, 1>{}, sB, sA, pkB, pkA);
  }
#pragma unroll
  for (int n = 0; n < 8; ++n) pv(pkB, n);  // of the last row

  // ---- the two key halves meet: references, denominators and accumulators of half 1 through LDS ----
  float* other = reinterpret_cast<float*>(lds) + qt * 64 * 36 + lane;  // word w of lane: 64 w + lane
  if (kg == 1) {
#pragma unroll
    for (int ct = 0; ct < 4; ++ct)
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) other[64 * (8 * ct + 4 * t + r)] = oacc[ct][t][r];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      other[64 * (32 + t)] = m_i[t];
      other[64 * (34 + t)] = l_i[t];
    }
  }
  __syncthreads();
  if (kg == 1) return;
  unsigned short* op = a.out + b * a.o_sb + h * a.o_sh + (int64_t)(q0 + lr) * a.o_sn;
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    // (a half all of whose keys are taken away: its reference is T::kLowest, its sums are zero)
    const float m1 = other[64 * (32 + t)], l1 = other[64 * (34 + t)];
    const float m = fmaxf(m_i[t], m1);
    const float f0 = fast_exp2(m_i[t] - m), f1 = fast_exp2(m1 - m);
    float l = l_i[t] * f0 + l1 * f1;
    l += __shfl_xor(l, 16, 64);
    l += xor32(l);
    const float inv = 1.0f / l;
#pragma unroll
    for (int ct = 0; ct < 4; ++ct) {
      float o[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) o[r] = (oacc[ct][t][r] * f0 + other[64 * (8 * ct + 4 * t + r)] * f1) * inv;
      *reinterpret_cast<u32x2*>(op + (int64_t)(16 * t) * a.o_sn + 16 * ct + 4 * lq) = u32x2{T::pack2(o[0], o[1]), T::pack2(o[2], o[3])};
    }
  }
}

// The unsplit form at hd 80 on 16 x 16 matrix instructions (see attn_global_split16_kernel for the lane's two queries and the order of its keys): 80 channels are two
// k steps of 32 and one of 16, five channel tiles of V^T without padding, and a sixth tile whose channels are one for every key, from registers, the denominators: 24
// instructions of 16 cycles a half row, where the 32 x 32 form (attn_global_bias_kernel, whose channels 80 to 95 were ones and zeros of V's rows) had 11 of 32.  What bounds it: a
// wavefront's vector instructions, 64 a half row of which 16 are exponentials, and matrix instructions, issued one after another, and from about 256 workgroups of 256 queries on the
// power limit besides (15 to 17 %, the file's head).  They stand one by one in turn: three side by side are 3 to 4 % slower.  A key row neither begins with a read
// of its rel_h (read a row ahead) nor ends with a wait for the V fragments that are on their way (the barrier alone, behind vmcnt): 4 to 6 %.  The
// denominators as 16 additions 2 %, as v_dot2 7 % slower.
// us, 32 x 32 / so (bf16; fp16): 1 x 8 heads 63.1 / 61.7; 63.5 / 60.5, 1 x 12 77.6 / 78.0; 82.1 / 80.7, 1 x 16 91.1 / 86.9; 97.8 / 91.7, 2 x 16 181.7 / 173.0; 194.8 / 182.3, 4 x 12 268
// / 257; 288 / 271, 8 x 16 720 / 691; 768 / 738, 16 x 16 1431 / 1381; 1533 / 1457, 3 x 13 x 24 rows 40.3 / 38.4; 42.2 / 40.0; where
// the power limit is far it is behind for its matrix cycles, 384 a half row for 352: a batch of one up to a wavefront a SIMD level to 2 % (24 grids, two types; 1 x 8 x 32 rows 30.8 / 31.4; 30.9 / 31.2, 1 x 12 x 8 12.1 / 12.1;
// 12.0 / 12.1), on 144 of 256 CUs 3 to 4 % (1 x 12 x 48 rows 63.4 / 65.5; 65.2 / 68.1), where batches from four on are 1 to 7 % ahead at every number of wavefronts (8 x 16 x 4 rows 10.7 / 10.0; 10.9 / 10.0).  No
// line between the two forms can look at the batch, on which a slice's bits are not to depend (K read a half row ahead where it has landed: 12.6, 19.5).  The error against 64 bits is the same to three digits (2.33e-3, 2.92e-4 of the norm).
template <int WAVES>
struct Bias16Cfg {
  static constexpr int HD = 80, PIECES = HD / 8;        // 16-byte pieces of a row = wave instructions of a tile
  static constexpr int BM = 32 * WAVES;                 // queries per workgroup
  static constexpr int DPW = (PIECES + WAVES - 1) / WAVES;
  static constexpr int PITCH = HD * 2, TILE = 64 * PITCH;
  // LDS: two K tiles, three V tiles (of a row's V the second half is still to be read when the row two behind is requested), rel_h
  static constexpr int V_OFF = 2 * TILE;
  static constexpr int RH = 32;                         // key rows whose rel_h is at hand
  static constexpr int RELH_OFF = V_OFF + 3 * TILE;
  static constexpr int LDS_BYTES = RELH_OFF + RH * BM * 4;
  static_assert(LDS_BYTES <= (WAVES == 4 ? 80 : 160) * 1024, "workgroups per CU");
  // Rows lie as they come, but for the last two pieces of K, which are read eight bytes at a time and change places in eight rows of sixteen: 160
  // bytes are ten sixteenths of the banks, so that eight rows of 32 bytes are all of them once, and sixteen rows of
  // which half are read a piece further on (in the order in which reads of 16 bytes are served, once_swizzle's note).
  static SF_DEVICE int k_swizzle(int piece, int row) { return piece >= 8 ? (row >> 3) & 1 : 0; }
};

template <typename T, int WAVES>
__global__ __launch_bounds__(64 * WAVES, 2) void attn_global_bias16_kernel(AttnArgs a) {
  using C = Bias16Cfg<WAVES>;
  constexpr int HD = 80, CT = HD / 16;
  __shared__ __attribute__((aligned(16))) unsigned char lds[C::LDS_BYTES];
  float* relhT = reinterpret_cast<float*>(lds + C::RELH_OFF);  // [kh % RH][BM], * log2(e); a wavefront reads only its own columns

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lq = lane >> 4;

  const unsigned int nqb = a.N / C::BM;
  const unsigned int total = (unsigned int)(a.B * a.nH) * nqb;
  const unsigned int pid = xcd_contiguous_id(blockIdx.x, total);
  if (pid >= total) return;
  const int bh = pid / nqb, qb = pid % nqb;
  const int b = bh / a.nH, h = bh % a.nH;
  const int q0 = qb * C::BM + 32 * wave;  // the wavefront's first query: half of one grid row

  const unsigned short* kbase = a.k + b * a.k_sb + h * a.k_sh;
  const unsigned short* vbase = a.v + b * a.v_sb + h * a.v_sh;

  // ---- K / V rows: global memory -> LDS directly, wave instruction i of a tile fills pieces 64 i .. 64 i + 63 ----
  unsigned int koff[C::DPW], voff[C::DPW];  // bytes, from the tile's first key row; unsigned: scalar-base load form
#pragma unroll
  for (int m = 0; m < C::DPW; ++m) {
    const int P = 64 * (wave + WAVES * m) + lane, row = P / C::PIECES, piece = P % C::PIECES;
    koff[m] = (unsigned int)(row * (int)a.k_sn) * 2u + (piece ^ C::k_swizzle(piece, row)) * 16;
    voff[m] = (unsigned int)(row * (int)a.v_sn) * 2u + piece * 16;
  }
  const unsigned int lds_base = (unsigned int)(uintptr_t)((__attribute__((address_space(3))) unsigned char*)lds);
  auto k_dma = [&](int kt, int buf) __attribute__((always_inline)) {
    const unsigned char* src = reinterpret_cast<const unsigned char*>(kbase + (int64_t)kt * 64 * a.k_sn);
#pragma unroll
    for (int m = 0; m < C::DPW; ++m)
      if (wave + WAVES * m < C::PIECES) lds_dma16(src, koff[m], lds_base + buf * C::TILE + (wave + WAVES * m) * 1024);
  };
  auto v_dma = [&](int kt, unsigned int buf_off) __attribute__((always_inline)) {
    const unsigned char* src = reinterpret_cast<const unsigned char*>(vbase + (int64_t)kt * 64 * a.v_sn);
#pragma unroll
    for (int m = 0; m < C::DPW; ++m)
      if (wave + WAVES * m < C::PIECES) lds_dma16(src, voff[m], lds_base + C::V_OFF + buf_off + (wave + WAVES * m) * 1024);
  };
  k_dma(0, 0);
  v_dma(0, 0);
  k_dma(1, 1);  // N % 128 == 0: at least two key rows
  v_dma(1, C::TILE);

  // ---- Q^T operands: queries lr and 16 + lr; channels 32 s + 8 lq .. +7 of two long k steps, 64 + 4 lq .. +3 of a short one ----
  u32x4 qf[2][2];
  u32x2 qs[2];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const unsigned short* qp = a.q + b * a.q_sb + h * a.q_sh + (int64_t)(q0 + 16 * t + lr) * a.q_sn;
#pragma unroll
    for (int s = 0; s < 2; ++s) qf[t][s] = load_x8_global(qp + 32 * s + 8 * lq);
    qs[t] = *reinterpret_cast<const u32x2*>(qp + 64 + 4 * lq);
  }
  // Each workgroup touches its own share of the head's K and V first (see above).
  constexpr int NTOUCH = 2 * C::BM * C::PIECES / (64 * WAVES);
  unsigned int touched[NTOUCH];
#pragma unroll
  for (int i = 0; i < NTOUCH; ++i) {
    const int P = (tid + 64 * WAVES * i) % (C::BM * C::PIECES), row = P / C::PIECES, col = P % C::PIECES;
    const bool is_v = 2 * i >= NTOUCH;
    touched[i] = *reinterpret_cast<const unsigned int*>((is_v ? vbase : kbase) + (int64_t)(qb * C::BM + row) * (is_v ? a.v_sn : a.k_sn) + col * 8);
  }

  // operand reads: K row lr, its pieces 4 s + lq and, of eight bytes, 8 + lq / 2; V keys 4 lq + lr / 4, channels 16 ct + 4 (lr % 4) .. +3
  int krd[2], krs;
#pragma unroll
  for (int s = 0; s < 2; ++s) krd[s] = lr * C::PITCH + (4 * s + lq) * 16;
  krs = lr * C::PITCH + ((8 + (lq >> 1)) ^ C::k_swizzle(8, lr)) * 16 + 8 * (lq & 1);
  const int vrd = C::V_OFF + (4 * lq + (lr >> 2)) * C::PITCH + 8 * (lr & 3);

  // ---- bias: rel_w / sm_scale of the lane's queries is the initial accumulator of the score tiles of the two
  //      half rows; rel_h * log2(e) stands in LDS, 32 key rows at a time ----
  auto fill_relh = [&](int kh0) __attribute__((always_inline)) {
    // lane: query lane % 32, key rows kh0 + 16 (lane / 32) .. +15
    const int ql = lane & 31, part = 16 * (lane >> 5);
    const unsigned short* src = a.rh + b * a.rh_sb + h * a.rh_sh + (int64_t)(q0 + ql) * a.rh_sn + kh0 + part;
    unsigned short v[16];
    if (a.relh_x8) {
      *reinterpret_cast<u32x4*>(v) = load_x8_global(src);
      *reinterpret_cast<u32x4*>(v + 8) = load_x8_global(src + 8);
    } else {
#pragma unroll
      for (int e = 0; e < 16; ++e) v[e] = kh0 + part + e < a.gh ? src[e] : (unsigned short)0;
    }
#pragma unroll
    for (int e = 0; e < 16; ++e) relhT[(part + e) * C::BM + 32 * wave + ql] = T::from_bits(v[e]) * kLog2e;
  };
  struct Scores { f32x4 v[2][2]; };  // [16 keys][16 queries]
  Scores b1[2];                      // of the two half rows
  fill_relh(0);
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const unsigned short* rwp = a.rw + b * a.rw_sb + h * a.rw_sh + (int64_t)(q0 + 16 * t + lr) * a.rw_sn + 4 * lq;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const u32x2 w = *reinterpret_cast<const u32x2*>(rwp + 16 * k);
      b1[k >> 1].v[k & 1][t] = f32x4{T::lo(w[0]) * a.inv_scale, T::hi(w[0]) * a.inv_scale, T::lo(w[1]) * a.inv_scale, T::hi(w[1]) * a.inv_scale};
    }
  }
#pragma unroll
  for (int i = 0; i < NTOUCH; ++i) asm volatile("" : : "v"(touched[i]));
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's share of the first two rows has landed
  __syncthreads();

  // ---- main loop over half rows of 32 keys, pipelined inside a wavefront as attn_global_bias_kernel's ----
  f32x4 oacc[CT][2];
#pragma unroll
  for (int ct = 0; ct < CT; ++ct)
#pragma unroll
    for (int t = 0; t < 2; ++t) oacc[ct][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  f32x4 lacc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};  // denominators: a tile of channels that are one for every key
  float m_i[2] = {T::kLowest, T::kLowest};
  constexpr unsigned int ONES = T::kOne | T::kOne << 16;
  u32x4 ones = {ONES, ONES, ONES, ONES};
  asm volatile("" : "+v"(ones));
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) s16x4* trptr_t;
  u32x4 kf[2][2], vf[CT], pkA[2], pkB[2];
  u32x2 ks[2];
#pragma unroll
  for (int t = 0; t < 2; ++t) pkA[t] = pkB[t] = u32x4{0u, 0u, 0u, 0u};
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) vf[ct] = u32x4{0u, 0u, 0u, 0u};
  auto read_k = [&](int off) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
#pragma unroll
      for (int s = 0; s < 2; ++s) kf[k][s] = *reinterpret_cast<const u32x4*>(lds + krd[s] + off + k * 16 * C::PITCH);
      ks[k] = *reinterpret_cast<const u32x2*>(lds + krs + off + k * 16 * C::PITCH);
    }
  };
  auto read_v = [&](int ct, unsigned int off) __attribute__((always_inline)) {
    const unsigned char* p = lds + vrd + off + 32 * ct;
    const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((trptr_t)p));
    const u32x2 hi = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((trptr_t)(p + 16 * C::PITCH)));
    vf[ct] = u32x4{lo[0], lo[1], hi[0], hi[1]};
  };
  // instruction n of the twelve of a half row's scores (all four tiles of a k step before the next step) / of the ten of its P V
  auto score = [&](Scores& s, const Scores& first, int n) __attribute__((always_inline)) {
    const int step = n >> 2, k = (n >> 1) & 1, t = n & 1;
    if (step < 2) s.v[k][t] = T::mfma16(kf[k][step & 1], qf[t][step & 1], step == 0 ? first.v[k][t] : s.v[k][t]);
    else s.v[k][t] = T::mfma16_short(ks[k], qs[t], s.v[k][t]);
  };
  auto pv = [&](const u32x4 (&pk)[2], int n) __attribute__((always_inline)) { oacc[n >> 1][n & 1] = T::mfma16(vf[n >> 1], pk[n & 1], oacc[n >> 1][n & 1]); };
  auto sum = [&](const u32x4 (&pk)[2], int t) __attribute__((always_inline)) { lacc[t] = T::mfma16(ones, pk[t], lacc[t]); };
  // s, pk: scores and probabilities of this half row, its V at v_off, rel_h of its row b0; s_next: scores of the next one, from K at k_off with
  // the initial accumulator `first`; pk_prev: the one before, whose V is in registers
  auto half_row = [&](Scores& s, Scores& s_next, const Scores& first, u32x4 (&pk)[2], u32x4 (&pk_prev)[2], int k_off, unsigned int v_off,
                      const float (&b0)[2]) __attribute__((always_inline)) {
    read_k(k_off);
    __builtin_amdgcn_sched_barrier(0);
    float neg_mrow[2] = {b0[0] - m_i[0], b0[1] - m_i[1]};
    unsigned int seen = 0u;
    float e0, e1;  // a pair is packed one step after its exponentials were issued
    auto gather = [&](int w) __attribute__((always_inline)) {  // pair w: query w / 4, keys 16 (w / 2 % 2) + 4 lq + 2 (w % 2) and one more
      pk[w >> 2][w & 3] = T::pack2(e0, e1);
      if (w & 1) seen = T::note(seen, pk[w >> 2][(w & 3) - 1], pk[w >> 2][w & 3]);
    };
#pragma unroll
    for (int g = 0; g < 8; ++g) {
      const int t = g >> 2, k = (g >> 1) & 1, r = 2 * (g & 1);
      const float x0 = fmaf(s.v[k][t][r], a.c, neg_mrow[t]), x1 = fmaf(s.v[k][t][r + 1], a.c, neg_mrow[t]);
      // three instructions a step, apart: P V of the one before on the first three channel tiles, the scores, P V on the other two and
      // the denominators
      auto product = [&](int n) __attribute__((always_inline)) {
        if (g < 2) pv(pk_prev, 3 * g + n);
        else if (g < 6) score(s_next, first, 3 * (g - 2) + n);
        else if (n < 2) pv(pk_prev, 6 + 2 * (g - 6) + n);
        else sum(pk_prev, g - 6);
      };
      if (g > 0) gather(g - 1);
      __builtin_amdgcn_sched_barrier(0);
      product(0);
      __builtin_amdgcn_sched_barrier(0);
      e0 = fast_exp2(x0);
      __builtin_amdgcn_sched_barrier(0);
      product(1);
      __builtin_amdgcn_sched_barrier(0);
      e1 = fast_exp2(x1);
      __builtin_amdgcn_sched_barrier(0);
      product(2);
      if (g >= 2 && g < 5) read_v(g - 2, v_off);
      __builtin_amdgcn_sched_barrier(0);
    }
    read_v(3, v_off);
    read_v(4, v_off);
    gather(7);
    if (__any(T::outgrown(seen))) {  // move the references, as above
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        float mx = s.v[0][t][0];
#pragma unroll
        for (int w = 1; w < 8; ++w) mx = fmaxf(mx, s.v[w >> 2][t][w & 3]);
        mx = max_with_lane_xor32(fmaxf(mx, __shfl_xor(mx, 16, 64)));
        const float m_new = fmaxf(m_i[t], fmaf(mx, a.c, b0[t] + T::kMargin));
        const float alpha = fast_exp2(m_i[t] - m_new);
        m_i[t] = m_new;
        lacc[t] *= alpha;
        neg_mrow[t] = b0[t] - m_new;
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) oacc[ct][t] *= alpha;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          const f32x4 v = s.v[w >> 1][t];
          const float p0 = fast_exp2(fmaf(v[2 * (w & 1)], a.c, neg_mrow[t])), p1 = fast_exp2(fmaf(v[2 * (w & 1) + 1], a.c, neg_mrow[t]));
          pk[t][w] = T::pack2(p0, p1);
        }
      }
    }
  };

  const int nkt = a.N / 64;
  // V tiles rotate: row kt's, and the one row kt + 2 goes to (row kt - 1's)
  unsigned int v_cur = 0, v_free = 2 * C::TILE;
  constexpr unsigned int HALF = 32 * C::PITCH;
  Scores sA, sB;
  float b_next[2];
  auto read_relh = [&](int kt) __attribute__((always_inline)) {
    const float* rh = relhT + (kt % C::RH) * C::BM + 32 * wave + lr;
    b_next[0] = rh[0];
    b_next[1] = rh[16];
  };
  read_relh(0);
  read_k(0);
#pragma unroll
  for (int n = 0; n < 12; ++n) score(sA, b1[0], n);
  auto key_row = [&](int kt, auto buf_c) __attribute__((always_inline)) {
    constexpr int BUF = decltype(buf_c)::value;  // kt & 1, for constant LDS offsets
    // rel_h of this row is at hand, the next row's is read now (the wavefront's own columns: no barrier)
    const float b0[2] = {b_next[0], b_next[1]};
    if (kt + 1 == C::RH && nkt > C::RH) fill_relh(C::RH);
    read_relh(kt + 1);
    half_row(sA, sB, b1[1], pkA, pkB, BUF * C::TILE + (int)HALF, v_cur, b0);
    // row kt + 1 has landed (own share) and everybody has left K row kt and V row kt - 1: refill them.  (LDS reads are done in
    // order, and the youngest four are the half row's last two V fragments, of row kt: those may be on their way.)
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(4)\n\ts_barrier" ::: "memory");
    if (kt + 2 < nkt) {
      k_dma(kt + 2, BUF);
      v_dma(kt + 2, v_free);
    }
    // (after the last row kf is whatever the buffer holds: that product is not used)
    half_row(sB, sA, b1[0], pkB, pkA, (BUF ^ 1) * C::TILE, v_cur + HALF, b0);
    v_free = v_cur;
    v_cur = v_cur == 2 * C::TILE ? 0 : v_cur + C::TILE;
  };
  for (int kt = 0; kt < nkt; kt += 2) {  // nkt is even
    key_row(kt, std::integral_constant<int, 0>{});
    key_row(kt + 1, std::integral_constant<int, 1>{});
  }
#pragma unroll
  for (int n = 0; n < 2 * CT; ++n) pv(pkB, n);  // of the last half row
  sum(pkB, 0);
  sum(pkB, 1);

  unsigned short* op = a.out + b * a.o_sb + h * a.o_sh + (int64_t)(q0 + lr) * a.o_sn + 4 * lq;
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const float inv = 1.0f / lacc[t][0];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
      const f32x4 o = oacc[ct][t];
      *reinterpret_cast<u32x2*>(op + (int64_t)(16 * t) * a.o_sn + 16 * ct) = u32x2{T::pack2(o[0] * inv, o[1] * inv), T::pack2(o[2] * inv, o[3] * inv)};
    }
  }
}

// Which form of the global kernel.  Split keys round differently from unsplit ones, so that choice looks at head_dim
// alone: a slice has the same bits whatever batch it travels in.  hd 64 is split (us in bf16, split / unsplit with 8 / with 4
// wavefronts, 4096 tokens: 1 x 8 heads 49 / 68 / 50, 1 x 12: 65 / 69 / 76, 2 x 9: 101 / 143 / 118, 1 x 16: 87 / 79 / 83, 4 x 12: 239 / 236 / 236,
// 8 x 16: 629 / 622 / 617), hd 80, where only two such workgroups fit a CU, is not (55 / 73 / 56, 84 / 76 / 83, 130 / 159 / 136, 106 / 92 / 96, 307 / 272 / 274,
// 818 / 715 / 718; 8 x 16 691 now, attn_global_bias16_kernel).  8 wavefronts or 4, which agree bit for bit: by how the workgroups of 256
// queries (one per CU) and of 128 (two) divide among the 256 CUs.  The prices are microseconds of one full round over
// 64 key rows and, of 128 queries, of a last one with one workgroup per CU.
// Returns 8, 4, or 2 for the key-split form.
static int bias_form(const AttnArgs& a, int hd) {
  const int force = knob(KNOB_ATTN_WAVES);
  const bool by8 = a.N % 256 == 0;
  if (force == 4 || force == 8) return force == 8 && by8 ? 8 : 4;
  const int split = knob_or(KNOB_ATTN_SPLIT, 1);
  if (split == 2 || (split != 0 && hd == 64)) return 2;
  const int64_t slices = (int64_t)a.B * a.nH, wgs4 = slices * (a.N / 128), wgs8 = slices * (a.N / 256), rest4 = wgs4 % 512;
  const int full4 = hd == 64 ? 80 : 88, one4 = hd == 64 ? 53 : 56, full8 = hd == 64 ? 79 : 86;
  const int64_t p4 = wgs4 / 512 * full4 + (rest4 == 0 ? 0 : rest4 <= 256 ? one4 : full4);
  return by8 && (wgs8 + 255) / 256 * full8 <= p4 ? 8 : 4;
}
template <typename T, int HD>
static void launch_bias(const AttnArgs& a, int form, hipStream_t stream) {
  auto grid = [&](int queries) { return dim3((unsigned int)(((int64_t)a.B * a.nH * (a.N / queries) + 7) / 8 * 8)); };
  if constexpr (HD == 80) {
    if (form == 8) hipLaunchKernelGGL((attn_global_bias16_kernel<T, 8>), grid(256), dim3(512), 0, stream, a);
    else if (form == 4) hipLaunchKernelGGL((attn_global_bias16_kernel<T, 4>), grid(128), dim3(256), 0, stream, a);
    else hipLaunchKernelGGL((attn_global_split_kernel<T>), grid(64), dim3(256), 0, stream, a);
  } else {
    if (form == 8) hipLaunchKernelGGL((attn_global_bias_kernel<T, 8>), grid(256), dim3(512), 0, stream, a);
    else if (form == 4) hipLaunchKernelGGL((attn_global_bias_kernel<T, 4>), grid(128), dim3(256), 0, stream, a);
    else if ((int64_t)a.B * a.nH * (a.N / 64) <= 256) hipLaunchKernelGGL((attn_global_split16_kernel<T, true>), grid(64), dim3(256), 0, stream, a);
    else hipLaunchKernelGGL((attn_global_split16_kernel<T, false>), grid(64), dim3(256), 0, stream, a);
  }
}

int attn_global_bias_launch(const AttnArgs& a0, int hd, int dtype, hipStream_t stream) {
  AttnArgs a = a0;
  // rel_h rows can be read 16 bytes at a time, and the last piece read lies inside them
  a.relh_x8 = a.gh % 32 == 0 && a.rh_sn % 8 == 0 && a.rh_sh % 8 == 0 && a.rh_sb % 8 == 0 && aligned16(a.rh);
  const int form = bias_form(a, hd);
  if (dtype == SAMFAST_F16) {
    if (hd == 64) launch_bias<ElemF16, 64>(a, form, stream); else launch_bias<ElemF16, 80>(a, form, stream);
  } else {
    if (hd == 64) launch_bias<ElemBf16, 64>(a, form, stream); else launch_bias<ElemBf16, 80>(a, form, stream);
  }
  return check_launch("attn_global_bias_kernel");
}

}  // namespace samfast
