// One matrix product y = x . w^T for the element types of this library (int8, bf16, fp16): output tiles of 256 rows and 256 or 320
// columns, or 320 rows and 256 columns (int8, and the half types without a residual, also 256 rows and 192 columns), one resident workgroup of eight wavefronts per CU, two per SIMD that take turns at the matrix pipe.
//
// What bounds it, at 65536 x 1280 -> 3840 in int8 (265 us; 197 on all-zero codes, where no power limit acts): the products
// alone are 163 us at the rate that bare loops of the same instruction sustain under the power limit on codes like an encoder's
// (139 on zeros), and the rest is the tiles' ends, in which hardly anything is multiplied: four and a half vector instructions per value
// (eight with the residual), four cycles each, are 5400 cycles of a SIMD beside the loop's 21000.  (Not the burst of stores: the CUs or
// XCDs started up to half a tile's time apart took the same 198-206 us on zeros.  Cycle counts by probes that are not kept; the
// pipe is busy 0.93-0.96 of the loop.)  So the choices here are about energy per product, or about cycles without products:
//   * v_mfma_*_16x16x(64 bytes): bare loops of them (bench.py --mfma-ceiling) sustain 3.95 POP/s on Gaussian codes (bf16: 1.93 PFLOP/s)
//     where the 32x32 forms sustain 3.5 (1.8): half the accumulator bytes per product cross the register file;
//   * 256 x 256 tiles: a third fewer operand bytes from the L2s than 128 x 256 (loops without the loads ran 17 % faster at the
//     same pipe occupancy, without the LDS reads 7 %: probes that are not kept);
//   * turns: the wavefronts 0-3 multiply while 4-7 (their SIMD partners) read fragments and request tiles, and
//     the other way round, a barrier between turns of 32 matrix instructions.  The same code with both halves in
//     step keeps the pipe busy 0.59 of the time.
// A k tile is 128 bytes of every row, so row-major operands are read in whole lines as well as K-block-major ones.  Two
// of them fit the LDS; a wavefront multiplies its 64 rows by the lower 64 of its 128 columns in the first turn and
// by the upper 64 in the second.  After the first the X rows and the lower columns are free again, after the
// second the upper ones, and each part is requested anew as soon as it is free: every load has one and a half k tiles
// (2500 cycles) to arrive although only two are held.
//
// Epilogues: int8 (float(acc) * sx[m]) * sw[n] + bias[n] in three separately rounded fp32 operations, the half
// types acc + bias[n]; rounded to the output type; then nothing, (half types) GELU of the rounded value, or + residual (one more
// rounding).  A wavefront's columns are dealt to the LDS rows so that a lane ends with four adjacent ones and stores
// 128-byte segments straight from the accumulators, between the turns, both sides at once: a wavefront alone issues an instruction every
// 5.2 cycles, two together one every 4.3.  (One side behind the other, and with every store's address made anew, 1045 instead of 676
// instructions, an end was 10800 cycles for now 6300: 65536 x 1280 -> 3840 292 -> 265 us, -> 5120 373 -> 347, 1280 -> 1280 with the residual
// 134.5 -> 126, 20480 x 1024 -> 3072 70 -> 60, bf16 20480 x 1024 -> 4096 with GELU 167 -> 155.)  (Held in registers and sent out a few per turn of
// the next tile, as gemm_i8_persist_kernel does, the stores lengthened every turn: 65536 x 1280 -> 3840 took 363 us for 310.)
//
// Inside the ViT-H encoder at 65536 rows, us per launch (means of a kernel trace), before / with this kernel: 1280 -> 3840 309 / 261 (2.47 POP/s),
// 1280 -> 5120 345 (2.49), 5120 -> 1280 with the residual 404 / 324 (2.65), 1280 -> 1280 with it 136 / 127 (0.4 GB of rows through HBM).
#pragma once

#include "gemm_i8_shared.hpp"
#include "attn_relpos_shared.hpp"

#include <type_traits>

#pragma clang fp contract(off)

namespace samfast {

struct PPArgs {
  const unsigned char* x;  // byte addresses; x_pitch / w_pitch bytes between rows, *_kstep between the 64-byte pieces of a row
  const unsigned char* w;
  unsigned short* out;
  const float* sx;         // int8: row scales, column scales
  const float* sw;
  const void* bias;        // int8: fp32, else the element type; may be null
  const unsigned short* residual;
  int64_t ldo, ld_res;     // elements
  int64_t x_kstep, w_kstep;
  unsigned int x_pitch, w_pitch;
  int M, N, nk;            // nk: 128-byte k tiles
  int tiles_m, tiles_n, group_m;
};

struct PPInt8 {
  typedef i32x4 acc_t;
  typedef ElemBf16 Out;
  static constexpr bool SCALED = true;
  static SF_DEVICE acc_t mma(i32x4 a, i32x4 b, acc_t c) { return __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0); }
};
struct PPBf16 {
  typedef f32x4 acc_t;
  typedef ElemBf16 Out;
  static constexpr bool SCALED = false;
  static SF_DEVICE acc_t mma(i32x4 a, i32x4 b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
};
struct PPF16 {
  typedef f32x4 acc_t;
  typedef ElemF16 Out;
  static constexpr bool SCALED = false;
  typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
  static SF_DEVICE acc_t mma(i32x4 a, i32x4 b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
  }
};

enum { PP_PLAIN = 0, PP_GELU = 1, PP_RESIDUAL = 2 };

// vmcnt <= N and every LDS read of this wavefront done
template <int N>
SF_DEVICE void pp_wait() {
  __builtin_amdgcn_s_waitcnt(0x0070 | (N & 15) | ((N >> 4) << 14));
}

// TM: 16-row fragments of a wavefront (the tile has 64 TM rows).  TN: 16-column fragments of a wavefront's half of the tile (the
// tile has 32 TN columns).  A turn multiplies H of them.  The fragments' columns are dealt so that a lane ends with quads and at most one pair of adjacent columns:
// element e of a quad q is column 64 q + 4 lr + e of the half, of the pair 64 NQ + 2 lr + e.
template <int TN, int TM>
struct PPTile {
  static_assert((TN == 6 || TN == 8 || TN == 10) && TM + TN / 2 <= 9 && TM >= 4, "tiles built: 256 x {192, 256, 320}, 320 x 256");
  static constexpr int BM = 64 * TM, BN = 32 * TN, H = TN / 2;
  static constexpr int NQ = TN / 4;
  static constexpr bool PAIR = TN % 4 != 0;
  static constexpr int STAGE = (BM + BN) * 128;        // one k tile of X and W
  static constexpr int SCALES = BM * 4 + 2 * BN * 4;   // int8: sx, sw, bias; half types: bias in the first bytes
  static constexpr int NLOADS = TM + H;                // of a wavefront per k tile
  static constexpr int NSTORES = 4 * TM * (NQ + PAIR);
  static_assert(2 * STAGE + SCALES <= 160 * 1024, "LDS of a CU");
  static_assert(NLOADS + NSTORES < 64, "vmcnt threshold");
  // column of the half that fragment j of a turn holds in its row r
  static SF_DEVICE int column(int turn, int j, int r) {
    if (TN == 6) return 3 * turn + j < 4 ? 4 * r + 3 * turn + j : 64 + 2 * r + 3 * turn + j - 4;  // (the quad's last element is the second turn's)
    return j < 4 ? 64 * turn + 4 * r + j : 64 * NQ + 2 * r + turn;
  }
  // fragment (of both turns) of element e of quad q / of the pair
  static constexpr int quad(int q, int e) { return q * H + e; }
  static constexpr int pair(int e) { return TN == 6 ? 4 + e : e * H + H - 1; }
};

// NT: non-temporal stores
template <class E, int EPI, int TN, bool NT, int TM = 4>
__global__ __launch_bounds__(512, 2) void gemm_pingpong_kernel(PPArgs a) {
  typedef typename E::Out Out;
  using P = PPTile<TN, TM>;
  constexpr bool RES = EPI == PP_RESIDUAL;
  constexpr int H = P::H;
  __shared__ __attribute__((aligned(16))) unsigned char lds[2 * P::STAGE + P::SCALES];
  unsigned char* sc = lds + 2 * P::STAGE;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave & 3, wn = wave >> 2;  // 16 TM rows, half of the columns; wn is also the side that takes turns
  const int lr = lane & 15, lq = lane >> 4;

  // ---- the tiles of this workgroup: XCD x owns a contiguous range, its workgroups walk it side by side -----------
  const unsigned int total = (unsigned int)a.tiles_m * (unsigned int)a.tiles_n;
  const unsigned int xcd = blockIdx.x & 7u, slot = blockIdx.x >> 3, per_x = gridDim.x >> 3;
  const unsigned int chunk = (total + 7u) >> 3;
  const unsigned int first = xcd * chunk + slot;
  const unsigned int last = min(total, (xcd + 1u) * chunk);
  if (slot >= chunk || first >= last) return;  // uniform over the workgroup
  const int nt = (int)((last - first + per_x - 1u) / per_x);
  // Origin of tile ti.  Tiles at the lower and right edge are moved back inside (M >= BM, N >= BN), so that every load is in
  // bounds; the rows and columns that belong to the tile before (skip_m, skip_n) are not stored.
  auto tile_origin = [&](int ti, int& m0, int& n0, int& skip_m, int& skip_n) __attribute__((always_inline)) {
    const unsigned int pid = first + (unsigned int)ti * per_x;
    const unsigned int per_group = (unsigned int)a.group_m * a.tiles_n;
    const unsigned int first_m = (pid / per_group) * a.group_m;
    const unsigned int gsz = min((unsigned int)a.tiles_m - first_m, (unsigned int)a.group_m);
    const unsigned int in_group = pid % per_group;
    m0 = (int)(first_m + in_group % gsz) * P::BM;
    n0 = (int)(in_group / gsz) * P::BN;
    skip_m = max(m0 + P::BM - a.M, 0);
    skip_n = max(n0 + P::BN - a.N, 0);
    m0 -= skip_m;
    n0 -= skip_n;
  };

  typedef __attribute__((address_space(1))) const void* gptr_t;
  typedef __attribute__((address_space(3))) void* lptr_t;
  // ---- tile loads.  A wave instruction fills eight LDS rows of 128 bytes.  16-byte chunk c of LDS row r lives at
  // position c ^ ((r >> 1) & 7): a fragment read (16 rows, four chunks, served in the groups of once_swizzle's note)
  // then touches every bank once.  W rows lie half by half, in it turn by turn, in it fragment by fragment.
  // Of the 4 H eights of W rows that a turn reads, wavefronts 0-3 request LO of the first turn and H - LO of the second each,
  // wavefronts 4-7 the others.
  unsigned int off_x, off_w[H];
  int at_w[H];  // their LDS rows
  constexpr int LO = (H + 1) / 2;
  const int lo = wn == 0 ? LO : H - LO;  // this wavefront's loads for the first turn
#pragma unroll
  for (int i = 0; i < H; ++i) {
    const int turn = i >= lo, v = turn ? (wn == 0 ? wm * (H - LO) : 4 * (H - LO) + wm * LO) + i - lo
                                       : (wn == 0 ? wm * LO : 4 * LO + wm * (H - LO)) + i;
    at_w[i] = (v / (2 * H)) * 16 * TN + turn * 16 * H + (v % (2 * H)) * 8;
  }
  {
    auto chunk_of = [&](int row) __attribute__((always_inline)) { return (lane & 7) ^ ((row >> 1) & 7); };
    const int cx = chunk_of(wave * 8 + (lane >> 3));
    off_x = (unsigned int)(wave * 8 + (lane >> 3)) * a.x_pitch + (unsigned int)((cx >> 2) * a.x_kstep) + (cx & 3) * 16;
#pragma unroll
    for (int i = 0; i < H; ++i) {
      const int half = at_w[i] / (16 * TN), in = at_w[i] % (16 * TN), turn = in / (16 * H), j = in % (16 * H) / 16;
      const int r = in % 16 + (lane >> 3), cw = chunk_of(r);
      const int col = half * 16 * TN + P::column(turn, j, r);
      off_w[i] = (unsigned int)col * a.w_pitch + (unsigned int)((cw >> 2) * a.w_kstep) + (cw & 3) * 16;
    }
  }
  const unsigned char *xk, *wk;  // tile row 0 / column 0 in the k tile that is requested next
  auto load = [&](const unsigned char* base, unsigned int o, int row, int stage) __attribute__((always_inline)) {
    asm volatile("" : "+s"(base));  // uniform base, 32-bit lane offset
    asm volatile("" : "+v"(o));
    __builtin_amdgcn_global_load_lds((gptr_t)(base + o), (lptr_t)(lds + stage + row * 128), 16, 0, 0);
  };
  auto load_x = [&](int stage) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < TM; ++i) load(xk + (int64_t)(64 * i) * a.x_pitch, off_x, (wave + 8 * i) * 8, stage);
  };
  auto load_w = [&](int turn, int stage) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < H; ++i) {
      const bool mine = H % 2 == 0 ? (i >= LO) == (turn == 1) : i < H - LO ? turn == 0 : i >= LO ? turn == 1 : (i >= lo) == (turn == 1);
      if (mine) load(wk, off_w[i], P::BM + at_w[i], stage);
    }
  };
  int m0, n0, skip_m, skip_n, lt = 0, lk = 0;
  auto first_ktile = [&]() __attribute__((always_inline)) {
    int m, n, sm, sn;
    tile_origin(lt, m, n, sm, sn);
    xk = a.x + (int64_t)m * a.x_pitch;
    wk = a.w + (int64_t)n * a.w_pitch;
  };
  first_ktile();
  tile_origin(0, m0, n0, skip_m, skip_n);
  auto next_ktile = [&]() __attribute__((always_inline)) {
    xk += 2 * a.x_kstep;
    wk += 2 * a.w_kstep;
    if (++lk == a.nk) {
      // the first k tiles of the next tile (behind the last one: its own again, read by nobody)
      lk = 0;
      if (lt + 1 < nt) ++lt;
      first_ktile();
    }
  };
  // scales and bias of the tile, 64 lanes of 4 bytes an instruction, the same number for every wavefront (some repeated)
  auto load_scales = [&]() __attribute__((always_inline)) {
    if constexpr (E::SCALED) {
      constexpr int XS = P::BM / 64, WS = P::BN / 64, SLICES = XS + 2 * WS;
#pragma unroll
      for (int e = 0; e < (SLICES + 7) / 8; ++e) {
        const int s = (wave + 8 * e) % SLICES;
        const int part = s < XS ? 0 : s < XS + WS ? 1 : 2, q = (part == 0 ? s : (s - XS) % WS) * 64;
        const float* src = part == 0 ? a.sx + m0 : (part == 1 || !a.bias ? a.sw : reinterpret_cast<const float*>(a.bias)) + n0;
        const int dst = (part == 0 ? 0 : part == 1 ? P::BM * 4 : P::BM * 4 + P::BN * 4) + q * 4;
        __builtin_amdgcn_global_load_lds((gptr_t)(src + q + lane), (lptr_t)(sc + dst), 4, 0, 0);
      }
    } else {
      // columns in pairs (N is even); 320 columns are two and a half slices, 192 one and a half: they overlap
      const int q = P::BN == 320 ? (wave % 3) * 96 : (wave & 1) * (P::BN - 128);
      if (a.bias) __builtin_amdgcn_global_load_lds((gptr_t)(reinterpret_cast<const unsigned short*>(a.bias) + n0 + q + 2 * lane), (lptr_t)(sc + q * 2), 4, 0, 0);
    }
  };

  // ---- fragments and products: rows 16 i + lr of the wavefront's 16 TM, columns through j --------------------------
  const int frag = (lq ^ ((lr >> 1) & 7)) * 16;
  const int x_off[2] = {(wm * 16 * TM + lr) * 128 + frag, (wm * 16 * TM + lr) * 128 + (frag ^ 64)};
  const int w_off[2] = {(P::BM + wn * 16 * TN + lr) * 128 + frag, (P::BM + wn * 16 * TN + lr) * 128 + (frag ^ 64)};
  i32x4 fx[2][TM], fw[2][H];
  typename E::acc_t acc[TM][TN];
  auto read = [&](int turn, int stage) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      if (turn == 0)
#pragma unroll
        for (int i = 0; i < TM; ++i) fx[k][i] = *reinterpret_cast<const i32x4*>(lds + stage + x_off[k] + i * 2048);
#pragma unroll
      for (int j = 0; j < H; ++j) fw[k][j] = *reinterpret_cast<const i32x4*>(lds + stage + w_off[k] + (turn * H + j) * 2048);
    }
  };
  auto multiply = [&](auto turn, auto zero) __attribute__((always_inline)) {
    constexpr int T = decltype(turn)::value;
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int jj = 0; jj < H; ++jj) {
          const int j = i & 1 ? H - 1 - jj : jj;  // one operand stays from each instruction to the next
          const typename E::acc_t z = {};
          acc[i][T * H + j] = E::mma(fx[k][i], fw[k][j], decltype(zero)::value && k == 0 ? z : acc[i][T * H + j]);
        }
    // (the products are pure values to the compiler; this pins them to their turn)
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < H; ++j) asm volatile("" : "+v"(acc[i][T * H + j]));
    __builtin_amdgcn_s_setprio(0);
  };
  auto meet = [&]() __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };

  // ---- output: rows 16 (TM wm + i) + 4 lq + r, quads and pair of columns from col0 on ------------------------------
  typedef __attribute__((address_space(1))) unsigned char* gbyte_t;
  const int col0 = wn * 16 * TN;
  auto lane_again = [&]() __attribute__((always_inline)) {  // (made again at every use: kept, it would be spilled)
    int l = lane;
    asm volatile("" : "+v"(l));
    return l;
  };
  // Walks the rows of the tile at `tile` in the order in which they are finished: a uniform base that moves by the pitch and a 32-bit
  // lane offset made once per tile (as loop invariants of the kernel the offsets of all rows would be kept in registers).
  struct Walk {
    const unsigned char* p;
    unsigned int pitch, quad, pair;
    SF_DEVICE gbyte_t at(int g) const { return (gbyte_t)(uintptr_t)p + (g < P::NQ ? quad : pair) + 128 * g; }
    SF_DEVICE void down(int rows) {
      p += rows * pitch;
      asm volatile("" : "+s"(p));
    }
  };
  auto walk = [&](const unsigned short* tile, int64_t ld, int i) __attribute__((always_inline)) {
    const int l = lane_again();
    Walk w;
    w.pitch = (unsigned int)ld * 2u;
    asm volatile("" : "+s"(w.pitch));
    w.p = reinterpret_cast<const unsigned char*>(tile + col0) + (int64_t)(wm * 16 * TM + 16 * i) * w.pitch;
    asm volatile("" : "+s"(w.p));
    w.quad = (unsigned int)(4 * (l >> 4)) * w.pitch + 8 * (l & 15);
    asm volatile("" : "+v"(w.quad));
    w.pair = P::PAIR ? w.quad - 4 * (l & 15) : 0;
    return w;
  };
  typedef __attribute__((address_space(1))) u32x2* gquad_t;
  typedef __attribute__((address_space(1))) unsigned int* gpair_t;
  // residual values of the first row group: requested in the last k tile (where the operands leave registers for them)
  constexpr bool AHEAD = RES && TM == 4;
  constexpr int EARLY = P::NQ * 4 + (P::PAIR ? 4 : 0);
  u32x2 res[RES ? TM : 1][4][P::NQ];
  unsigned int res_pair[RES && P::PAIR ? TM : 1][4];
  auto residual_walk = [&](int i) __attribute__((always_inline)) { return walk(a.residual + (int64_t)m0 * a.ld_res + n0, a.ld_res, i); };
  auto load_residual = [&](Walk& w, int i) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
#pragma unroll
      for (int g = 0; g < P::NQ; ++g) res[i][r][g] = *(gquad_t)w.at(g);
      if constexpr (P::PAIR) res_pair[i][r] = *(gpair_t)w.at(P::NQ);
      w.down(r < 3 ? 1 : 13);
    }
  };
  // Both sides finish between the same two barriers, the lower one ahead by what it converts under the upper one's last products: two
  // wavefronts share a SIMD's vector unit.  Where the conversion is an add and half a pack per value, they finish one behind the other,
  // each under a turn of the other's products.
  constexpr bool TOGETHER = E::SCALED || EPI != PP_PLAIN;
  auto finish = [&](auto whole) __attribute__((always_inline)) {
    constexpr bool FULL = decltype(whole)::value;
    const int l = lane_again(), lr = l & 15, lq = l >> 4;
    Walk from = {};
    if constexpr (RES) {
      from = residual_walk(AHEAD ? 1 : 0);
      if constexpr (!AHEAD) load_residual(from, 0);
      load_residual(from, 1);
      load_residual(from, 2);
      __builtin_amdgcn_sched_barrier(0);
    }
    // column scales and bias of the quads and the pair
    float sw[P::NQ + 1][4], bias[P::NQ + 1][4];
#pragma unroll
    for (int g = 0; g < P::NQ + P::PAIR; ++g) {
      const int n = g < P::NQ ? 4 : 2, col = col0 + 64 * g + n * lr;
#pragma unroll
      for (int e = 0; e < n; ++e) {
        if constexpr (E::SCALED) {
          sw[g][e] = reinterpret_cast<const float*>(sc + P::BM * 4 + col * 4)[e];
          bias[g][e] = a.bias ? reinterpret_cast<const float*>(sc + P::BM * 4 + P::BN * 4 + col * 4)[e] : 0.f;
        } else {
          const unsigned int b = a.bias ? reinterpret_cast<const unsigned int*>(sc + col * 2)[e >> 1] : 0u;
          bias[g][e] = e & 1 ? Out::hi(b) : Out::lo(b);
        }
      }
    }
    Walk to = walk(a.out + (int64_t)m0 * a.ldo + n0, a.ldo, 0);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      if constexpr (RES)
        if (i >= 1 && i + 2 < TM) load_residual(from, i + 2);  // (three of the row groups at a time: registers)
      f32x4 sx;
      if constexpr (E::SCALED) sx = *reinterpret_cast<const f32x4*>(sc + (wm * 16 * TM + 16 * i + 4 * lq) * 4);
      // two adjacent columns of row r, rounded; group g, elements e and e + 1, plus the residual pair v
      auto two = [&](int r, int g, int e, unsigned int v) __attribute__((always_inline)) {
        float y[2];
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          const auto s = acc[i][g < P::NQ ? P::quad(g, e + c) : P::pair(e + c)][r];
          if constexpr (E::SCALED) {
            // three separately rounded fp32 operations (no fused multiply-add)
            float t = (float)s * sx[r];
            t = t * sw[g][e + c];
            y[c] = t + bias[g][e + c];
          } else {
            y[c] = s + bias[g][e + c];
          }
        }
        unsigned int o = Out::pack2(y[0], y[1]);
        if constexpr (EPI == PP_GELU) {
          // activation of the rounded Linear output, as a separate GELU would see it
          static_assert(!E::SCALED, "int8 products with GELU are other kernels'");
          o = Out::pack2(gelu_value(Out::lo(o)), gelu_value(Out::hi(o)));
        }
        if constexpr (RES) o = Out::pack2(Out::lo(o) + Out::lo(v), Out::hi(o) + Out::hi(v));
        return o;
      };
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = wm * 16 * TM + 16 * i + 4 * lq + r;
#pragma unroll
        for (int g = 0; g < P::NQ; ++g) {
          const u32x2 v = RES ? res[RES ? i : 0][r][g] : u32x2{0u, 0u};
          const u32x2 o = {two(r, g, 0, v[0]), two(r, g, 2, v[1])};
          const gquad_t dst = (gquad_t)to.at(g);
          if (FULL || (row >= skip_m && col0 + 64 * g + 4 * lr >= skip_n)) {
            if (NT) __builtin_nontemporal_store(o, dst);
            else *dst = o;
          }
        }
        if constexpr (P::PAIR) {
          const unsigned int o = two(r, P::NQ, 0, RES ? res_pair[RES ? i : 0][r] : 0u);
          const gpair_t dst = (gpair_t)to.at(P::NQ);
          if (FULL || (row >= skip_m && col0 + 64 * P::NQ + 2 * lr >= skip_n)) {
            if (NT) __builtin_nontemporal_store(o, dst);
            else *dst = o;
          }
        }
        to.down(r < 3 ? 1 : 13);
        __builtin_amdgcn_sched_barrier(0);  // keep the conversion narrow
      }
      if (TOGETHER && i == 0 && wn == 0) meet();
    }
  };

  // ---- prologue: k tile 0, and of k tile 1 what the first turn of a k tile needs ---------------------------------
  load_x(0);
  load_w(0, 0);
  load_w(1, 0);
  next_ktile();
  load_x(P::STAGE);
  load_w(0, P::STAGE);
  pp_wait<P::NLOADS>();  // the X rows and first columns of k tile 0
  meet();
  if (wn == 1) meet();  // from here on the upper half is one turn behind

  int stage = 0;
  // One k tile.  First turn: X rows and its columns are read; the second turn's columns of the k tile behind this one are
  // requested (their place was read in the turn before this).  Second turn: its columns read; X rows and the first
  // turn's columns of the k tile two behind requested.  Either wait leaves a k tile's worth of the youngest loads in flight: what
  // the next turn of either half reads was requested before those.  EXTRA other operations (a whole tile's stores in front of
  // its first k tile, residual values ahead of the last) are younger than what is waited for, if `extra` says that they were issued.
  auto ktile = [&](auto zero, auto extra_n, bool extra) __attribute__((always_inline)) {
    using T0 = std::integral_constant<int, 0>;
    using T1 = std::integral_constant<int, 1>;
    constexpr int EXTRA = decltype(extra_n)::value;
    constexpr bool LAST = AHEAD && !decltype(zero)::value && EXTRA > 0;
    const int other = stage ^ P::STAGE;
    read(0, stage);
    load_w(1, other);
    next_ktile();
    if constexpr (LAST) {
      Walk w = residual_walk(0);
      load_residual(w, 0);
    }
    if (EXTRA > 0 && extra) pp_wait<P::NLOADS + EXTRA>();
    else pp_wait<P::NLOADS>();
    meet();
    multiply(T0{}, zero);
    meet();
    read(1, stage);
    load_x(stage);
    load_w(0, stage);
    if constexpr (decltype(zero)::value) load_scales();
    if (EXTRA > 0 && extra) pp_wait<P::NLOADS + EXTRA>();
    else pp_wait<P::NLOADS>();
    meet();
    multiply(T1{}, zero);
    meet();
    stage = other;
  };
  using Yes = std::true_type;
  using No = std::false_type;
  bool stored = false;  // a whole tile's stores are on their way
  for (int ti = 0; ti < nt; ++ti) {
    ktile(Yes{}, std::integral_constant<int, P::NSTORES>{}, stored);
    for (int k = 1; k < a.nk - (AHEAD ? 1 : 0); ++k) ktile(No{}, std::integral_constant<int, 0>{}, false);
    if constexpr (AHEAD) ktile(No{}, std::integral_constant<int, EARLY>{}, true);
    stored = skip_m == 0 && skip_n == 0;
    if (stored) finish(Yes{});
    else finish(No{});
    if (TOGETHER && wn == 1) meet();
    if (ti + 1 < nt) tile_origin(ti + 1, m0, n0, skip_m, skip_n);
  }
  if (wn == 0) meet();
  __builtin_amdgcn_s_waitcnt(0x0070);  // the last loads land before the LDS is given back
}

// ---- outputs the GPU holds once: 128-row tiles, K shared between the sides ------------------------------------------
// An image's products onto few columns: 4096 rows and 768, 1024 or 1280 columns are exactly 256 tiles of 128 x {96, 128, 160}.  The
// wavefronts 0-3 multiply the lower 64 bytes of every k tile, 4-7 the upper ones; each holds 64 rows and half
// of the columns, and the two sides' sums meet in LDS at the end, where each side finishes half of the rows.  So few columns leave a
// wavefront registers for two k tiles' fragments: it reads the next ones, and requests a k tile, between its products, with one barrier per k tile.
// (The sides by turns as above, one multiplying while the other read, were two barriers and two latencies of the LDS around 320 cycles of
// products.  bf16 with the residual, us, by turns / so, operands in the caches: 4096 x 5120 -> 1280 53.3 / 48.1, 4096 x 4096 -> 1024 36.5 / 32.4, 4096 x 3072 -> 768 27.0 / 22.0,
// 4096 x 1280 -> 1280 18.3 / 17.4, 4096 x 768 -> 768 9.9 / 8.5.)  What bounds it now is how the operands come: 288 rows of 128 bytes for
// 640 cycles of products are 58 of the 64 bytes per clock that a CU takes in.
// Long loops' weights, which come from HBM in an encoder whose weights exceed the last-level cache, are touched once, a line by each
// thread of the grid, row by row: the loop asks all CUs' rows for one line each at a time, and waited for HBM at every k tile
// (weights and rows not in the L2s: 4096 x 5120 -> 1280 60.2 / 50.3, 4096 x 4096 -> 1024 39.0 / 34.0, 4096 x 3072 -> 768 29.8 / 25.0, 2048 x 5120 -> 1280 45.1 / 36.2; all of it in
// them: 49.0 / 49.0, 32.4 / 33.0, 21.9 / 22.4, 31.5 / 32.6; a ViT-H image with bf16 Linears 6640 / 6200, ViT-L 3810 / 3640, ViT-B 1650 / 1600).  At 20 k tiles and fewer it is
// level or slower (4096 x 1280 -> 1280 20.7 / 21.3), and where the grid has fewer threads than W lines it costs more than the part that is touched
// saves (touched / not, times as long as by turns: 113 products out of HBM 0.988 / 0.981, the worst twentieth 1.04 / 1.02; 21 out of the caches 0.885 / 0.850; a second
// line a thread 1.02 times as long as touched): nothing is touched there.
// Library's product + residual in the next LayerNorm / by turns + LayerNorm: 4096 x 5120 -> 1280 61.3 / 55.9, 4096 x 1280 -> 1280
// 31.1 / 23.6, 4096 x 768 -> 768 31.6 / 18.6.  (int8 keeps gemm_i8_once.hip.)
template <int TN>
struct PPSplitTile {
  static_assert(TN >= 3 && TN <= 5, "widths built: 96, 128, 160");
  static constexpr int BM = 128, BN = 32 * TN;
  static constexpr int STAGE = (BM + BN) * 128;
  static constexpr int NST = TN == 3 ? 5 : 4;
  static constexpr int BIAS = 512;                    // bytes, two requests of 64 lanes
  static constexpr int LO = (TN + 1) / 2;             // loads of W per k tile for wavefronts 0-3 (two of X); 4-7: TN - LO
  static constexpr int N0 = TN == 3 ? 2 : 4;          // adjacent columns of a lane; the others (TN - N0: none or one) follow 16 N0 further on
  static_assert(NST * STAGE + BIAS <= 160 * 1024 && 16 * TN * 1024 <= NST * STAGE, "LDS of a CU");
};

template <class E, int EPI, int TN>
__global__ __launch_bounds__(512, 2) void gemm_pingpong_split_kernel(PPArgs a) {
  typedef typename E::Out Out;
  using P = PPSplitTile<TN>;
  constexpr bool RES = EPI == PP_RESIDUAL, ONE = TN > P::N0;
  static_assert(!E::SCALED, "half types");
  constexpr int NST = P::NST, N0 = P::N0, NP = N0 / 2;  // NP: pairs of a lane's adjacent columns
  __shared__ __attribute__((aligned(16))) unsigned char lds[NST * P::STAGE + P::BIAS];
  unsigned char* sc = lds + NST * P::STAGE;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int side = wave >> 2, wm = (wave >> 1) & 1, wn = wave & 1;
  const int lr = lane & 15, lq = lane >> 4;
  const unsigned int total = (unsigned int)a.tiles_m * (unsigned int)a.tiles_n;
  const unsigned int pid = xcd_contiguous_id(blockIdx.x, total);
  if (pid >= total) return;  // uniform over the workgroup
  const unsigned int per_group = (unsigned int)a.group_m * a.tiles_n;
  const unsigned int first_m = (pid / per_group) * a.group_m;
  const unsigned int gsz = min((unsigned int)a.tiles_m - first_m, (unsigned int)a.group_m);
  const unsigned int in_group = pid % per_group;
  int m0 = (int)(first_m + in_group % gsz) * P::BM, n0 = (int)(in_group / gsz) * P::BN;
  // tiles at the edges are moved back inside (M >= 128, N >= BN), see above
  const int skip_m = max(m0 + P::BM - a.M, 0), skip_n = max(n0 + P::BN - a.N, 0);
  m0 -= skip_m;
  n0 -= skip_n;

  typedef __attribute__((address_space(1))) const void* gptr_t;
  typedef __attribute__((address_space(3))) void* lptr_t;
  typedef __attribute__((address_space(1))) unsigned char* gbyte_t;
  typedef __attribute__((address_space(1))) unsigned int* gword_t;

  // ---- output geometry: rows wm * 64 + 32 side + 16 i + 4 lq + r; the lane's adjacent columns, and of the column behind them
  // the pair (even, odd) of row r that even lanes store, of row r + 1 that odd ones do
  const int col0 = wn * 16 * TN + N0 * lr, col1 = wn * 16 * TN + 16 * N0 + (lr & ~1), row0 = wm * 64 + 32 * side + 4 * lq;
  auto at = [&](const unsigned short* p, int64_t ld, int i, int r, bool one) __attribute__((always_inline)) {
    const int row = row0 + 16 * i + r + (one ? lr & 1 : 0);
    return (gbyte_t)(uintptr_t)(p + (int64_t)m0 * ld + n0) + (unsigned int)((row * (int)ld + (one ? col1 : col0)) * 2);
  };
  unsigned int res[RES ? 2 : 1][4][NP], res_one[RES && ONE ? 2 : 1][2];
  if constexpr (RES) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if constexpr (NP == 2) {
          const u32x2 v = *(__attribute__((address_space(1))) u32x2*)at(a.residual, a.ld_res, i, r, false);
          res[i][r][0] = v[0];
          res[i][r][NP - 1] = v[1];
        } else {
          res[i][r][0] = *(gword_t)at(a.residual, a.ld_res, i, r, false);
        }
      }
      if constexpr (ONE) {
        res_one[i][0] = *(gword_t)at(a.residual, a.ld_res, i, 0, true);
        res_one[i][1] = *(gword_t)at(a.residual, a.ld_res, i, 2, true);
      }
    }
    __builtin_amdgcn_sched_barrier(0);  // the oldest operations in flight: no threshold below counts them
  }

  // ---- bias, 64 lanes of 4 bytes an instruction ----------------------------------------------------------------------
  if (a.bias) {
    // columns in pairs (N is even)
    const int q = (wave & 1) * 128;
    __builtin_amdgcn_global_load_lds((gptr_t)(reinterpret_cast<const unsigned short*>(a.bias) + n0 + min(q + 2 * lane, P::BN - 2)), (lptr_t)(sc + q * 2), 4, 0, 0);
  }

  // ---- tile loads: eights of rows as above.  Every wavefront two of X; of W 0-3 take LO each, 4-7 the others ----------
  unsigned int off_x, off_w[P::LO];
  int at_w[P::LO];
  const int nw = side == 0 ? P::LO : TN - P::LO;
  {
    const int r = wave * 8 + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
    off_x = (unsigned int)r * a.x_pitch + (unsigned int)((c >> 2) * a.x_kstep) + (c & 3) * 16;
#pragma unroll
    for (int i = 0; i < P::LO; ++i) {
      // LDS row at_w: half by half, fragment by fragment; fragment j of a lane row is column N0 lr + j, or 16 N0 + lr
      at_w[i] = min(side == 0 ? (wave & 3) * P::LO + i : 4 * P::LO + (wave & 3) * (TN - P::LO) + i, 4 * TN - 1) * 8;
      const int in = at_w[i] % (16 * TN), j = in / 16, rr = in % 16 + (lane >> 3), cw = (lane & 7) ^ ((rr >> 1) & 7);
      const int col = at_w[i] / (16 * TN) * 16 * TN + (j < N0 ? N0 * rr + j : 16 * N0 + rr);
      off_w[i] = (unsigned int)col * a.w_pitch + (unsigned int)((cw >> 2) * a.w_kstep) + (cw & 3) * 16;
    }
  }
  const unsigned char* xk = a.x + (int64_t)m0 * a.x_pitch;
  const unsigned char* wk = a.w + (int64_t)n0 * a.w_pitch;
  auto load = [&](const unsigned char* base, unsigned int o, int row, int stage) __attribute__((always_inline)) {
    asm volatile("" : "+s"(base));
    asm volatile("" : "+v"(o));
    __builtin_amdgcn_global_load_lds((gptr_t)(base + o), (lptr_t)(lds + stage + row * 128), 16, 0, 0);
  };
  // load l of this wavefront's 2 + nw for a k tile
  auto fill = [&](int l, int stage) __attribute__((always_inline)) {
    if (l < 2) load(xk + (int64_t)(64 * l) * a.x_pitch, off_x, (wave + 8 * l) * 8, stage);
    else if (l - 2 < TN - P::LO || l - 2 < nw) load(wk, off_w[l < 2 ? 0 : l - 2], P::BM + at_w[l < 2 ? 0 : l - 2], stage);
  };
  auto advance = [&]() __attribute__((always_inline)) {
    xk += 2 * a.x_kstep;
    wk += 2 * a.w_kstep;
  };
  // at most `tiles` k tiles of this wavefront's loads still in flight; LDS reads done
  auto arrive = [&](auto tiles) __attribute__((always_inline)) {
    constexpr int T = decltype(tiles)::value;
    if (P::LO == TN - P::LO || side == 0) pp_wait<T * (2 + P::LO)>();
    else pp_wait<T * (2 + TN - P::LO)>();
  };
  auto meet = [&]() __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };

  const int frag = ((lq + 4 * side) ^ ((lr >> 1) & 7)) * 16;
  const int x_off = (wm * 64 + lr) * 128 + frag, w_off = (P::BM + wn * 16 * TN + lr) * 128 + frag;
  typename E::acc_t acc[4][TN];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = typename E::acc_t{};
  const int nk = a.nk;  // >= NST
#pragma unroll
  for (int p = 0; p < NST; ++p) {
#pragma unroll
    for (int l = 0; l < 2 + P::LO; ++l) fill(l, p * P::STAGE);
    advance();
  }
  unsigned int touched = 0;
  if (nk >= 32 && (unsigned int)a.N * nk <= total * 512u) {  // this thread's line of W
    const unsigned int line = min(pid * 512u + tid, (unsigned int)a.N * nk - 1u), row = line / (unsigned int)nk;
    touched = *(gword_t)((gbyte_t)(uintptr_t)a.w + (int64_t)row * a.w_pitch + (line - row * nk) * 128);
  }
  i32x4 fx[2][4], fw[2][TN];
  constexpr int READS = 4 + TN;
  auto read = [&](int buf, int r, int stage) __attribute__((always_inline)) {
    if (r < TN) fw[buf][r < TN ? r : 0] = *reinterpret_cast<const i32x4*>(lds + stage + w_off + r * 2048);
    else fx[buf][r < TN ? 0 : r - TN] = *reinterpret_cast<const i32x4*>(lds + stage + x_off + (r - TN) * 2048);
  };
  // k tile t: its products; between them its stage, whose fragments every wavefront holds, is requested anew for t + NST (`more`), and t + 1's
  // fragments are read (`next`); t + 2 is awaited
  auto ktile = [&](auto buf, auto more, auto next, int here, int ahead) __attribute__((always_inline)) {
    constexpr int B = decltype(buf)::value;
    int slot = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int jj = 0; jj < TN; ++jj, ++slot) {
        const int j = i & 1 ? TN - 1 - jj : jj;
        acc[i][j] = E::mma(fx[B][i], fw[B][j], acc[i][j]);
        __builtin_amdgcn_sched_barrier(0);
        if (decltype(next)::value && slot < READS) read(1 - B, slot, ahead);
        if (decltype(more)::value && slot >= 4 * TN - 2 - P::LO) fill(slot - (4 * TN - 2 - P::LO), here);
        __builtin_amdgcn_sched_barrier(0);
      }
    if constexpr (decltype(more)::value) {
      advance();
      arrive(std::integral_constant<int, NST - 2>{});
    } else {
      pp_wait<0>();
    }
    if constexpr (decltype(next)::value) meet();
  };
  using B0 = std::integral_constant<int, 0>;
  using B1 = std::integral_constant<int, 1>;
  using Yes = std::true_type;
  using No = std::false_type;
  auto up = [&](int s) __attribute__((always_inline)) { return s == (NST - 1) * P::STAGE ? 0 : s + P::STAGE; };
  auto begin = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < READS; ++r) read(buf, r, 0);
    arrive(std::integral_constant<int, NST - 2>{});
    meet();
  };
  int here = 0, left = nk;
  arrive(std::integral_constant<int, NST - 1>{});
  meet();
  // two at a time, so that the fragments' two places are known; an odd one first
  if ((nk - NST) & 1) {
    begin(1);
    ktile(B1{}, Yes{}, Yes{}, here, up(here));
    here = up(here);
    --left;
  } else {
    begin(0);
  }
  for (; left > NST; left -= 2) {
    const int there = up(here);
    ktile(B0{}, Yes{}, Yes{}, here, there);
    here = up(there);
    ktile(B1{}, Yes{}, Yes{}, there, here);
  }
#pragma unroll
  for (int p = 0; p < NST; ++p) {
    if (p == NST - 1) p & 1 ? ktile(B1{}, No{}, No{}, here, here) : ktile(B0{}, No{}, No{}, here, here);
    else p & 1 ? ktile(B1{}, No{}, Yes{}, here, up(here)) : ktile(B0{}, No{}, Yes{}, here, up(here));
    here = up(here);
  }

  asm volatile("" : : "v"(touched));
  // ---- the sides' sums meet: side 0 finishes row groups 0 and 1, side 1 the other two -----------------------------------
  typedef typename E::acc_t acc_t;
  acc_t* red = reinterpret_cast<acc_t*>(lds) + (wave & 3) * 2 * TN * 64 + lane;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const acc_t upper = acc[2 + i][j], lower = acc[i][j];  // (values: a choice between places would put the sums into memory)
      acc[i][j] = side == 0 ? lower : upper;
      red[side * 8 * TN * 64 + (i * TN + j) * 64] = side == 0 ? upper : lower;
    }
  pp_wait<0>();
  meet();
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] += red[(1 - side) * 8 * TN * 64 + (i * TN + j) * 64];

  // ---- output ----------------------------------------------------------------------------------------------------------
  const bool full = skip_m == 0 && skip_n == 0;
  float bias[TN];
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int col = j < N0 ? col0 + j : wn * 16 * TN + 16 * N0 + lr;
    bias[j] = a.bias ? Out::lo((unsigned int)reinterpret_cast<const unsigned short*>(sc)[col]) : 0.f;
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    auto value = [&](int j, int r) __attribute__((always_inline)) { return acc[i][j][r] + bias[j]; };
    auto last_step = [&](unsigned int o, unsigned int v) __attribute__((always_inline)) {
      if constexpr (EPI == PP_GELU) o = Out::pack2(gelu_value(Out::lo(o)), gelu_value(Out::hi(o)));
      if constexpr (RES) o = Out::pack2(Out::lo(o) + Out::lo(v), Out::hi(o) + Out::hi(v));
      return o;
    };
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      unsigned int o[NP];
#pragma unroll
      for (int p = 0; p < NP; ++p) o[p] = last_step(Out::pack2(value(2 * p, r), value(2 * p + 1, r)), RES ? res[RES ? i : 0][r][p] : 0u);
      const gbyte_t dst = at(a.out, a.ldo, i, r, false);
      if (full || (row0 + 16 * i + r >= skip_m && col0 >= skip_n)) {
        if constexpr (NP == 2) *(__attribute__((address_space(1))) u32x2*)dst = u32x2{o[0], o[NP - 1]};
        else *(gword_t)dst = o[0];
      }
    }
    if constexpr (ONE) {
#pragma unroll
      for (int r = 0; r < 4; r += 2) {
        // lanes 2 n and 2 n + 1 hold columns 2 n, 2 n + 1 of both rows: the even one collects row r, the odd one row r + 1
        const float a0 = value(TN - 1, r), a1 = value(TN - 1, r + 1);
        const float other = __shfl_xor(lr & 1 ? a0 : a1, 1, 64);
        const unsigned int o = last_step(lr & 1 ? Out::pack2(other, a1) : Out::pack2(a0, other), RES ? res_one[RES ? i : 0][r >> 1] : 0u);
        const int row = row0 + 16 * i + r + (lr & 1);
        if (full || (row >= skip_m && col1 >= skip_n)) *(gword_t)at(a.out, a.ldo, i, r, true) = o;
      }
    }
  }
}

// ---- host side ---------------------------------------------------------------------------------------------------------
// Time of a launch in units of one 16-column fragment of 64 rows for one k tile: rounds of the CUs, each as long as its k tiles and a start
// and an end worth eight more of them, a tile two to three fragments more expensive than its columns.  The tile with the
// least; `used`: the share of those CU-cycles that makes output.
// us, 256 / 320 columns: int8 4096 x 1280 -> 5120 (two rounds / one) 33.1 / 27.6, 8192 x 1280 -> 5120 (three / two) 53.5 / 52.1, 32768 x 1280 -> 3840 (eight /
// six) 151 / 139, 24576 x 1280 -> 5120 (eight / six) 145 / 138, but 24576 x 1280 -> 3840 (six / five) 110.5 / 112.4, at equal numbers of columns
// per CU 65536 x 1280 -> 3840 276 / 275; loops under ten k tiles pay more for the wide tile's end: 24576 x 768 -> 3072 (five / four)
// 64.4 / 70.3, 24576 x 1024 -> 3072 (five / four) 77.7 / 81.3, 12288 x 1024 -> 3072 (three / two) 44.4 / 42.1.  bf16 12288 x 1280 -> 5120 (four / three) 141 / 134,
// 24576 x 1280 -> 5120 276 / 261, but 24576 x 1024 -> 3072 121 / 124.
// `narrow`, unless 0: the price of 192 columns, where the caller builds them: half types 8.1 (with GELU 8.4: a round more of them than of wider tiles, 0.97 of the price at 8.1, was 1.00 times as long over 15 products, 23243 x 5120 -> 1408
// in three rounds for two 263 / 282; without GELU 0.976 over 20), int8 8.7 (both less in the first rounds), with the residual 9.  256 / 192, rounds, bf16:
// 4096 x 768 -> 3072 with GELU (one / one) 27.0 / 23.9, 4096 x 1024 -> 3072 25.9 / 23.7, 8192 x 768 -> 3072 with GELU (two / two) 45.6 / 40.0, 28672 x 1024 ->
// 3072 (six / seven) 141 / 133; but 20480 x 1024 -> 3072 (four / five) 96.7 / 96.9, 32768 x 768 -> 3072 with GELU (six / eight) 145 / 152; 320 / 192: 12288 x 1024 -> 3072 (two /
// three) 61.0 / 58.5, but 24576 x 768 -> 2304 (three / five) 73.1 / 73.4.  int8, the smaller members / 192: 8192 x 768 -> 3072 25.0 / 22.7, 8192 x 1024 -> 3072 29.6 / 26.6, 6144 x
// 1280 -> 3840 34.1 / 29.1, 4096 x 1024 -> 3072 18.3 / 16.9; 320 / 192 (two / three) 16384 x 768 -> 2304 32.6 / 31.0, 12288 x 1024 -> 3072 38.0 / 36.0; but 256 / 192 (six / seven)
// 28672 x 768 -> 3072 67.6 / 71.4, (five / six) 32768 x 768 -> 2304 58.8 / 60.1.
// With the residual, int8: 16384 x 5120 -> 1280 (two / two) 108 / 96, 12288 x 3072 -> 768 (one / one) 36.5 / 32.6, 8192 x 5120 -> 1280 52.5 / 50.6;
// but 320 rows / 192 columns (one / two) 24576 x 3072 -> 768 50.2 / 59.2.
// The residual's registers leave no room for 320 columns, but for 320 rows, which few columns and many rows fill better.  256 / 320
// rows: int8 20480 x 4096 -> 1024 (two rounds / one) 89.2 / 67.6, 24576 x 3072 -> 768 69.6 / 51.0, 57344 x 4096 -> 1024 (four / three) 215 /
// 203, 57344 x 5120 -> 1280 (five / four) 315 / 313, bf16 696 / 622; in equal rounds 16384 x 4096 -> 1024 bf16 103 / 112.
struct PPChoice {
  int tm, tn;
  int64_t rounds;
  double used;
};
static inline PPChoice pp_choose(int64_t M, int N, int nk, bool residual, double narrow = 0.0) {
  PPChoice best = {0, 0, 0, 0.0};
  double least = 0.0;
  auto candidate = [&](int tm, int tn, double fragments) {
    if (N < 32 * tn || M < 64 * tm) return;
    const int64_t rounds = (((M + 64 * tm - 1) / (64 * tm)) * ((N + 32 * tn - 1) / (32 * tn)) + 255) / 256;
    const double cost = (double)rounds * fragments * (nk + 8);
    if (best.tn == 0 || cost < least) {
      best = PPChoice{tm, tn, rounds, (double)M * N / (256.0 * rounds * 64 * tm * 32 * tn)};
      least = cost;
    }
  };
  candidate(4, 8, 10.0);
  if (residual) candidate(5, 8, 12.4);
  else candidate(4, 10, nk < 10 ? 13.2 : 12.5);
  if (narrow > 0.0) candidate(4, 6, narrow);
  return best;
}

// what the kernels take beside the shape rules of their callers: 32-bit offsets inside a tile
static inline bool pp_addressable(const PPArgs& a) { return a.ldo < (1ll << 22) && a.ld_res < (1ll << 22) && a.nk >= 5; }

static inline unsigned int pp_grid(const PPArgs& a) { return (unsigned int)min((int64_t)256, ((int64_t)a.tiles_m * a.tiles_n + 7) / 8 * 8); }

}  // namespace samfast
