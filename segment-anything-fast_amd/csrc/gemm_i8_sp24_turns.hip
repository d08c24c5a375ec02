// int8 GEMM with a 2:4-sparse weight operand, outputs of whole rounds of large tiles: 256 tokens and 256 or 320 channels, one resident
// workgroup of eight wavefronts per CU, two per SIMD that take turns at the matrix pipe, as the dense gemm_pingpong_kernel does.
//
// What bounds it is memory, not products: at 131072 x 1280 -> 5120 (600 us, 455 on zeros) 304 on zeros are the loop with its loads, most of the
// rest 1.3 GB of output; without the products it takes the same time, without the loads 160 less (timings of patched copies that are not
// kept, counters beside them).  So the choices are about bytes and about the units they pass:
//   * 256 x 320 tiles: 58368 bytes of operands per 1280 cycles of products, 45.6 a clock (46.4 with the padded piece of the index words), for 72
//     in the 128-token kernel and 52 in 256 x 256 (taken where 320 channels fit badly);
//   * the index words as 16-byte loads, behind the weights that they belong to: 4 bytes a lane, each cost as much as 16;
//   * the output through LDS.  The sparse operand has to be the instruction's rows, so a lane ends with channels of one token and its
//     neighbours have other tokens: stored from there, 16 bytes are an access of their own, 10000 of them per tile at one a cycle, twice
//     that with the residual.  Turned round in 4 KB that the wavefront owns, eight lanes hold a whole line;
//   * outputs beyond the last-level cache streamed: left in the L2s they pushed the operands out.
//   * scales and bias of a lane's channels kept over the units of its output that share them.
// us, 128-token kernel / stored from the accumulators / turned round / streamed / whole lines: 131072 x 1280 -> 5120 704 / 702 / 684 / 598 / 578,
// 131072 x 5120 -> 1280 with the residual 605 / 547 / 545 / - / 516.  Scales read anew for every 16 tokens / kept: 131072 x 1280 -> 5120 597 / 567, 131072 x
// 1024 -> 3072 325 / 308, 65536 x 1280 -> 5120 303 / 290, 131072 x 5120 -> 1280 with the residual 515 / 512.  A third k tile in LDS (256 x 256): nothing.  Three k tiles of X, its
// fragments read under the products before theirs (the output turned round where a k tile was): on zeros 5120 -> 1280 471 / 453, on codes 518 / 535 and 1280 -> 5120 571 / 599.
// Inside the ViT-H encoder, both Linears of the MLP 2:4, 32 images 115.7 -> 111.2 ms, 16 58.6 -> 55.5, one 5.52 -> 5.22.
#include "gemm_i8_sparse24_shared.hpp"
#include "gemm_pingpong.hpp"
#include "samfast_bench.h"

// every fp32 step below is rounded on its own
#pragma clang fp contract(off)

namespace samfast {

// TN: 16-channel fragments of a wavefront's half of the tile (the tile has 32 TN channels); a turn multiplies H of them.
// Fragment f of a half holds in its row i the channel 32 (f / 2) + 8 (i / 4) + 4 (f % 2) + i % 4: a lane ends with eight adjacent ones.
template <int TN>
struct STTile {
  static_assert(TN == 8 || TN == 10, "tiles built: 256 x {256, 320}");
  static constexpr int BM = 256, BN = 32 * TN, H = TN / 2;
  static constexpr int WUNITS = 2 * H, IUNITS = (2 * H + 3) / 4, UNITS = WUNITS + IUNITS;  // a turn's pieces of 1 KB: weights, indices
  static constexpr int TURN = UNITS * 1024;
  static constexpr int STAGE = BM * 128 + 2 * TURN;   // a k tile, of which two are held
  static constexpr int SCALES = BM * 4 + 2 * BN * 4;
  static constexpr int NSTORES = 4 * H;
  static_assert(UNITS > 8 && UNITS <= 16, "one or two pieces for each wavefront");
  static_assert(2 * STAGE + SCALES + 8 * 4096 + 16 <= 160 * 1024, "LDS of a CU");
  static constexpr int PAIRS = H / 2 * 2, UNITS_OUT = PAIRS + H % 2;
  // first channel of a half's pairs of fragment pairs, of its odd one
  static SF_DEVICE int first(int half) { return half * (TN == 10 ? 192 : 128); }
  static SF_DEVICE int odd(int half) { return 128 + 32 * half; }
  static SF_DEVICE int channel(int half, int f, int i) {
    return (f < 2 * PAIRS ? first(half) + 32 * (f >> 1) : odd(half)) + 8 * (i >> 2) + 4 * (f & 1) + (i & 3);
  }
};

// A fragment read (16 rows, two of eight chunks that lie two apart, served as lanes {0-3, 12-15, 20-27}, {4-11, 16-19, 28-31} and the same of
// the upper half) touches every bank once: the rows of either part are sent to one half of the positions.
SF_DEVICE int st_swizzle(int row) {
  const int m = row >> 1;
  return (m & 1) | ((m >> 1) & 2) | (((m << 1) ^ m) & 4);
}

template <int EPI, int TN, bool NT>
__global__ __launch_bounds__(512, 2) void gemm_i8_sp24_turns_kernel(SparseArgs a) {
  using P = STTile<TN>;
  constexpr bool RES = EPI == SEPI_RESIDUAL;
  constexpr int H = P::H;
  __shared__ __attribute__((aligned(16))) unsigned char lds[2 * P::STAGE + P::SCALES + 8 * 4096 + 16];
  unsigned char* sc = lds + 2 * P::STAGE;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave & 3, wn = wave >> 2;  // 64 tokens, half of the channels; wn is also the side that takes turns

  // ---- the tiles of this workgroup: XCD x owns a contiguous range, its workgroups walk it side by side -----------
  const unsigned int total = (unsigned int)a.tiles_x * (unsigned int)a.tiles_w;
  const unsigned int xcd = blockIdx.x & 7u, slot = blockIdx.x >> 3, per_x = gridDim.x >> 3;
  const unsigned int chunk = (total + 7u) >> 3;
  const unsigned int first = xcd * chunk + slot;
  const unsigned int last = min(total, (xcd + 1u) * chunk);
  if (slot >= chunk || first >= last) return;  // uniform over the workgroup
  const int nt = (int)((last - first + per_x - 1u) / per_x);
  // tiles at the edges are moved back inside (M >= BM, N >= BN); what belongs to the tile before is not stored
  auto tile_origin = [&](int ti, int& m0, int& n0, int& skip_m, int& skip_n) __attribute__((always_inline)) {
    const unsigned int pid = first + (unsigned int)ti * per_x;
    const unsigned int per_group = (unsigned int)a.group_x * a.tiles_w;
    const unsigned int first_m = (pid / per_group) * a.group_x;
    const unsigned int gsz = min((unsigned int)a.tiles_x - first_m, (unsigned int)a.group_x);
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
  // ---- tile loads.  X in eights of rows, 16-byte chunk c of LDS row r at position c ^ st_swizzle(r).  A turn's weights: fragment by
  // fragment, 64-k block by block, 16 rows of 32 bytes; behind them the index words, per fragment 128 bytes of either block.
  unsigned int off_x, off_w[2][2];
  const bool two = wave < P::UNITS - 8, second_idx = wave + 8 >= P::WUNITS;
  {
    const int r = wave * 8 + (lane >> 3), c = (lane & 7) ^ st_swizzle(r);
    off_x = (unsigned int)r * (unsigned int)a.x_row_pitch + (unsigned int)((c >> 2) * a.x_kstep) + (c & 3) * 16;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int unit = wave + 8 * u;
        if (u == 0 || !second_idx) {
          const int f = 2 * unit + (lane >> 5), i = (lane & 31) >> 1;
          const int half = f / (2 * H), kb = f / H & 1, j = f % H, h = lane & 1;
          off_w[t][u] = ((unsigned int)(kb * a.N) + P::channel(half, t * H + j, i)) * 32u + h * 16;
        } else {
          const int f = min(4 * (unit - P::WUNITS) + (lane >> 4), 2 * H - 1), kb = lane >> 3 & 1;  // (behind the last one: repeated, read by nobody)
          off_w[t][u] = ((unsigned int)(kb * a.N) + P::channel(f / H, t * H + f % H, 2 * (lane & 7))) * 8u;
        }
      }
  }
  const int8_t *xk, *wk, *ik;  // tile row 0 / channel 0 in the k tile that is requested next
  auto load = [&](const int8_t* base, unsigned int o, int dst) __attribute__((always_inline)) {
    asm volatile("" : "+s"(base));  // uniform base, 32-bit lane offset
    asm volatile("" : "+v"(o));
    __builtin_amdgcn_global_load_lds((gptr_t)(base + o), (lptr_t)(lds + dst), 16, 0, 0);
  };
  auto load_x = [&](int stage) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 4; ++i) load(xk + (int64_t)(64 * i) * a.x_row_pitch, off_x, stage + (wave + 8 * i) * 1024);
  };
  auto load_w = [&](int turn, int stage) __attribute__((always_inline)) {
    const int at = stage + P::BM * 128 + turn * P::TURN + wave * 1024;
    load(wk, off_w[turn][0], at);
    if (two) load(second_idx ? ik : wk, off_w[turn][1], at + 8192);
  };
  int m0, n0, skip_m, skip_n, lt = 0, lk = 0;
  const int nk = a.K / 128;
  auto first_ktile = [&]() __attribute__((always_inline)) {
    int m, n, sm, sn;
    tile_origin(lt, m, n, sm, sn);
    xk = a.x + (int64_t)m * a.x_row_pitch;
    wk = a.wc + (int64_t)n * 32;
    ik = reinterpret_cast<const int8_t*>(a.widx) + (int64_t)n * 8;
  };
  first_ktile();
  tile_origin(0, m0, n0, skip_m, skip_n);
  auto next_ktile = [&]() __attribute__((always_inline)) {
    xk += 2 * a.x_kstep;
    wk += (int64_t)a.N * 64;
    ik += (int64_t)a.N * 16;
    if (++lk == nk) {
      // the first k tiles of the next tile (behind the last one: its own again, read by nobody)
      lk = 0;
      if (lt + 1 < nt) ++lt;
      first_ktile();
    }
  };
  auto load_scales = [&]() __attribute__((always_inline)) {
    constexpr int XS = P::BM / 64, WS = P::BN / 64, SLICES = XS + 2 * WS;
#pragma unroll
    for (int e = 0; e < (SLICES + 7) / 8; ++e) {
      const int s = (wave + 8 * e) % SLICES;
      const int part = s < XS ? 0 : s < XS + WS ? 1 : 2, q = (part == 0 ? s : (s - XS) % WS) * 64;
      const float* src = part == 0 ? a.sx + m0 : (part == 1 || !a.bias ? a.sw : a.bias) + n0;
      const int dst = (part == 0 ? 0 : part == 1 ? P::BM * 4 : P::BM * 4 + P::BN * 4) + q * 4;
      __builtin_amdgcn_global_load_lds((gptr_t)(src + q + lane), (lptr_t)(sc + dst), 4, 0, 0);
    }
  };

  // ---- fragments and products ------------------------------------------------------------------------------------------
  // v_smfmac_i32_16x16x128_i8 (measured): lane (j, Q) of the dense operand holds the k slots 32 Q .. 32 Q + 31 of column j, lane (i, q) of
  // the sparse one the kept values of row i in the slots 64 (q % 2) + 32 u + 16 (q / 2) + 0 .. 15, u = 0, 1 for its lower and upper 8 bytes.
  // Here lane (i, q) reads the stored half q % 2 of 64-k block q / 2; the slots are then k 64 (q / 2) + 32 u + 16 (q % 2) + 0 .. 15, and lane
  // (j, Q) of the dense operand reads the 16-byte chunks 2 (Q % 2) + Q / 2 and four more of its 128-byte row.
  const int lr = lane & 15, lq = lane >> 4;
  const int frag = (((lq & 1) * 2 + (lq >> 1)) ^ st_swizzle(lr)) * 16;
  const int x_off[2] = {(wm * 64 + lr) * 128 + frag, (wm * 64 + lr) * 128 + (frag ^ 64)};
  const int w_off = P::BM * 128 + (wn * 2 + (lq >> 1)) * H * 512 + (2 * lr + (lq & 1)) * 16;
  const int i_off = P::BM * 128 + P::WUNITS * 1024 + wn * H * 256 + (lq >> 1) * 128 + lr * 8 + (lq & 1) * 4;
  i32x8 fx[4];
  i32x4 fw[H];
  int fi[H];
  i32x4 acc[4][TN];
  auto read = [&](int turn, int stage) __attribute__((always_inline)) {
    if (turn == 0)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const i32x4 lo = *reinterpret_cast<const i32x4*>(lds + stage + x_off[0] + i * 2048);
        const i32x4 hi = *reinterpret_cast<const i32x4*>(lds + stage + x_off[1] + i * 2048);
        fx[i] = i32x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      }
#pragma unroll
    for (int j = 0; j < H; ++j) {
      fw[j] = *reinterpret_cast<const i32x4*>(lds + stage + turn * P::TURN + w_off + j * 512);
      fi[j] = *reinterpret_cast<const int*>(lds + stage + turn * P::TURN + i_off + j * 256);
    }
  };
  auto multiply = [&](auto turn) __attribute__((always_inline)) {
    constexpr int T = decltype(turn)::value;
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int jj = 0; jj < H; ++jj) {
        const int j = i & 1 ? H - 1 - jj : jj;  // one operand stays from each instruction to the next
        acc[i][T * H + j] = __builtin_amdgcn_smfmac_i32_16x16x128_i8(fw[j], fx[i], acc[i][T * H + j], fi[j], 0, 0);
      }
    // (the products are pure values to the compiler; this pins them to their turn)
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < H; ++j) asm volatile("" : "+v"(acc[i][T * H + j]));
    __builtin_amdgcn_s_setprio(0);
  };
  auto meet = [&]() __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };
  auto arrive = [&](auto extra_n, bool extra) __attribute__((always_inline)) {
    constexpr int EXTRA = decltype(extra_n)::value;
    if (EXTRA > 0 && extra) {
      if (two) pp_wait<8 + EXTRA>();
      else pp_wait<6 + EXTRA>();
    } else {
      if (two) pp_wait<8>();
      else pp_wait<6>();
    }
  };

  // ---- output: tokens 16 (4 wm + i) + lr, channels 16 TN wn + 32 p + 8 lq ------------------------------------------------
  typedef __attribute__((address_space(1))) unsigned char* gbyte_t;
  typedef __attribute__((address_space(1))) u32x4* gpiece_t;
  auto lane_again = [&]() __attribute__((always_inline)) {  // (made again at every use: kept, it would be spilled)
    int l = lane;
    asm volatile("" : "+v"(l));
    return l;
  };
  auto finish = [&](auto whole) __attribute__((always_inline)) {
    constexpr bool FULL = decltype(whole)::value;
    const int l = lane_again(), lr = l & 15, lq = l >> 4;
    const int row0 = wm * 64, first = P::first(wn), odd = P::odd(wn);
    const unsigned int pitch = (unsigned int)a.ldo * 2u, rpitch = RES ? (unsigned int)a.ld_res * 2u : 0u;
    const unsigned char* to = reinterpret_cast<const unsigned char*>(reinterpret_cast<unsigned short*>(a.out) + (int64_t)(m0 + row0) * a.ldo + n0);
    const unsigned char* from = RES ? reinterpret_cast<const unsigned char*>(a.residual + (int64_t)(m0 + row0) * a.ld_res + n0) : nullptr;
    unsigned char* const turn = sc + P::SCALES + wave * 4096;
    // piece i of unit u: 8 tokens from row_of on and 64 channels, of the odd pair 16 tokens and 32 channels
    auto wide = [&](int u) { return u < P::PAIRS; };
    auto row_of = [&](int u, int i) { return wide(u) ? 32 * (u & 1) + 8 * i : 16 * i; };
    auto lane_row = [&](int u) { return wide(u) ? l >> 3 : l >> 2; };
    auto lane_chunk = [&](int u) { return wide(u) ? l & 7 : l & 3; };
    auto column = [&](int u) { return wide(u) ? first + 64 * (u >> 1) : odd; };
    auto place = [&](const unsigned char* tile, unsigned int pitch, int u, int i) __attribute__((always_inline)) {
      const unsigned char* b = tile + (int64_t)row_of(u, i) * pitch + 2 * column(u);
      asm volatile("" : "+s"(b));
      return (gpiece_t)((gbyte_t)(uintptr_t)b + ((unsigned int)lane_row(u) * pitch + 16 * lane_chunk(u)));
    };
    u32x4 res[4], o[4];
    auto load_residual = [&](int u) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < 4; ++i) res[i] = *place(from, rpitch, u, i);
    };
    float sx[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) sx[i] = *reinterpret_cast<const float*>(sc + (row0 + 16 * i + lr) * 4);
    // Scales and bias of a lane's eight channels of a pair: kept while the two wide units that share 64 channels need them, or, where the
    // residual leaves no registers for both pairs, read for twice 16 tokens.  Read anew for every 16 tokens they were two thirds of an end's LDS
    // operations.
    constexpr bool KEEP = !RES || TN == 8;
    f32x4 scale[1 + KEEP][1 + KEEP], shift[1 + KEEP][1 + KEEP];
    auto constants = [&](int slot, int t, int channel) __attribute__((always_inline)) {
      const int at = P::BM * 4 + (channel + 8 * lq + 4 * t) * 4;
      scale[slot][KEEP ? t : 0] = *reinterpret_cast<const f32x4*>(sc + at);
      shift[slot][KEEP ? t : 0] = *reinterpret_cast<const f32x4*>(sc + (a.bias ? P::BN * 4 + at : P::SCALES + 8 * 4096));
    };
#pragma unroll
    for (int u = 0; u <= P::UNITS_OUT; ++u) {
      if (u < P::UNITS_OUT) {
        if (KEEP && !(wide(u) && u & 1)) {
#pragma unroll
          for (int d = 0; d < (wide(u) ? 2 : 1); ++d)
#pragma unroll
            for (int t = 0; t < 2; ++t) constants(d, t, column(u) + 32 * d);
        }
#pragma unroll
        for (int d = 0; d < 2; ++d) {
          // twice 16 tokens by 32 channels: token fragments i0 and i0 + 1, channel pair p
          const int i0 = wide(u) ? 2 * (u & 1) : 2 * d, p = wide(u) ? (u & ~1) + d : P::PAIRS;
          u32x4 v4[2];
#pragma unroll
          for (int t = 0; t < 2; ++t) {
            const int k = KEEP && wide(u) ? d : 0, kt = KEEP ? t : 0;
            if (!KEEP) constants(0, t, column(u) + (wide(u) ? 32 * d : 0));
            const f32x4 sw = scale[k][kt], bias = shift[k][kt];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
              float y[4];
#pragma unroll
              for (int r = 0; r < 4; ++r) {
                // three separately rounded fp32 operations (no fused multiply-add)
                float v = (float)acc[i0 + j][2 * p + t][r] * sx[i0 + j];
                v = v * sw[r];
                y[r] = v + bias[r];
              }
              v4[j][2 * t] = pack_bf16x2(y[0], y[1]);
              v4[j][2 * t + 1] = pack_bf16x2(y[2], y[3]);
            }
          }
          // through the wavefront's own 4 KB: a lane has 16 bytes of a token, neighbouring lanes other tokens
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            const int in = wide(u) ? j * 2048 + lr * 128 + (((4 * d + lq) ^ (lr >> 1)) * 16) : (2 * d + j) * 1024 + lr * 64 + ((lq ^ (-(lr >> 2) & 3)) * 16);
            *reinterpret_cast<u32x4*>(turn + in) = v4[j];
          }
          __builtin_amdgcn_sched_barrier(0);  // keep the conversion narrow
        }
      }
      if (u > 0) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if constexpr (RES) {
            const u32x4 v = res[i];
#pragma unroll
            for (int c = 0; c < 4; ++c)
              o[i][c] = pack_bf16x2(bf16_lo_to_f32(o[i][c]) + bf16_lo_to_f32(v[c]), bf16_hi_to_f32(o[i][c]) + bf16_hi_to_f32(v[c]));
          }
          const gpiece_t dst = place(to, pitch, u - 1, i);
          if (FULL || (row0 + row_of(u - 1, i) + lane_row(u - 1) >= skip_m && column(u - 1) + 8 * lane_chunk(u - 1) >= skip_n)) {
            if (NT) __builtin_nontemporal_store(o[i], dst);
            else *dst = o[i];
          }
        }
      }
      if (u < P::UNITS_OUT) {
        const int row = lane_row(u), chunk = lane_chunk(u);
#pragma unroll
        for (int i = 0; i < 4; ++i)
          o[i] = *reinterpret_cast<const u32x4*>(turn + (wide(u) ? i * 1024 + row * 128 + ((chunk ^ ((row >> 1) + 4 * (i & 1))) * 16)
                                                                 : i * 1024 + row * 64 + ((chunk ^ (-(row >> 2) & 3)) * 16)));
        // (one unit ahead; with two in flight registers were spilled, 131072 x 5120 -> 1280 567 us for 547)
        if constexpr (RES) load_residual(u);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (u == 0 && wn == 0) meet();
    }
  };

  // no bias: zeros
  if (tid == 0) *reinterpret_cast<u32x4*>(sc + P::SCALES + 8 * 4096) = u32x4{0u, 0u, 0u, 0u};

  // ---- prologue: k tile 0, and of k tile 1 what the first turn of a k tile needs ---------------------------------
  load_x(0);
  load_w(0, 0);
  load_w(1, 0);
  next_ktile();
  load_x(P::STAGE);
  load_w(0, P::STAGE);
  arrive(std::integral_constant<int, 0>{}, false);  // X and the first channels of k tile 0
  meet();
  if (wn == 1) meet();  // from here on the upper half is one turn behind

  int stage = 0;
  // One k tile, its loads and waits as in gemm_pingpong_kernel
  auto ktile = [&](auto first_of_tile, auto extra_n, bool extra) __attribute__((always_inline)) {
    using T0 = std::integral_constant<int, 0>;
    using T1 = std::integral_constant<int, 1>;
    constexpr bool ZERO = decltype(first_of_tile)::value;
    const int other = P::STAGE - stage;
    auto clear = [&](int turn) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < H; ++j) acc[i][turn * H + j] = i32x4{0, 0, 0, 0};
    };
    read(0, stage);
    load_w(1, other);
    next_ktile();
    if constexpr (ZERO) clear(0);
    arrive(extra_n, extra);
    meet();
    multiply(T0{});
    meet();
    read(1, stage);
    load_x(stage);
    load_w(0, stage);
    if constexpr (ZERO) {
      load_scales();
      clear(1);
    }
    arrive(extra_n, extra);
    meet();
    multiply(T1{});
    meet();
    stage = other;
  };
  using Yes = std::true_type;
  using No = std::false_type;
  bool stored = false;  // a whole tile's stores are on their way
  for (int ti = 0; ti < nt; ++ti) {
    ktile(Yes{}, std::integral_constant<int, P::NSTORES>{}, stored);
    for (int k = 1; k < nk; ++k) ktile(No{}, std::integral_constant<int, 0>{}, false);
    stored = skip_m == 0 && skip_n == 0;
    if (stored) finish(Yes{});
    else finish(No{});
    if (wn == 1) meet();
    if (ti + 1 < nt) tile_origin(ti + 1, m0, n0, skip_m, skip_n);
  }
  if (wn == 0) meet();
  __builtin_amdgcn_s_waitcnt(0x0070);  // the last loads land before the LDS is given back
}

// Columns / 32 of the tile, 0: neither fits; rounds of the CUs and the share of their time that makes output.
struct STChoice {
  int tn;
  int64_t rounds;
  double used;
};
// A round of 320 channels takes 1.19 rounds of 256: 131072 x 1280 -> 5120 18.8 / 15.8 us, 5120 -> 1280 65.4 / 55.4, 1024 -> 4096 16.5 / 13.8.
static STChoice st_choose(const SparseArgs& a) {
  STChoice best = {0, 0, 0.0};
  const int force = knob_or(KNOB_SPARSE_TURNS, 1);
  double least = 0.0;
  for (int tn = 8; tn <= 10; tn += 2) {
    if (a.M < 256 || a.N < 32 * tn || (force >= 8 && force != tn)) continue;
    const int64_t rounds = (((int64_t)a.M + 255) / 256 * ((a.N + 32 * tn - 1) / (32 * tn)) + 255) / 256;
    const double cost = rounds * (tn == 8 ? 10.0 : 11.9);
    if (best.tn != 0 && cost >= least) continue;
    best = STChoice{tn, rounds, (double)a.M * a.N / (256.0 * rounds * 256 * 32 * tn)};
    least = cost;
  }
  return best;
}

static bool whole_lines(const void* p, int64_t ld) { return reinterpret_cast<uintptr_t>(p) % 128 == 0 && ld % 64 == 0; }

bool gemm_i8_sp24_turns_covers(int epi, const SparseArgs& a) {
  const int mode = knob_or(KNOB_SPARSE_TURNS, 1);
  if (mode <= 0 || (epi != SEPI_SCALE_BIAS && epi != SEPI_RESIDUAL)) return false;
  // 32-bit lane offsets inside a tile
  if (a.K % 128 != 0 || a.K < 640 || a.ldo >= (1ll << 22) || (epi == SEPI_RESIDUAL && a.ld_res >= (1ll << 22))) return false;
  const STChoice c = st_choose(a);
  if (c.tn == 0 || mode >= 8) return c.tn != 0;
  // The lines (us, the 128-token kernel / this one, Gaussian codes, K-block major; 2700 products of 640 to 5120 by 768 to 8192, half
  // of them drawn at random, stand behind them).
  // Rows that are whole cache lines: eight lanes hold 128 bytes of a row, and where its lines lie elsewhere every store, and the residual's
  // loads, are two of them in part.  Streamed ones 32288 x 640 -> 4904 112 / 252, else 8012 x 1024 -> 4904 39.8 / 51.2, 38665 x 640 -> 1992 63.2 / 68.9,
  // with the residual 20496 x 640 -> 5096 122 / 177, 47794 x 768 -> 1992 120 / 163; nothing at the longest loops (24143 x 4096 -> 1992 122.0 / 122.0).
  if (!whole_lines(a.out, a.ldo) || (epi == SEPI_RESIDUAL && !whole_lines(a.residual, a.ld_res))) return false;
  if (epi == SEPI_RESIDUAL) {
    // The residual's loads lengthen every tile's end, in which nothing is multiplied, so that loops have to be the longer the more
    // ends there are, and the column tiles few:
    //   256 channels, from three rounds on, 0.85 of them used: up to 1280 columns and from 2560 on 131072 x 4096 -> 1024 411 / 384, 65536 x 3072 -> 1024
    //     173 / 164; but 57344 x 2048 -> 768 89.5 / 89.3, 40960 x 3072 -> 3072 283 / 289
    //   320, 0.8 used: one round from 1024 on or up to 1280 columns 8192 x 1024 -> 2304 28.0 / 26.9, 13632 x 896 -> 1280 26.5 / 24.6; but 11654 x 640 -> 1536 24.0 / 24.7.
    //     Two rounds, or up to 1280 columns: from 2048 on 10317 x 2048 -> 3840 70.0 / 68.5, 65536 x 2560 -> 1280 187 / 173, 40960 x 5120 -> 1280 201 / 193; but
    //     16338 x 1280 -> 2304 51.2 / 53.3, 69627 x 640 -> 1280 109 / 119.  Others from nine rounds and 3072 on: 40504 x 4096 -> 5120 561 / 531; but five
    //     rounds 40960 x 2560 -> 2560 213 / 216, 16943 x 1536 -> 8192 194 / 212
    const bool narrow = a.N <= 1280;
    if (c.tn == 8) return c.rounds >= 3 && c.used >= 0.85 && narrow && a.K >= 2560;
    if (c.used < 0.8) return false;
    if (c.rounds == 1) return narrow || a.K >= 1024;
    return narrow || c.rounds == 2 ? a.K >= 2048 : c.rounds >= 9 && a.K >= 3072;
  }
  // Outputs that the 128-token kernel's tiles hold in one round, two of them on a CU, are its own: 4096 x 1024 -> 4096 (512 tiles) 18.5 / 19.7, 16384 x
  // 1280 -> 1024 20.8 / 22.1, 4096 x 640 -> 3840 13.9 / 15.5; but 528 (4200 x 1024 -> 4096) 24.6 / 21.2.
  if (((int64_t)a.M + 127) / 128 * ((a.N + 255) / 256) <= 512) return false;
  // By `used`:
  //   256 channels 0.92, on loops beyond 1536 0.95: 0.98 (36149 x 768 -> 4096) 120 / 117, 0.94 (28672 x 896 -> 3840) 95.0 / 94.4, 1.0 (16384 x 2560 -> 3072) 86.9 / 86.9;
  //     but 0.9 (27377 x 768 -> 3840) 85.2 / 86.2, 0.94 (16453 x 2560 -> 3840) 111 / 113
  //   320 0.88: 0.89 (14612 x 3072 -> 5120) 144 / 139, 1.0 (65536 x 1280 -> 5120) 358 / 302; but 0.86 (23968 x 1280 -> 3840) 99.3 / 101.3.  Within two rounds
  //     0.8: 0.83 (4261 x 768 -> 4096) 21.8 / 19.1, 0.84 (11496 x 5120 -> 3072) 119 / 106, but 0.75 (4096 x 768 -> 3072) 14.5 / 15.9.  Beyond them on loops
  //     shorter than 1024 0.91: 0.92 (30232 x 640 -> 5120) 116 / 108, but 0.9 (24576 x 768 -> 3072) 60.7 / 62.1
  if (c.tn == 8) return c.used >= (a.K <= 1536 ? 0.92 : 0.95);
  return c.used >= (c.rounds <= 2 ? 0.8 : a.K >= 1024 ? 0.88 : 0.91);
}

int gemm_i8_sp24_turns_launch(int epi, const SparseArgs& args, hipStream_t stream) {
  SparseArgs a = args;
  const int tn = st_choose(a).tn;
  a.tiles_x = (a.M + 255) / 256;
  a.tiles_w = (a.N + 32 * tn - 1) / (32 * tn);
  a.group_x = 4;
  const unsigned int grid = (unsigned int)min((int64_t)256, ((int64_t)a.tiles_x * a.tiles_w + 7) / 8 * 8);
  const bool nt = (int64_t)a.M * a.N * 2 >= (256ll << 20);
#define SF_ST(E, TN, NT) hipLaunchKernelGGL((gemm_i8_sp24_turns_kernel<E, TN, NT>), dim3(grid), dim3(512), 0, stream, a)
  if (epi == SEPI_RESIDUAL) { if (tn == 8) SF_ST(SEPI_RESIDUAL, 8, false); else SF_ST(SEPI_RESIDUAL, 10, false); }
  else if (nt) { if (tn == 8) SF_ST(SEPI_SCALE_BIAS, 8, true); else SF_ST(SEPI_SCALE_BIAS, 10, true); }
  else { if (tn == 8) SF_ST(SEPI_SCALE_BIAS, 8, false); else SF_ST(SEPI_SCALE_BIAS, 10, false); }
#undef SF_ST
  return check_launch("gemm_i8_sp24_turns_kernel");
}

}  // namespace samfast

extern "C" int samfast_bench_sparse24_turns(int64_t M, int N, int K, int epilogue, int64_t row_stride) {
  using namespace samfast;
  SF_REQUIRE(M > 0 && M < (1ll << 31) - 256 && N > 0 && K > 0 && row_stride >= N, "bench_sparse24_turns: bad shape M=%lld N=%d K=%d", (long long)M, N, K);
  SparseArgs a = {};
  a.M = (int)M; a.N = N; a.K = K; a.ldo = a.ld_res = row_stride;
  const int epi = epilogue == SAMFAST_EPILOGUE_NONE ? SEPI_SCALE_BIAS : epilogue == SAMFAST_EPILOGUE_RESIDUAL ? SEPI_RESIDUAL : SEPI_GELU;
  return gemm_i8_sp24_turns_covers(epi, a) ? 32 * st_choose(a).tn : 0;
}
