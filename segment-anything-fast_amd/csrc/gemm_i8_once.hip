// int8 GEMM for outputs that the GPU holds once: one 512-thread workgroup per CU, one tile per
// workgroup (an image's Linears: 4096 rows, 768 to 5120 columns).
//
// What bounds such a launch is not the matrix pipe (19 GOP are 6 us of it) but latency and operand
// traffic: there is no second tile whose loop hides a workgroup's start and end, and small tiles fetch
// every operand many times (64 x 128 tiles of 4096 x 3072 -> 768: 226 MB through 64 B/clk a CU, where
// 128 x 96 ones take 176 MB; the loads wait for the L2s' misses, and starting the workgroups at different k or
// touching the panels ahead made it worse: 3.9 MB of operands an XCD share 4 MB of L2).  So the tile is the one that deals the output to the CUs evenly - 64 x
// {64, 96, 128} (some hundred rows, or few columns), 128 x {96, 128, 160} or 256 x {192, 256, 320}: widths of 768, 1024 and 1280 give exactly 256 tiles of 4096
// rows, as do their fourfold - and the 160 KB of LDS hold three to five stages of it:
//   * eight wavefronts, 64 x 16 TN outputs each.  At 256 rows they sit 4 x 2; at 128 rows 2 x 2 in two
//     groups that take every second k tile (a wavefront of half the size would read 1.4 times the operand
//     bytes from LDS), at 64 rows two columns of them in four groups; their integer sums are exchanged through LDS at the end, each group finishing its share of the rows;
//   * a stage is global -> LDS loads only; the threshold of outstanding loads leaves NST - 2 stages in
//     flight across the one barrier of an iteration.  The loads stand between the products: a wavefront waits in line with a load, 16 cycles
//     for each that is ahead of it, and in front of the products they made an iteration of 4096 x 3072 -> 768 694 cycles, 384 of products and 448 of
//     loads (us, in front / between: 4096 x 1280 -> 1280 14.9 / 14.4, 1024 x 5120 -> 1280 19.0 / 18.1, 3000 x 3072 -> 768 15.1 / 14.6).  Not so
//     where an operand is row-major and the tile has 128 rows: the two groups' k tiles are halves of the same lines, and requests that go out together,
//     in front of the products, share them (in front / between: both row-major 643 x 2176 -> 4952 14.1 / 15.0, 897 x 4992 -> 4096 with GELU 29.5 / 30.8; over 263 products 0.986 times as
//     long; row-major weights alone, a Linear's, 250 of them 0.993; both K-block major, 137 of them, 1.017);
//   * v_mfma_i32_16x16x64_i8 with W as A and X as B: a lane ends with four adjacent columns of one row.  The
//     fragments of the next k tile are read while this one's MFMAs run, where registers allow (TN <= 5);
//   * the residual rows are requested before the loop (128-row tiles), scales and bias land in LDS under it,
//     and the tile leaves through LDS in whole row segments, 16 bytes a lane.
// Integer sums and the epilogue's arithmetic are those of the other members: the same bits.
#include "gemm_i8_shared.hpp"
#include <type_traits>

// every fp32 step below is rounded on its own (no fused multiply-add), as in the other forms
#pragma clang fp contract(off)

namespace samfast {

template <int BM_, int TN_>
struct OnceCfg {
  static constexpr int BM = BM_, TN = TN_, TM = 4;
  static constexpr int KG = BM == 64 ? 4 : BM == 128 ? 2 : 1;  // groups of wavefronts, each on every KG-th k tile
  static constexpr int BN = 32 * TN;
  static constexpr int PART = (BM + BN) * GLD;         // one group's share of a stage
  static constexpr int STAGE = KG * PART;
  static constexpr int NST = STAGE <= 28672 ? 5 : STAGE <= 36864 ? 4 : 3;
  static constexpr bool AHEAD = TN <= 5;               // fragments read one iteration ahead
  static constexpr int WROWS = BN * KG / 8;            // W rows of a stage that a wavefront loads; X rows: 32
  static constexpr int NLD = 2 + (WROWS + 15) / 16;    // load instructions per stage and wavefront
  static constexpr int BNP = (BN + 63) / 64 * 64;
  static constexpr int SW_OFF = BM * 4, BIAS_OFF = SW_OFF + BNP * 4, SC_BYTES = BIAS_OFF + BNP * 4;
  static constexpr int PITCH = BN * 2 + 16;            // staged output rows
  static constexpr int ROWS = BM == 256 ? 128 : BM;    // rows staged at a time
  static constexpr int CH = BN / 8, PIECES = ROWS * CH, PASSES = (PIECES + 511) / 512;  // 16-byte pieces per row; passes of the workgroup over them
  static_assert(BM == 64 || BM == 128 || BM == 256, "row tiles built");
  static_assert(ROWS * PITCH <= NST * STAGE && (KG == 1 || 4 * KG * TN * 2048 <= NST * STAGE), "epilogue buffers fit the stages");
  static_assert(NST * STAGE + SC_BYTES <= 160 * 1024, "LDS of a CU");
  static_assert((NST - 1) * NLD + 2 + PASSES < 64, "vmcnt threshold");
};

// 16-byte chunk c of LDS row r lives at chunk position c ^ once_swizzle(r).  A fragment read of 16 rows x 4
// chunks is served as lanes {0-3, 12-15, 20-27}, {4-11, 16-19, 28-31} and the same of the upper half; with
// this rotation each of those touches every bank once (with lds_swizzle, made for 32 rows of one chunk, two
// lanes met in each bank: 5700 of 31000 cycles at 4096 x 3072 -> 768).
SF_DEVICE int once_swizzle(int row) { return -(row >> 2) & 3; }

template <int N>
SF_DEVICE void wait_vm() {
  __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
}

// A wave instruction of 16 bytes from base + off to LDS at dst for the lower 32 lanes, without the branch that a condition on the lane would
// put between the products (all lanes are active where it stands).
SF_DEVICE void load_lower_half(const int8_t* base, unsigned int off, unsigned int dst) {
  asm volatile("s_mov_b64 exec, 0xffffffff\n\tglobal_load_lds_dwordx4 %0, %1\n\ts_mov_b64 exec, -1" : : "v"(off), "s"(base), "{m0}"(dst) : "memory");
}

// FRONT: the loads in front of the products (see above)
template <int EPI, int BM, int TN, bool FRONT = false>
__global__ __launch_bounds__(512, 2) void gemm_i8_once_kernel(GemmArgs a) {
  using C = OnceCfg<BM, TN>;
  static_assert(!FRONT || (BM == 128 && C::AHEAD), "built for 128 rows");
  constexpr int TM = C::TM, KG = C::KG, BN = C::BN, NST = C::NST, NLD = C::NLD;
  __shared__ __attribute__((aligned(16))) unsigned char lds[C::NST * C::STAGE + C::SC_BYTES];
  unsigned char* sc = lds + NST * C::STAGE;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = KG == 4 ? wave >> 1 : KG == 2 ? wave >> 2 : 0;
  const int wm = KG == 4 ? 0 : KG == 2 ? (wave >> 1) & 1 : wave >> 1, wn = wave & 1;
  const int lr = lane & 15, lq = lane >> 4;

  const unsigned int total = (unsigned int)a.tiles_m * (unsigned int)a.tiles_n;
  const unsigned int pid = xcd_contiguous_id(blockIdx.x, total);
  if (pid >= total) return;  // uniform over the workgroup
  const unsigned int per_group = (unsigned int)a.group_m * a.tiles_n;
  const unsigned int first_m = (pid / per_group) * a.group_m;
  const unsigned int gsz = min((unsigned int)a.tiles_m - first_m, (unsigned int)a.group_m);
  const unsigned int in_group = pid % per_group;
  const int m0 = (int)(first_m + in_group % gsz) * BM;
  const int n0 = (int)(in_group / gsz) * BN;

  typedef __attribute__((address_space(1))) const void* gptr_t;
  typedef __attribute__((address_space(3))) void* lptr_t;

  // phase-2 geometry of the epilogue: piece p of this thread is 16 bytes of staged row row_of(p)
  auto piece = [&](int p, int& t, int& ch) { const int i = tid + 512 * p; t = i / C::CH; ch = i % C::CH; };
  auto out_row = [&](int t, int h) {  // staged row t of half h
    return KG != 1 ? t : (t >> 5) * 64 + h * 32 + (t & 31);
  };
  static_assert(EPI != EPI_RESIDUAL_BF16 || KG != 1, "the residual epilogue is built for up to 128 rows");
  u32x4 res[C::PASSES];
  auto load_residual = [&] {
#pragma unroll
    for (int p = 0; p < C::PASSES; ++p) {
      int t, ch;
      piece(p, t, ch);
      const int m = min(m0 + t, a.M - 1), n = min(n0 + ch * 8, a.N - 8);  // N % 8 == 0
      res[p] = *reinterpret_cast<const u32x4*>(a.residual + (int64_t)m * a.ld_res + n);
    }
  };
  // tile loads: wavefront lw of LW loads X rows 32 lw .. and W rows WROWS lw .. of its group's part
  constexpr int LW = 8 / KG;
  const int lw = wave % LW;
  unsigned int off[NLD];
#pragma unroll
  for (int i = 0; i < NLD; ++i) {
    const int row = (i < 2 ? 32 * lw + 16 * i : C::WROWS * lw + 16 * (i - 2)) + (lane >> 2);
    const int chunk = (lane & 3) ^ once_swizzle(row);
    off[i] = (unsigned int)((i < 2 ? min(m0 + row, a.M - 1) * a.x_pitch : min(n0 + row, a.N - 1) * a.w_pitch) + chunk * 16);
  }
  const int nk = a.K / GBK, nt = (nk + KG - 1) / KG;  // nt > NST (the dispatch sees to it)
  auto fill = [&](int t, int stage) {
    // (KG == 4: where the last k tiles are fewer than the groups, some fetch one again that they do not multiply)
    const int kt = KG == 4 ? min(t * KG + grp, nk - 1) : t * KG + grp;
    const int8_t* xb = a.x + kt * a.x_kstep;
    const int8_t* wb = a.w + kt * a.w_kstep;
    asm volatile("" : "+s"(xb), "+s"(wb));  // tile bases stay scalar: scalar-base load form
    unsigned char* part = lds + stage * C::STAGE + grp * C::PART;
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
      unsigned int o = off[i];
      asm volatile("" : "+v"(o));
      const int8_t* src = (i < 2 ? xb : wb) + o;
      unsigned char* dst = part + (i < 2 ? 32 * lw + 16 * i : BM + C::WROWS * lw + 16 * (i - 2)) * GLD;
      const bool half = C::WROWS % 16 != 0 && i == NLD - 1;  // eight rows: the lower 32 lanes
      if (half) load_lower_half(i < 2 ? xb : wb, o, (unsigned int)(uintptr_t)(lptr_t)dst);
      else __builtin_amdgcn_global_load_lds((gptr_t)src, (lptr_t)dst, 16, 0, 0);
    }
  };

  fill(0, 0);
  if constexpr (EPI == EPI_RESIDUAL_BF16) load_residual();
  // scales and bias, 64 values per wave instruction; two instructions per wavefront, some of them repeats
  constexpr int XS = BM / 64, WS = C::BNP / 64, SLICES = XS + 2 * WS;
  static_assert(SLICES <= 16, "two slices per wavefront");
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const int s = (wave + 8 * e) % SLICES;
    const int cs = s < XS ? s : (s - XS) % WS;
    const float* base = s < XS ? a.sx : (s < XS + WS || !a.bias) ? a.sw : a.bias;
    const int at = s < XS ? min(m0 + cs * 64 + lane, a.M - 1) : min(n0 + cs * 64 + lane, a.N - 1);
    unsigned char* dst = sc + (s < XS ? 0 : s < XS + WS ? C::SW_OFF : C::BIAS_OFF) + cs * 256;
    __builtin_amdgcn_global_load_lds((gptr_t)(base + at), (lptr_t)dst, 4, 0, 0);
  }
  constexpr int EXTRA = 2 + (EPI == EPI_RESIDUAL_BF16 ? C::PASSES : 0);  // loads between the first stage and the second
#pragma unroll
  for (int p = 1; p < NST; ++p) fill(p, p);
  i32x4 acc[TN][TM];
#pragma unroll
  for (int j = 0; j < TN; ++j)
#pragma unroll
    for (int i = 0; i < TM; ++i) acc[j][i] = i32x4{0, 0, 0, 0};

  const int frag = lr * GLD + ((lq ^ once_swizzle(lr)) * 16);
  const int x_off = grp * C::PART + wm * 64 * GLD + frag;
  const int w_off = grp * C::PART + (BM + wn * (BN / 2)) * GLD + frag;
  struct Frags { i32x4 w[TN], x[TM]; };
  auto read = [&](Frags& f, int stage) {
    const unsigned char* s = lds + stage * C::STAGE;
#pragma unroll
    for (int i = 0; i < TM; ++i) f.x[i] = *reinterpret_cast<const i32x4*>(s + x_off + i * 16 * GLD);
#pragma unroll
    for (int j = 0; j < TN; ++j) f.w[j] = *reinterpret_cast<const i32x4*>(s + w_off + j * 16 * GLD);
  };
  auto multiply = [&](const Frags& f) {
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int i = 0; i < TM; ++i) acc[j][i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(f.w[j], f.x[i], acc[j][i], 0, 0, 0);
  };
  // own share of the tile that `left` later ones follow has landed; own LDS reads are done; all wavefronts meet
  auto arrive = [&](int left) {
    __builtin_amdgcn_s_waitcnt(0xC07F);
    if (left >= NST - 1) wait_vm<(NST - 1) * NLD + EXTRA>();  // the first tile
    else if (left == NST - 2) wait_vm<(NST - 2) * NLD>();
    else if (NST > 4 && left == 2) wait_vm<2 * NLD>();
    else if (left == 1) wait_vm<NLD>();
    else wait_vm<0>();
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };
  int st = 0;
  auto next_stage = [&](int s) { return s == NST - 1 ? 0 : s + 1; };
  using Yes = std::integral_constant<bool, true>;
  using No = std::integral_constant<bool, false>;
  if constexpr (C::AHEAD) {
    // iteration t: the stage of tile t (read in the iteration before) is refilled, tile t + 1 is read.
    // `steady`: NST later tiles follow
    Frags f0, f1;
    arrive(NST - 1);
    read(f0, 0);
    auto iteration = [&](int t, Frags& now, Frags& next, auto steady) {
      constexpr bool STEADY = decltype(steady)::value;
      if constexpr (STEADY) arrive(NST - 2);
      else arrive(min(nt - 2 - t, NST - 2));
      const int free = st;
      if (FRONT && (STEADY || t + NST < nt)) fill(t + NST, free);
      st = next_stage(st);
      if (STEADY || t + 1 < nt) read(next, st);
      if (STEADY || KG < 4 || t * KG + grp < nk) multiply(now);
      if (!FRONT && (STEADY || t + NST < nt)) fill(t + NST, free);
      if (FRONT && STEADY) {
        // one fragment read behind each of the first MFMAs
#pragma unroll
        for (int g = 0; g < TM + TN; ++g) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
      } else if (STEADY) {
        // two fragment reads behind each of the first MFMAs, then the requests spread over the others: a wavefront waits in line with a
        // request, 16 cycles for each that is ahead of it
        constexpr int READS = TM + TN, FIRST = (READS + 1) / 2, EACH = (TM * TN - FIRST) / NLD;
#pragma unroll
        for (int g = 0; g < FIRST; ++g) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
        }
#pragma unroll
        for (int g = 0; g < NLD; ++g) {
          __builtin_amdgcn_sched_group_barrier(0x008, EACH, 0);
          __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    int t = 0;
    for (; t + 1 + NST < nt; t += 2) {
      iteration(t, f0, f1, Yes{});
      iteration(t + 1, f1, f0, Yes{});
    }
    for (; t + 1 < nt; t += 2) {
      iteration(t, f0, f1, No{});
      iteration(t + 1, f1, f0, No{});
    }
    if (t < nt) iteration(t, f0, f1, No{});
  } else {
    // iteration t: tile t is read and multiplied, the stage of tile t - 1 is refilled
    Frags f;
    auto iteration = [&](int t, auto steady) {
      constexpr bool STEADY = decltype(steady)::value;
      if constexpr (STEADY) arrive(NST - 2);
      else arrive(t == 0 ? NST - 1 : min(nt - 1 - t, NST - 2));
      read(f, st);
      multiply(f);
      if (STEADY || (t > 0 && t - 1 + NST < nt)) fill(t - 1 + NST, st == 0 ? NST - 1 : st - 1);
      if (STEADY) {
        __builtin_amdgcn_sched_group_barrier(0x100, TM + TN, 0);
#pragma unroll
        for (int g = 0; g < NLD; ++g) {
          __builtin_amdgcn_sched_group_barrier(0x008, TM * TN / (NLD + 1), 0);
          __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
        }
      }
      st = next_stage(st);
      __builtin_amdgcn_sched_barrier(0);
    };
    iteration(0, No{});
    int t = 1;
    for (; t - 1 + NST < nt; ++t) iteration(t, Yes{});
    for (; t < nt; ++t) iteration(t, No{});
  }

  // ---- epilogue ----
  __builtin_amdgcn_s_waitcnt(0xC07F);
  __builtin_amdgcn_s_barrier();  // nobody reads operand stages any more
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (KG == 2) {
    // group 0 finishes the row tiles 0 and 1 of every wavefront, group 1 the tiles 2 and 3
    i32x4* red = reinterpret_cast<i32x4*>(lds);
    const int slot = (wave & 3) * 2 * TN * 64 + lane;
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int i = 0; i < 2; ++i)
        red[grp * 8 * TN * 64 + slot + (2 * j + i) * 64] = grp == 0 ? acc[j][2 + i] : acc[j][i];
    __builtin_amdgcn_s_waitcnt(0xC07F);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int i = 0; i < 2; ++i)
        acc[j][i] = (grp == 0 ? acc[j][i] : acc[j][2 + i]) + red[(1 - grp) * 8 * TN * 64 + slot + (2 * j + i) * 64];
    __builtin_amdgcn_s_waitcnt(0xC07F);
    __builtin_amdgcn_s_barrier();  // the sums have been read: the staged tile may take their place
    __builtin_amdgcn_sched_barrier(0);
  }
  if constexpr (KG == 4) {
    // group g finishes row tile g; the other groups' sums of it: [row tile][group][half of the columns][j][lane]
    i32x4* red = reinterpret_cast<i32x4*>(lds) + lane;
    auto place = [&](int tile, int g) { return ((tile * 4 + g) * 2 + wn) * TN * 64; };
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (i != grp)  // uniform
#pragma unroll
        for (int j = 0; j < TN; ++j) red[place(i, grp) + j * 64] = acc[j][i];
    __builtin_amdgcn_s_waitcnt(0xC07F);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 1; i < 4; ++i)
      if (i == grp)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[j][0] = acc[j][i];
#pragma unroll
    for (int d = 1; d < 4; ++d)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[j][0] += red[place(grp, (grp + d) & 3) + j * 64];
    __builtin_amdgcn_s_waitcnt(0xC07F);
    __builtin_amdgcn_s_barrier();  // the sums have been read: the staged tile may take their place
    __builtin_amdgcn_sched_barrier(0);
  }
  const bool full = m0 + BM <= a.M && n0 + BN <= a.N;
  unsigned short* outp = reinterpret_cast<unsigned short*>(a.out);
#pragma unroll
  for (int h = 0; h < (KG == 1 ? 2 : 1); ++h) {
    if (h > 0) {
      __builtin_amdgcn_s_waitcnt(0xC07F);
      __builtin_amdgcn_s_barrier();  // the previous half has been read
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int i = 0; i < (KG == 4 ? 1 : 2); ++i) {
      const int at = KG == 4 ? 16 * grp + lr : wm * 64 + (KG == 2 ? grp : h) * 32 + 16 * i + lr;  // row of the tile
      const int t = KG != 1 ? at : wm * 32 + 16 * i + lr;                                          // staged row
      const float sx = *reinterpret_cast<const float*>(sc + at * 4);
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int col = wn * (BN / 2) + 16 * j + 4 * lq;
        const f32x4 sw = *reinterpret_cast<const f32x4*>(sc + C::SW_OFF + col * 4);
        f32x4 bv = {0.f, 0.f, 0.f, 0.f};
        if (a.bias) bv = *reinterpret_cast<const f32x4*>(sc + C::BIAS_OFF + col * 4);
        const i32x4 v = acc[j][KG != 1 ? i : 2 * h + i];
        float y[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          // three separately rounded fp32 operations (no fused multiply-add)
          float s = (float)v[e] * sx;
          s = s * sw[e];
          y[e] = s + bv[e];
        }
        u32x2 o = {pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3])};
        if (EPI == EPI_GELU_BF16) {
          // activation of the bf16-rounded Linear output, as a separate GELU would see it
          o[0] = pack_bf16x2(gelu_erf(bf16_lo_to_f32(o[0])), gelu_erf(bf16_hi_to_f32(o[0])));
          o[1] = pack_bf16x2(gelu_erf(bf16_lo_to_f32(o[1])), gelu_erf(bf16_hi_to_f32(o[1])));
        }
        *reinterpret_cast<u32x2*>(lds + t * C::PITCH + col * 2) = o;
      }
    }
    __builtin_amdgcn_s_waitcnt(0xC07F);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int p = 0; p < C::PASSES; ++p) {
      int t, ch;
      piece(p, t, ch);
      const int m = m0 + out_row(t, h), n = n0 + ch * 8;
      if (C::PIECES % 512 != 0 && p == C::PASSES - 1 && t >= C::ROWS) continue;
      u32x4 val = *reinterpret_cast<const u32x4*>(lds + t * C::PITCH + ch * 16);
      if (EPI == EPI_RESIDUAL_BF16) {
#pragma unroll
        for (int c = 0; c < 4; ++c)
          // bf16 add of the bf16-rounded Linear output and the residual stream
          val[c] = pack_bf16x2(bf16_lo_to_f32(val[c]) + bf16_lo_to_f32(res[p][c]),
                               bf16_hi_to_f32(val[c]) + bf16_hi_to_f32(res[p][c]));
      }
      if (full || (m < a.M && n < a.N)) *reinterpret_cast<u32x4*>(outp + (int64_t)m * a.ldo + n) = val;
    }
  }
}

// Rows * 16 + TN of the tile for this output, 0 = another member: the smallest tile of which the CUs hold
// the whole output at once (us in back-to-back launches, the other members / this one, K-block major).
//   64 rows, from 20 k tiles on.  64 x 64: 635 x 5120 -> 1280 with the residual 18.4 / 11.7, 900 x 3072 -> 768 10.8 / 8.5, 724 x 1664 -> 768 9.1 / 6.2, 2392 x 1280 ->
//     256 8.4 / 5.8, 290 x 1536 -> 1984 8.9 / 6.1; 64 x 96: 1638 x 4096 -> 768 15.9 / 12.2, 1122 x 1664 -> 1024 9.5 / 7.8; 64 x 128: 1327 x 4096 -> 1280 16.7 / 14.3,
//     1450 x 1664 -> 1280 10.1 / 9.3 (128 x 96 10.0).  Of 50 such outputs none was slower.
//   128 rows, K >= 1280, from a few hundred rows on.  4096 rows: 3072 -> 768 18.8 / 14.7, 4096 -> 1024 25.6 / 21.5,
//     5120 -> 1280 38.0 / 30.0, 1280 -> 1280 14.7 / 13.0, 1536 -> 768 10.9 / 9.8; 1024 x 5120 -> 1280 23.4 / 17.4,
//     700 x 5120 -> 1280 25.1 / 17.3.  Shorter loops are start and end only: 768 -> 768 8.2 / 8.1, 1024 -> 1024 9.7 / 9.8.
//   256 rows, K >= 1280, three quarters of the CUs or more, no residual.  4096 rows: 1280 -> 5120 32.5 / 30.1 (GELU 38.4 /
//     36.6), 2560 -> 5120 57.5 / 48.9, 5120 -> 3840 77.6 / 69.5, 1280 -> 3840 25.4 / 24.8; 5000 x 2048 -> 2560 33.5 / 31.8.
//     K = 768: 4096 -> 3072 15.4 / 16.2, a lone workgroup's start and end cost more than the larger tile saves.
//   more than 256 tiles: a second round beside nothing else (8192 x 4096 -> 1024 39 / 47).
static int once_shape(int epi, const GemmArgs& a) {
  const int force = knob_or(KNOB_GEMM_ONCE, 1);
  if (force <= 0) return 0;
  if (force > 1) return force;
  if (a.K < 1280) return 0;
  auto tiles = [&](int bm, int tn) { return (int64_t)((a.M + bm - 1) / bm) * ((a.N + 32 * tn - 1) / (32 * tn)); };
  for (int tn = 2; tn <= 4; ++tn)
    if (tiles(64, tn) <= 256) return 64 * 16 + tn;
  for (int tn = 3; tn <= 5; ++tn)
    if (tiles(128, tn) <= 256) return 128 * 16 + tn;
  if (epi == EPI_RESIDUAL_BF16) return 0;
  for (int tn = 6; tn <= 10; tn += 2)
    if (tiles(256, tn) <= 256) return tiles(256, tn) >= 192 ? 256 * 16 + tn : 0;
  return 0;
}

bool gemm_i8_once_covers(int epi, const GemmArgs& a) {
  if (epi == EPI_I32 || a.dst_row || a.tile_counters || a.stream_out) return false;
  const int s = once_shape(epi, a), nk = a.K / GBK;
  // more k tiles per group than stages
  if (s / 16 == 64) return nk >= 20;
  if (s / 16 == 128) return nk % 2 == 0 && nk / 2 > 5;
  return s / 16 == 256 && nk > 5 && epi != EPI_RESIDUAL_BF16;
}

int gemm_i8_once_launch(int epi, const GemmArgs& a0, hipStream_t stream) {
  GemmArgs a = a0;
  const int shape = once_shape(epi, a), bm = shape / 16, bn = 32 * (shape % 16);
  a.tiles_m = (a.M + bm - 1) / bm;
  a.tiles_n = (a.N + bn - 1) / bn;
  a.group_m = 4;  // an XCD's 32 tiles: 4 row tiles x 8 column tiles, 2 to 4 MB of operands in its L2
  const unsigned int grid = (unsigned int)((a.tiles_m * a.tiles_n + 7) / 8 * 8);
  const bool front = a.x_pitch != GBK || a.w_pitch != GBK;  // a row-major operand
#define SF_ONCE(E, B, ...) hipLaunchKernelGGL((gemm_i8_once_kernel<E, B, __VA_ARGS__>), dim3(grid), dim3(512), 0, stream, a)
#define SF_ONCE_F(E, T) do { if (front) SF_ONCE(E, 128, T, true); else SF_ONCE(E, 128, T); } while (0)
#define SF_ONCE_128(T)                                                              \
  case 128 * 16 + T:                                                                \
    if (epi == EPI_GELU_BF16) SF_ONCE_F(EPI_GELU_BF16, T);                          \
    else if (epi == EPI_RESIDUAL_BF16) SF_ONCE_F(EPI_RESIDUAL_BF16, T);             \
    else SF_ONCE_F(EPI_SCALE_BIAS_BF16, T);                                         \
    break
#define SF_ONCE_64(T)                                                               \
  case 64 * 16 + T:                                                                 \
    if (epi == EPI_GELU_BF16) SF_ONCE(EPI_GELU_BF16, 64, T);                        \
    else if (epi == EPI_RESIDUAL_BF16) SF_ONCE(EPI_RESIDUAL_BF16, 64, T);           \
    else SF_ONCE(EPI_SCALE_BIAS_BF16, 64, T);                                       \
    break
#define SF_ONCE_256(T)                                                              \
  case 256 * 16 + T:                                                                \
    if (epi == EPI_GELU_BF16) SF_ONCE(EPI_GELU_BF16, 256, T);                       \
    else SF_ONCE(EPI_SCALE_BIAS_BF16, 256, T);                                      \
    break
  switch (shape) {
    SF_ONCE_64(2);
    SF_ONCE_64(3);
    SF_ONCE_64(4);
    SF_ONCE_128(3);
    SF_ONCE_128(4);
    SF_ONCE_128(5);
    SF_ONCE_256(6);
    SF_ONCE_256(8);
    SF_ONCE_256(10);
    default: set_error("gemm_i8_once: no tile %d", shape); return (int)SAMFAST_E_UNSUPPORTED;
  }
#undef SF_ONCE_256
#undef SF_ONCE_64
#undef SF_ONCE_128
#undef SF_ONCE_F
#undef SF_ONCE
  return check_launch("gemm_i8_once_kernel");
}

}  // namespace samfast
