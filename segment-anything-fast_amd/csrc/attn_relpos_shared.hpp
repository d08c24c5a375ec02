// Definitions shared by the attention kernels (attn_relpos.hip, attn_window_rows.hip).
#pragma once

#include "samfast_internal.hpp"
#include <type_traits>

namespace samfast {

struct AttnArgs {
  const unsigned short* q;
  const unsigned short* k;
  const unsigned short* v;
  const unsigned short* rh;  // FUSED: rel_pos_h table (2gh-1, hd); else rel_h (B,nH,N,gh)
  const unsigned short* rw;  // FUSED: rel_pos_w table (2gw-1, hd); else rel_w (B,nH,N,gw)
  unsigned short* out;
  int64_t q_sb, q_sh, q_sn;
  int64_t k_sb, k_sh, k_sn;
  int64_t v_sb, v_sh, v_sn;
  int64_t o_sb, o_sh, o_sn;
  int64_t rh_sb, rh_sh, rh_sn;
  int64_t rw_sb, rw_sh, rw_sn;
  int B, nH, gh, gw, N;
  float c;          // sm_scale * log2(e)
  float inv_scale;  // 1 / sm_scale
  // window kernel on image-ordered tokens (ws > 0): B counts images of img_h x img_w tokens,
  // a workgroup's window (iy, ix) covers tokens (iy*ws + y, ix*ws + x); positions outside the
  // image are padding tokens whose K / V rows are pad_k / pad_v (nH * hd values each)
  int img_h, img_w, ws, wins_x, wins_y;
  const unsigned short* pad_k;
  const unsigned short* pad_v;
  int relh_x8;  // attn_global_bias.hip: rel_h rows can be read 16 bytes at a time
  int rel_x2;   // window kernel: rows of the caller's factors can be read 4 bytes at a time
  int whole, parts, part_tiles;  // window kernel: items with a workgroup each; the others are `parts` workgroups of part_tiles query tiles
  // Window kernel: operands of the launches behind this one.  One word of every kSoonLine bytes is read, by wavefronts that have nothing
  // else to do, so that they stand in the last-level cache when they are wanted.  Nothing depends on it.
  // (At the end: of the arguments every launch looks at, in memory of the host's, no cache line more.)
  int soon_n;
  unsigned int soon_lines[SAMFAST_MAX_SOON];
  const unsigned int* soon[SAMFAST_MAX_SOON];
};

constexpr int kSoonLine = 64;  // what a miss of one word brings (at 128 the other halves still came from HBM)
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLazyLog2 = 8.0f;  // softmax reference lags the running maximum by at most 2^8

// The two 16-bit element types of q / k / v / out (and of the bias factors): what differs between
// them is the matrix instruction, the conversions and three bit patterns.  Eight elements travel
// as four 32-bit words (u32x4) everywhere outside these functions.
struct ElemBf16 {
  static constexpr unsigned int kOne = 0x3F80u;   // 1.0
  // global kernel with the caller's factors: how far (log2) above the maximum the exponent reference is put when it is
  // moved; bf16 probabilities keep their eight bits at any size.  note() gathers packed pairs, outgrown() says whether
  // one of them has reached 2: the top exponent bit, so that or-ing them is enough.
  static constexpr float kMargin = 16.0f;
  static SF_DEVICE unsigned int note(unsigned int seen, unsigned int w0, unsigned int w1) { return seen | w0 | w1; }
  static SF_DEVICE bool outgrown(unsigned int seen) { return (seen & 0x40004000u) != 0u; }
  // kernels with the caller's factors: the exponent reference (log2) before any key has been met.  Keys below it
  // are as good as masked.  Down to it every probability is finite: at 2^31 a reference and a difference from it
  // are each rounded by at most 64, so that a probability stays below 2^(128 - kMargin).
  static constexpr float kLowest = -2147483648.0f;
  static constexpr unsigned int kMask = 0xF149u;  // -1e30: added to a score (before the scale), it removes the key
  static SF_DEVICE f32x16 mfma(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
  static SF_DEVICE f32x4 mfma16(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
  // sixteen of k: four values a lane
  static SF_DEVICE f32x4 mfma16_short(u32x2 a, u32x2 b, f32x4 c) {
    typedef short s16x4 __attribute__((ext_vector_type(4)));
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4, a), __builtin_bit_cast(s16x4, b), c, 0, 0, 0);
  }
  static SF_DEVICE unsigned int pack2(float lo, float hi) { return pack_bf16x2(lo, hi); }
  static SF_DEVICE float lo(unsigned int w) { return bf16_lo_to_f32(w); }
  static SF_DEVICE float hi(unsigned int w) { return bf16_hi_to_f32(w); }
  static SF_DEVICE float from_bits(unsigned short h) { return bf16_bits_to_f32(h); }
};
struct ElemF16 {
  typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
  typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
  static constexpr unsigned int kOne = 0x3C00u;   // 1.0
  // as above, but a probability below 2^-14 is short of bits: the reference never stands above the maximum, and it
  // moves when a probability exceeds 2^kLazyLog2 (one v_pk_maximum3_f16 for two pairs; with bf16's
  // or, and therefore a ceiling of 2, 8 x 16 x 4096 x 80 took 820 us for 769, so often did the reference move)
  static constexpr float kMargin = 0.0f;
  static SF_DEVICE unsigned int note(unsigned int seen, unsigned int w0, unsigned int w1) {
    const f16x2 a = __builtin_bit_cast(f16x2, seen), b = __builtin_bit_cast(f16x2, w0), c = __builtin_bit_cast(f16x2, w1);
    return __builtin_bit_cast(unsigned int, __builtin_elementwise_maximum(__builtin_elementwise_maximum(a, b), c));
  }
  static SF_DEVICE bool outgrown(unsigned int seen) {
    const f16x2 m = __builtin_bit_cast(f16x2, seen);
    return m[0] > (_Float16)256.0f || m[1] > (_Float16)256.0f;
  }
  static constexpr float kLowest = -134217728.0f;  // as above, with 2^27, roundings of 4 and the end of the type at 2^16
  static constexpr unsigned int kMask = 0xFB53u;  // -60000 (fp16 ends at 65504): times scale*log2(e) still below -2^12
  static SF_DEVICE f32x16 mfma(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
  static SF_DEVICE f32x4 mfma16(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
  static SF_DEVICE f32x4 mfma16_short(u32x2 a, u32x2 b, f32x4 c) {
    typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
    return __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(f16x4, a), __builtin_bit_cast(f16x4, b), c, 0, 0, 0);
  }
  static SF_DEVICE unsigned int pack2(float lo, float hi) {  // round to nearest even
    const f32x2 v = {lo, hi};
    return __builtin_bit_cast(unsigned int, __builtin_convertvector(v, f16x2));
  }
  static SF_DEVICE float from_bits(unsigned short h) { return (float)__builtin_bit_cast(_Float16, h); }
  static SF_DEVICE float lo(unsigned int w) { return from_bits((unsigned short)(w & 0xffffu)); }
  static SF_DEVICE float hi(unsigned int w) { return from_bits((unsigned short)(w >> 16)); }
};

// Walks them (see AttnArgs::soon) in chunks of 64 lines, every `step`th one; all of it uniform.
struct SoonWalk {
  const AttnArgs& a;
  int s = 0;
  unsigned int line, lines;  // of operand s: the chunk's first, and all
  const unsigned int* p;
  SF_DEVICE SoonWalk(const AttnArgs& args, unsigned int chunk) : a(args), line(64u * chunk), lines(args.soon_lines[0]), p(args.soon[0]) {}
  SF_DEVICE bool more() {
    while (s < a.soon_n && line >= lines) {
      line -= (lines + 63u) & ~63u;  // (to chunks: at least this much)
      if (++s < a.soon_n) {
        lines = a.soon_lines[s];
        p = a.soon[s];
      }
    }
    return s < a.soon_n;
  }
  SF_DEVICE const unsigned int* word(int lane) const { return p + (kSoonLine / 4) * min(line + lane, lines - 1u); }
  SF_DEVICE void on(unsigned int step) { line += 64u * step; }
};

SF_DEVICE u32x4 load_x8_global(const unsigned short* p) { return *reinterpret_cast<const u32x4*>(p); }

template <typename T>
SF_DEVICE u32x4 cvt_x8(const f32x16& s, int base) {
  u32x4 w;
#pragma unroll
  for (int i = 0; i < 4; ++i) w[i] = T::pack2(s[base + 2 * i], s[base + 2 * i + 1]);
  return w;
}

// max(v, v of lane ^ 32) without an LDS round trip: v_permlane32_swap exchanges the upper half
// of its first operand with the lower half of its second, after which every lane holds its own
// value in one of the two and its partner's in the other
SF_DEVICE float max_with_lane_xor32(float v) {
  typedef unsigned int u32x2_t __attribute__((ext_vector_type(2)));
  const unsigned int b = __float_as_uint(v);
  const u32x2_t r = __builtin_amdgcn_permlane32_swap(b, b, false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// One wave instruction: 64 pieces of 16 bytes from base + off to LDS at `dst` (piece of lane l: dst + 16 l).
// Written out because the compiler would make every LDS read that follows wait for the builtin's loads;
// whoever calls it waits for the arrival by hand (vmcnt) before the barrier in front of the readers.  The destination is
// an operand in m0, so that the compiler knows the register is taken and moves it there itself.
SF_DEVICE void lds_dma16(const unsigned char* base, unsigned int off, unsigned int dst) {
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(off), "s"(base), "{m0}"(dst) : "memory");
}

// How the global kernels keep one key grid row (64 keys) of K and of V in LDS: rows of 16-byte pieces, placed so
// that no read of a wavefront meets a bank twice.
//   K is read 16 bytes per lane, 32 keys at a time.  HD = 64: 128-byte rows, piece c of row r at position
//   c ^ (r / 2 % 8); HD = 80: 160-byte rows, position c ^ (r / 8 % 2).
//   V is read by ds_read_b64_tr_b16, four keys x 64 bytes per half wavefront.  HD = 64: the row's two 64-byte
//   halves change places in rows 2, 3 of every four; HD = 80: 192-byte rows (16 words past a multiple of
//   the banks), the two spare pieces hold (1, 0, ...) and zeros: channel 80 of every key is one, and
//   the P V product delivers the softmax denominator in its otherwise unused output rows.
template <int HD>
struct GridRow {
  static constexpr int KS = HD / 16;           // score k-steps
  static constexpr int DT = (HD + 31) / 32;    // output channel tiles
  static constexpr bool ONES_ROW = HD % 32 != 0;
  static constexpr int KP = HD / 8, VP = ONES_ROW ? 12 : HD / 8;  // pieces per row = wave instructions per tile
  static constexpr int KTILE = 64 * KP * 16, VTILE = 64 * VP * 16;
  static SF_DEVICE int k_swizzle(int row) { return HD == 64 ? (row >> 1) & 7 : (row >> 3) & 1; }
  // byte offset inside the source row of the piece at LDS position P of a tile (or -1: a spare piece)
  static SF_DEVICE int k_source(int P, int& row) {
    row = P / KP;
    return ((P % KP) ^ k_swizzle(row)) * 16;
  }
  static SF_DEVICE int v_source(int P, int& row) {
    row = P / VP;
    const int pos = P % VP;
    if (ONES_ROW) return pos < HD / 8 ? pos * 16 : -1;
    return (pos ^ (4 * ((row >> 1) & 1))) * 16;
  }
  // LDS offset inside a K tile of the lane's operand piece (key lr, channels 16 ks + 8 lh)
  static SF_DEVICE int k_read(int lr, int lh, int ks) { return lr * (KP * 16) + (((2 * ks + lh) ^ k_swizzle(lr)) * 16); }
  // LDS offset inside a V tile of the lane's transposing read, output tile dt (key and channel of a source lane:
  // see attn_global_kernel)
  static SF_DEVICE int v_read(int lane, int dt) {
    const int g = lane >> 4, sl = lane & 15, key = 4 * (g >> 1) + (sl >> 2);
    const int half = ONES_ROW ? dt : dt ^ ((key >> 1) & 1);
    return key * (VP * 16) + half * 64 + 32 * (g & 1) + 8 * (sl & 3);
  }
};

// A factor of the caller's as an operand of the window kernels' bias products, whose other operand is zeros and ones: divided
// by the scale and not below T::kMask, the value that takes a key away (0 * -inf would be a NaN for every key; a NaN stays one).
template <typename T>
SF_DEVICE float bias_slot(float factor, const AttnArgs& a) {
  return __builtin_elementwise_maximum(factor * a.inv_scale, T::from_bits(T::kMask));
}

// all LDS operations this wavefront has issued are complete and ordered
SF_DEVICE void wave_lds_fence() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// one-hot vector of eight 16-bit elements: element e is 1.0 iff slot == 8*lh + e
template <typename T>
SF_DEVICE u32x4 onehot_x8(int slot, int lh) {
  const int e = slot - 8 * lh;  // may be outside [0, 8)
  u32x4 w;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    unsigned int v = 0u;
    if ((e >> 1) == i) v = (e & 1) ? (T::kOne << 16) : T::kOne;
    w[i] = v;
  }
  return w;
}

// Global attention with caller-computed bias factors (attn_global_bias.hip)
int attn_global_bias_launch(const AttnArgs& a, int hd, int dtype, hipStream_t stream);

// Window kernel with the keys laid out as grid rows padded to 16 (attn_window_rows.hip): whether it
// covers the call (gw <= 16, gh <= 14) and its launch.
bool attn_window_rows_covers(const AttnArgs& a);
int attn_window_rows_launch(const AttnArgs& a, int hd, int dtype, bool fused, hipStream_t stream);

}  // namespace samfast
