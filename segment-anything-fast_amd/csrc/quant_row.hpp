// The per-row int8 quantiser (optionally behind a LayerNorm) as device code shared by the
// stand-alone kernels (quant_rowwise.hip) and by the int8 GEMM, whose last workgroup of a row
// tile quantises the rows the tile's workgroups have just written (gemm_i8.hip).  One
// wavefront owns one row; both users run exactly this code, so their codes and scales agree
// bit for bit.
#pragma once

#include "samfast_internal.hpp"

// every fp32 step below is rounded on its own (no fused multiply-add), so results
// can be reproduced bit for bit on a CPU
#pragma clang fp contract(off)

namespace samfast {

struct QuantArgs {
  const unsigned short* x;
  int64_t ldx;
  const unsigned short* gamma;  // LN only
  const unsigned short* beta;   // LN only
  const int32_t* src_row;       // LN only: source row per output row, -1 = all-zero row; may be null
  int8_t* xq;
  float* sx;
  int64_t M;
  int K;
  float eps;
  float inv_K;  // 1 / K for the LayerNorm statistics
  int kb64;  // 1: write xq K-block major, (K/64, M, 64)
};

// Wavefront-wide reductions without LDS traffic: four DPP steps combine the 16 lanes of a row
// (lane ^ 1, lane ^ 2, then the mirrored half row and the mirrored row, which by then hold the
// other quad's / other half's partial result), two lane-swap steps combine the four rows.
template <int CTRL>
SF_DEVICE float dpp_f32(float v) {
  return __uint_as_float((unsigned int)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(v), CTRL, 0xf, 0xf, true));
}
template <typename Op>
SF_DEVICE float wave_reduce(float v, Op op) {
  v = op(v, dpp_f32<0xB1>(v));   // quad_perm [1, 0, 3, 2]
  v = op(v, dpp_f32<0x4E>(v));   // quad_perm [2, 3, 0, 1]
  v = op(v, dpp_f32<0x141>(v));  // row_half_mirror
  v = op(v, dpp_f32<0x140>(v));  // row_mirror
  typedef unsigned int u32x2_t __attribute__((ext_vector_type(2)));
  unsigned int b = __float_as_uint(v);
  u32x2_t r = __builtin_amdgcn_permlane16_swap(b, b, false, false);  // rows 0<->1, 2<->3
  v = op(__uint_as_float(r[0]), __uint_as_float(r[1]));
  b = __float_as_uint(v);
  r = __builtin_amdgcn_permlane32_swap(b, b, false, false);          // halves of the wavefront
  return op(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
SF_DEVICE float wave_sum(float v) {
  return wave_reduce(v, [](float x, float y) { return x + y; });
}
// for values >= 0 (absolute maxima): the bit patterns order like the values, and the unsigned
// maximum needs no canonicalisation of its operands
SF_DEVICE float wave_max_nonneg(float v) {
  return wave_reduce(v, [](float x, float y) {
    return __uint_as_float(max(__float_as_uint(x), __float_as_uint(y)));
  });
}

// A row's scale and the factor that codes are made with: code = rint(v * factor), rounded once.
// The code wanted is rint(fl(v / scale)) with the correctly rounded IEEE quotient.  Values and maximum are bf16, so the exact
// 127 v / amax is a tie (k + 1/2) only at v = amax / 2, where it is 63.5, and, if 127 divides amax's significand (254), at ties of both parities for which
// scale and 1 / scale are powers of two; elsewhere it stays 2^-16 of its size and more away from one, beyond what the roundings of scale, quotient and
// factor (2^-24 each) move.  So any factor within a few units of 1 / scale gives the division's codes but for v = amax / 2, and there the
// factor is moved by one unit to the side on which the division lies: its quotient is 63.5 or more (code 64) where m >= scale * (127 - 2^-18), m being
// the maximum at its floor; the residual of m / scale is exact in one fused multiply-add.  All pairs of a bf16 row maximum and a bf16 value up to it
// (5.3e8) give the division's code.  In a row with an infinity the factor is 0: the codes are 0, as the low byte of the division's NaN.
struct QuantScale {
  float scale, factor;
  SF_DEVICE explicit QuantScale(float amax) {
    const float m = fmaxf(amax, 1e-5f);
    scale = m / 127.0f;
    const float inv = 1.0f / scale;
    const bool up = fmaf(-scale, 127.0f, m) >= scale * -0x1p-18f;  // the division gives 64
    const float over = fmaf(0.5f * m, inv, -63.5f);                // (exact in its sign)
    factor = __uint_as_float(__float_as_uint(inv) + (up && over < 0.f ? 1u : !up && over >= 0.f ? -1u : 0u));
  }
};

// EPC (4 or 8) values -> EPC int8 codes packed in EPC bytes.
// Adding 1.5 * 2^23 in the same fused multiply-add rounds the exact product half to even and leaves the code in the low
// byte (|v * factor| <= 127 (1 + 2^-22)).  One instruction per value; with the quotient itself made exact (q = v * inv, then q + (v - q * scale) *
// inv, then the addition: four) 188 / 382 / 1593 vector instructions per row of 1280 plain / 1280 with LayerNorm / 5120 with GELU, now 144 / 338 / 1374.
template <int EPC>
SF_DEVICE void quantize_chunk(const float (&v)[EPC], const QuantScale& s, unsigned int (&out)[EPC / 4]) {
  unsigned int m[EPC];
#pragma unroll
  for (int e = 0; e < EPC; ++e) m[e] = __float_as_uint(fmaf(v[e], s.factor, 12582912.0f));
#pragma unroll
  for (int g = 0; g < EPC / 4; ++g) {
    // byte 0 of each of four words -> one word (v_perm_b32: selector bytes pick from {hi, lo})
    const unsigned int lo = __builtin_amdgcn_perm(m[4 * g + 1], m[4 * g], 0x0c0c0400u);      // [m0.b0, m1.b0, 0, 0]
    const unsigned int hi = __builtin_amdgcn_perm(m[4 * g + 3], m[4 * g + 2], 0x04000c0cu);  // [0, 0, m2.b0, m3.b0]
    out[g] = lo | hi;
  }
}

// Absolute maximum of what the wavefront's lanes hold, without NaNs; returns whether there was one.  The maximum of the common path
// hands NaNs on, which costs nothing; a row with one is looked through again.
template <int N, int EPC>
SF_DEVICE bool wave_absmax(const float (&f)[N][EPC], float& amax) {
  amax = 0.f;
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int e = 0; e < EPC; ++e) amax = __builtin_elementwise_maximum(amax, fabsf(f[i][e]));
  amax = wave_max_nonneg(fabsf(amax));
  if (__builtin_amdgcn_readfirstlane(__float_as_uint(amax)) <= 0x7f800000u) return false;
  asm volatile("");  // (not to be run ahead of the branch)
  amax = 0.f;
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int e = 0; e < EPC; ++e) amax = fmaxf(amax, fabsf(f[i][e]));
  amax = wave_max_nonneg(amax);
  return true;
}

// A lane holds chunks lane, lane + 64, ... of EPC elements (NCH of them: K <= NCH * 64 * EPC).
// EPC = 8 (16-byte loads) is the general case; EPC = 4 (8-byte loads) is taken when it divides the
// row among the lanes without a remainder and EPC = 8 does not (K = 1280: five chunks of 4 per
// lane instead of three chunks of 8 of which the third is half empty).
template <int NCH, int EPC, bool LN>
struct RowQuantizer {
  static_assert(EPC == 4 || EPC == 8, "chunk width");
  static constexpr int W = EPC / 2;  // 32-bit words per input chunk
  typedef unsigned int in_t __attribute__((ext_vector_type(W)));

  // Requests the lane's chunks of one source row; nothing here waits for the data.
  // STREAM: the row is read once and never again (the 671 MB lin1 output at ViT-H batch 16).
  template <bool STREAM>
  static SF_DEVICE void load_row(const unsigned short* row_ptr, int nchunk, int lane, in_t (&xw)[NCH]) {
    const in_t* src = reinterpret_cast<const in_t*>(row_ptr);
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int c = lane + i * 64;
      const in_t z = {};
      xw[i] = z;
      if (c < nchunk) xw[i] = STREAM ? __builtin_nontemporal_load(src + c) : src[c];
    }
  }
  // the lane's slices of gamma and beta (LN): independent of the row
  static SF_DEVICE void load_affine(const unsigned short* gamma, const unsigned short* beta, int nchunk,
                                    int lane, in_t (&gw)[NCH], in_t (&bw)[NCH]) {
    const in_t* g4 = reinterpret_cast<const in_t*>(gamma);
    const in_t* b4 = reinterpret_cast<const in_t*>(beta);
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int c = min(lane + i * 64, nchunk - 1);
      gw[i] = g4[c];
      bw[i] = b4[c];
    }
  }

  // chunk 64 i + lane of output row `row` (i uniform): row-major at row*K + EPC*c; K-block major at
  // ((c*EPC/64)*M + row)*64 + (c*EPC)%64.  Written as a uniform base plus an unsigned 32-bit lane offset - M*K < 2^31 is
  // checked on the host - that is the same for every i: the stores take the scalar-base form and nothing of the address is
  // computed per chunk and lane.
  static SF_DEVICE void store_chunk(const QuantArgs& a, int64_t row, int i, int lane, const unsigned int (&codes)[EPC / 4]) {
    const unsigned int k = (unsigned int)lane * EPC;
    int8_t* base;
    unsigned int off;
    if (a.kb64) {
      base = a.xq + row * 64 + (int64_t)(i * EPC) * (a.M * 64);
      off = (k >> 6) * ((unsigned int)a.M * 64u) + (k & 63u);
    } else {
      base = a.xq + row * (int64_t)a.K + i * (64 * EPC);
      off = k;
    }
    unsigned int* dst = reinterpret_cast<unsigned int*>(base + off);
    if (EPC == 8) {
      const u32x2 o = {codes[0], codes[EPC / 4 - 1]};
      *reinterpret_cast<u32x2*>(dst) = o;
    } else {
      *dst = codes[0];
    }
  }

  // an all-zero output row (a padding token): codes 0, scale at its floor
  static SF_DEVICE void zero_row(const QuantArgs& a, int64_t row, int nchunk, int lane) {
    const unsigned int z[EPC / 4] = {};
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int c = lane + i * 64;
      if (c < nchunk) store_chunk(a, row, i, lane, z);
    }
    if (lane == 0) a.sx[row] = 1e-5f / 127.0f;
  }

  // gamma and beta (LN) as they were loaded, unpacked where they are used, or unpacked once for many rows
  struct PackedAffine {
    const in_t (&g)[NCH];
    const in_t (&b)[NCH];
    SF_DEVICE float gamma(int i, int e) const { return e % 2 ? bf16_hi_to_f32(g[i][e / 2]) : bf16_lo_to_f32(g[i][e / 2]); }
    SF_DEVICE float beta(int i, int e) const { return e % 2 ? bf16_hi_to_f32(b[i][e / 2]) : bf16_lo_to_f32(b[i][e / 2]); }
  };
  struct PlainAffine {
    float g[NCH][EPC], b[NCH][EPC];
    SF_DEVICE PlainAffine(const in_t (&gw)[NCH], const in_t (&bw)[NCH]) {
      const PackedAffine p = {gw, bw};
#pragma unroll
      for (int i = 0; i < NCH; ++i)
#pragma unroll
        for (int e = 0; e < EPC; ++e) g[i][e] = p.gamma(i, e), b[i][e] = p.beta(i, e);
    }
    SF_DEVICE float gamma(int i, int e) const { return g[i][e]; }
    SF_DEVICE float beta(int i, int e) const { return b[i][e]; }
  };

  // Everything after the loads: (LayerNorm,) absmax, scale, codes of output row `row`.
  static SF_DEVICE void finish_row(const QuantArgs& a, int64_t row, int nchunk, int lane,
                                   const in_t (&xw)[NCH], const in_t (&gw)[NCH], const in_t (&bw)[NCH]) {
    finish_row(a, row, nchunk, lane, xw, PackedAffine{gw, bw});
  }
  template <typename Affine>
  static SF_DEVICE void finish_row(const QuantArgs& a, int64_t row, int nchunk, int lane, const in_t (&xw)[NCH], const Affine& affine) {
    const float scale = finish(a, nchunk, lane, xw, affine, [&](int i, const unsigned int (&codes)[EPC / 4]) { store_chunk(a, row, i, lane, codes); });
    if (lane == 0) a.sx[row] = scale;
  }

  // The same with the codes of chunk 64 i + lane handed to store(i, codes); returns the row's scale (in every lane).
  template <typename Store>
  static SF_DEVICE float finish(const QuantArgs& a, int nchunk, int lane, const in_t (&xw)[NCH], const in_t (&gw)[NCH], const in_t (&bw)[NCH],
                                Store store) {
    return finish(a, nchunk, lane, xw, PackedAffine{gw, bw}, store);
  }
  template <typename Affine, typename Store>
  static SF_DEVICE float finish(const QuantArgs& a, int nchunk, int lane, const in_t (&xw)[NCH], const Affine& affine, Store store) {
    // the row as floats, unpacked once
    float f[NCH][EPC];
#pragma unroll
    for (int i = 0; i < NCH; ++i)
#pragma unroll
      for (int j = 0; j < W; ++j) {
        f[i][2 * j] = bf16_lo_to_f32(xw[i][j]);
        f[i][2 * j + 1] = bf16_hi_to_f32(xw[i][j]);
      }

    if (LN) {
      // two-pass mean / biased variance over the K real elements, fp32
      float s1 = 0.f;
#pragma unroll
      for (int i = 0; i < NCH; ++i)
#pragma unroll
        for (int j = 0; j < W; ++j) s1 += f[i][2 * j] + f[i][2 * j + 1];
      // statistics: multiplication by 1/K and a hardware reciprocal square root (1 ulp each; the
      // LayerNorm result is compared with the reference to one code step, not bit for bit)
      const float mean = wave_sum(s1) * a.inv_K;
      float s2 = 0.f;
#pragma unroll
      for (int i = 0; i < NCH; ++i) {
        if (lane + i * 64 < nchunk) {
#pragma unroll
          for (int j = 0; j < W; ++j) {
            const float d0 = f[i][2 * j] - mean, d1 = f[i][2 * j + 1] - mean;
            f[i][2 * j] = d0;
            f[i][2 * j + 1] = d1;
            s2 = fmaf(d1, d1, fmaf(d0, d0, s2));
          }
        }
      }
      const float rstd = __builtin_amdgcn_rsqf(fmaf(wave_sum(s2), a.inv_K, a.eps));
#pragma unroll
      for (int i = 0; i < NCH; ++i) {
        const int c = lane + i * 64;
        if (c < nchunk) {
#pragma unroll
          for (int j = 0; j < W; ++j) {
            // (x - mean) * rstd, then one fused multiply-add with gamma and beta
            const float y0 = fmaf(f[i][2 * j] * rstd, affine.gamma(i, 2 * j), affine.beta(i, 2 * j));
            const float y1 = fmaf(f[i][2 * j + 1] * rstd, affine.gamma(i, 2 * j + 1), affine.beta(i, 2 * j + 1));
            const unsigned int y = pack_bf16x2(y0, y1);  // the bf16 values a separate LayerNorm would have stored
            f[i][2 * j] = bf16_lo_to_f32(y);
            f[i][2 * j + 1] = bf16_hi_to_f32(y);
          }
        }
      }
    }

    float amax;
    // a row that holds a NaN gets a NaN scale, so that the Linear reading it returns NaN for this row as a float Linear would
    const bool row_nan = wave_absmax(f, amax);
    const QuantScale q(amax);
#pragma unroll
    for (int i = 0; i < NCH; ++i)
      if (lane + i * 64 < nchunk) {
        unsigned int codes[EPC / 4];
        quantize_chunk<EPC>(f[i], q, codes);
        store(i, codes);
      }
    return row_nan ? __uint_as_float(0x7fc00000u) : q.scale;
  }
};

// (NCH, EPC) the stand-alone kernels and the GEMM tail use for a row of K elements: 4-element
// chunks where they divide the row among the 64 lanes exactly and 8-element chunks do not
constexpr int quant_epc_for(int K) { return (K == 768 || K == 1280) ? 4 : 8; }
constexpr int quant_nch_for(int K) {
  if (K == 768) return 3;
  if (K == 1280) return 5;
  const int need = (K / 8 + 63) / 64;
  return need <= 2 ? 2 : need <= 3 ? 3 : need <= 4 ? 4 : need <= 6 ? 6 : need <= 8 ? 8
       : need <= 10 ? 10 : need <= 12 ? 12 : 16;
}

}  // namespace samfast
