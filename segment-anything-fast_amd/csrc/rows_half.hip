// Row-wise glue of a block whose Linears stay in the half type (no quantiser): residual add + LayerNorm in
// one pass, and the exact-erf GELU.  Both are memory-bound: what they save is passes - the add reads and
// writes the residual stream once and hands the normalised row on in the same launch, instead of an add
// kernel and a LayerNorm kernel (five row passes against four, and one launch against two).
#include "quant_row.hpp"
#include "attn_relpos_shared.hpp"

namespace samfast {

struct RowsArgs {
  const unsigned short* x;
  const unsigned short* r;  // ADD: added to x (rounded to the element type), may be null otherwise
  const unsigned short* gamma;
  const unsigned short* beta;
  unsigned short* sum;      // ADD: x + r
  unsigned short* out;      // LayerNorm of the row
  int64_t M;
  int K;
  float eps, inv_K;
};

constexpr int kRowWaves = 4;

// One wavefront per row; a lane holds chunks lane, lane + 64, ... of EPC elements (8, or 4 where that divides
// the row among the lanes exactly and 8 does not: 768, 1280).  Two-pass statistics in fp32, as the
// quantiser's LayerNorm.  4096 x 1280 (10.5 MB per operand, all in the last-level cache): 7.5 us with the add.
template <typename T, int NCH, int EPC, bool ADD>
__global__ __launch_bounds__(64 * kRowWaves) void layernorm_rows_kernel(RowsArgs a) {
  constexpr int W = EPC / 2;
  typedef unsigned int in_t __attribute__((ext_vector_type(W)));
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * kRowWaves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (row >= a.M) return;
  const int nchunk = a.K / EPC;
  const in_t* xs = reinterpret_cast<const in_t*>(a.x + row * a.K);
  const in_t* rs = reinterpret_cast<const in_t*>(a.r + row * a.K);
  const in_t* g4 = reinterpret_cast<const in_t*>(a.gamma);
  const in_t* b4 = reinterpret_cast<const in_t*>(a.beta);
  in_t xw[NCH], rw[NCH], gw[NCH], bw[NCH];
#pragma unroll
  for (int i = 0; i < NCH; ++i) {
    const int c = lane + 64 * i;
    const in_t z = {};
    xw[i] = rw[i] = z;
    if (c < nchunk) {
      xw[i] = xs[c];
      if (ADD) rw[i] = rs[c];
    }
    const int cc = min(c, nchunk - 1);
    gw[i] = g4[cc];
    bw[i] = b4[cc];
  }
  float f[NCH][EPC];
  float s1 = 0.f;
#pragma unroll
  for (int i = 0; i < NCH; ++i) {
    in_t sw;
#pragma unroll
    for (int j = 0; j < W; ++j) {
      sw[j] = ADD ? T::pack2(T::lo(xw[i][j]) + T::lo(rw[i][j]), T::hi(xw[i][j]) + T::hi(rw[i][j])) : xw[i][j];
      f[i][2 * j] = T::lo(sw[j]);
      f[i][2 * j + 1] = T::hi(sw[j]);
      s1 += f[i][2 * j] + f[i][2 * j + 1];
    }
    if (ADD && lane + 64 * i < nchunk) reinterpret_cast<in_t*>(a.sum + row * a.K)[lane + 64 * i] = sw;
  }
  const float mean = wave_sum(s1) * a.inv_K;
  float s2 = 0.f;
#pragma unroll
  for (int i = 0; i < NCH; ++i)
    if (lane + 64 * i < nchunk) {
#pragma unroll
      for (int e = 0; e < EPC; ++e) {
        f[i][e] -= mean;
        s2 = fmaf(f[i][e], f[i][e], s2);
      }
    }
  const float rstd = __builtin_amdgcn_rsqf(fmaf(wave_sum(s2), a.inv_K, a.eps));
#pragma unroll
  for (int i = 0; i < NCH; ++i)
    if (lane + 64 * i < nchunk) {
      in_t o;
#pragma unroll
      for (int j = 0; j < W; ++j)
        o[j] = T::pack2(fmaf(f[i][2 * j] * rstd, T::lo(gw[i][j]), T::lo(bw[i][j])),
                        fmaf(f[i][2 * j + 1] * rstd, T::hi(gw[i][j]), T::hi(bw[i][j])));
      reinterpret_cast<in_t*>(a.out + row * a.K)[lane + 64 * i] = o;
    }
}

template <typename T, bool ADD>
static int launch_layernorm(const RowsArgs& a, hipStream_t stream) {
  const dim3 grid((unsigned int)((a.M + kRowWaves - 1) / kRowWaves)), block(64 * kRowWaves);
  auto go = [&](auto nch, auto epc) {
    hipLaunchKernelGGL((layernorm_rows_kernel<T, decltype(nch)::value, decltype(epc)::value, ADD>), grid, block, 0, stream, a);
    return check_launch("layernorm_rows_kernel");
  };
  using std::integral_constant;
  using E4 = integral_constant<int, 4>;
  using E8 = integral_constant<int, 8>;
  if (a.K == 768) return go(integral_constant<int, 3>{}, E4{});
  if (a.K == 1280) return go(integral_constant<int, 5>{}, E4{});
  // the neck's 256 channels: every lane holds four of them (with 8 per lane half of the wavefront idles)
  if (a.K <= 256) return go(integral_constant<int, 1>{}, E4{});
  const int need = (a.K / 8 + 63) / 64;
  if (need <= 1) return go(integral_constant<int, 1>{}, E8{});
  if (need <= 2) return go(integral_constant<int, 2>{}, E8{});
  if (need <= 4) return go(integral_constant<int, 4>{}, E8{});
  return go(integral_constant<int, 8>{}, E8{});
}

// 16 bytes per lane and step; a workgroup covers 8 KB with both its steps in flight, and there are as many as that takes
// (4096 that loop: 303 us for 335 M values, this way 229).  4096 x 5120: 14.2 us, 5 x 4096 x 4096: 48.
template <typename T>
__global__ __launch_bounds__(256) void gelu_kernel(const unsigned short* x, unsigned short* y, int64_t chunks) {
  const int64_t stride = (int64_t)gridDim.x * 256;
  for (int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x; c < chunks; c += 2 * stride) {
    const bool second = c + stride < chunks;
    u32x4 v[2];
    v[0] = reinterpret_cast<const u32x4*>(x)[c];
    if (second) v[1] = reinterpret_cast<const u32x4*>(x)[c + stride];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      if (s == 1 && !second) break;
#pragma unroll
      for (int j = 0; j < 4; ++j) v[s][j] = T::pack2(gelu_value(T::lo(v[s][j])), gelu_value(T::hi(v[s][j])));
      reinterpret_cast<u32x4*>(y)[c + s * stride] = v[s];
    }
  }
}

}  // namespace samfast

extern "C" int samfast_layernorm(const void* x, const void* r, const void* gamma, const void* beta, float eps,
                                 void* sum, void* out, int64_t M, int K, int dtype, void* stream) {
  using namespace samfast;
  using us = unsigned short;
  if (dtype != SAMFAST_BF16 && dtype != SAMFAST_F16) SF_FAIL(SAMFAST_E_UNSUPPORTED, "layernorm: element type %d is neither SAMFAST_BF16 nor SAMFAST_F16", dtype);
  SF_REQUIRE(M >= 0 && K > 0 && K % 8 == 0 && K <= 4096, "layernorm: bad shape M=%lld K=%d (K must be a multiple of 8, <= 4096)", (long long)M, K);
  SF_REQUIRE((M + 3) / 4 < (1ll << 31), "layernorm: M too large");
  SF_REQUIRE((r == nullptr) == (sum == nullptr), "layernorm: the added rows and the sum go together");
  SF_REQUIRE(M == 0 || (x && gamma && beta && out), "layernorm: null pointer");
  SF_REQUIRE(eps >= 0.f, "layernorm: eps must not be negative");
  SF_REQUIRE(aligned16(x) && aligned16(r) && aligned16(gamma) && aligned16(beta) && aligned16(sum) && aligned16(out),
             "layernorm: operands must be 16-byte aligned");
  if (M == 0) return SAMFAST_OK;
  RowsArgs a = {(const us*)x, (const us*)r, (const us*)gamma, (const us*)beta, (us*)sum, (us*)out, M, K, eps, 1.0f / (float)K};
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  if (dtype == SAMFAST_F16) return r ? launch_layernorm<ElemF16, true>(a, s) : launch_layernorm<ElemF16, false>(a, s);
  return r ? launch_layernorm<ElemBf16, true>(a, s) : launch_layernorm<ElemBf16, false>(a, s);
}

extern "C" int samfast_gelu(const void* x, void* y, int64_t n, int dtype, void* stream) {
  using namespace samfast;
  if (dtype != SAMFAST_BF16 && dtype != SAMFAST_F16) SF_FAIL(SAMFAST_E_UNSUPPORTED, "gelu: element type %d is neither SAMFAST_BF16 nor SAMFAST_F16", dtype);
  SF_REQUIRE(n >= 0 && n % 8 == 0, "gelu: %lld values are not a multiple of 8", (long long)n);
  SF_REQUIRE(n == 0 || (x && y && aligned16(x) && aligned16(y)), "gelu: null or unaligned pointer");
  if (n == 0) return SAMFAST_OK;
  const int64_t chunks = n / 8;
  const unsigned int grid = (unsigned int)min((chunks + 511) / 512, (int64_t)1 << 30);
  if (dtype == SAMFAST_F16)
    hipLaunchKernelGGL(gelu_kernel<ElemF16>, dim3(grid), dim3(256), 0, reinterpret_cast<hipStream_t>(stream), (const unsigned short*)x, (unsigned short*)y, chunks);
  else
    hipLaunchKernelGGL(gelu_kernel<ElemBf16>, dim3(grid), dim3(256), 0, reinterpret_cast<hipStream_t>(stream), (const unsigned short*)x, (unsigned short*)y, chunks);
  return check_launch("gelu_kernel");
}
