// Sam.preprocess for the encoder's half type in one launch: (x - mean) / std per channel in fp32, zeros to the right and below, rounded to
// the type the encoder reads.  As tensor operations it is five passes over up to 12 MB of fp32, 34 us of one image; one
// pass over the pixels is bound by its launch: 5.4 us.
#include "attn_relpos_shared.hpp"

// subtraction and division rounded one by one, as the tensor operations round them
#pragma clang fp contract(off)

namespace samfast {

struct PreprocessArgs {
  const void* x;      // (B, 3, h, w)
  const float* mean;  // 3 values each
  const float* std;
  unsigned short* y;  // (B, 3, S, S)
  int64_t chunks;     // of eight outputs
  int h, w, S;
};

template <class Out, typename In>
__global__ __launch_bounds__(256) void preprocess_kernel(PreprocessArgs a) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= a.chunks) return;
  const int per_row = a.S / 8;
  const int c0 = (int)(i % per_row) * 8;
  const int64_t row = i / per_row;  // of (B, 3, S)
  const int r = (int)(row % a.S);
  const int64_t plane = row / a.S;
  u32x4 o = {0u, 0u, 0u, 0u};
  if (r < a.h && c0 < a.w) {
    const float mean = a.mean[plane % 3], std = a.std[plane % 3];
    const In* src = reinterpret_cast<const In*>(a.x) + (plane * a.h + r) * a.w + c0;
    In v[8];
    const int n = min(8, a.w - c0);
    if (n == 8) {
      __builtin_memcpy(v, src, 8 * sizeof(In));  // (rows of any length: no alignment is assumed)
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = e < n ? src[e] : (In)0;
    }
    float f[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) f[e] = e < n ? ((float)v[e] - mean) / std : 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = Out::pack2(f[2 * e], f[2 * e + 1]);
  }
  reinterpret_cast<u32x4*>(a.y)[i] = o;
}

// Patches of 16 x 16 pixels as rows (channel, y, x), what the patch embedding multiplies.  A wavefront takes four patches' pixels of one channel, 16 bytes a
// lane: whole 128-byte lines of eight image rows, then of the eight below, and runs of 256 bytes to each patch's row.  Bound by its launch and two passes over the pixels:
// us, recorded, a permuted copy by torch / this: one image of 1024 x 1024 7.8 / 3.6, two 14.6 / 4.9, five 28.0 / 10.7, sixteen 77.6 / 30.6 (6.6 TB/s).
struct PatchArgs {
  const u32x4* x;  // (B, C, 16 gh, 16 gw), pieces of eight pixels
  u32x4* y;        // (B, gh, gw, C, 16, 2)
  unsigned int waves;
  int C, gh, gw, groups;  // groups of four patches in a row of them
};

__global__ __launch_bounds__(256) void patch_rows_kernel(PatchArgs a) {
  const unsigned int w = blockIdx.x * 4u + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (w >= a.waves) return;
  const int lane = threadIdx.x & 63, dy = lane >> 3, half = lane & 1;
  const int gx = 4 * (int)(w % a.groups) + ((lane >> 1) & 3);
  unsigned int q = w / a.groups;
  const int c = (int)(q % a.C);
  q /= a.C;
  const int gy = (int)(q % a.gh);
  const int64_t b = q / a.gh;
  if (gx >= a.gw) return;
  const u32x4* src = a.x + (((b * a.C + c) * a.gh + gy) * 16 + dy) * (2 * a.gw) + 2 * gx + half;
  u32x4* dst = a.y + (((b * a.gh + gy) * a.gw + gx) * a.C + c) * 32 + 2 * dy + half;
  const u32x4 v0 = src[0], v1 = src[16 * a.gw];
  dst[0] = v0;
  dst[16] = v1;
}

}  // namespace samfast

extern "C" int samfast_patch_rows(const void* x, void* y, int64_t B, int C, int H, int W, void* stream) {
  using namespace samfast;
  SF_REQUIRE(B >= 0 && C > 0 && C <= (1 << 16) && H > 0 && W > 0 && H % 16 == 0 && W % 16 == 0 && H <= (1 << 16) && W <= (1 << 16),
             "patch_rows: bad shape B=%lld C=%d %dx%d", (long long)B, C, H, W);
  if (B == 0) return SAMFAST_OK;
  // a launch has fewer than 2^32 threads
  const int64_t per_image = (int64_t)C * (H / 16) * ((W / 16 + 3) / 4);
  SF_REQUIRE(B <= SAMFAST_PATCH_ROWS_MAX / per_image, "patch_rows: too large");
  SF_REQUIRE(x && y && aligned16(x) && aligned16(y), "patch_rows: null or unaligned pointer");
  PatchArgs a = {reinterpret_cast<const u32x4*>(x), reinterpret_cast<u32x4*>(y), 0, C, H / 16, W / 16, (W / 16 + 3) / 4};
  a.waves = (unsigned int)(B * per_image);
  hipLaunchKernelGGL(patch_rows_kernel, dim3((a.waves + 3u) / 4u), dim3(256), 0, reinterpret_cast<hipStream_t>(stream), a);
  return check_launch("patch_rows_kernel");
}

extern "C" int samfast_preprocess(const void* x, int x_is_u8, const float* mean, const float* std, void* y, int64_t B, int h, int w, int S,
                                  int dtype, void* stream) {
  using namespace samfast;
  if (dtype != SAMFAST_BF16 && dtype != SAMFAST_F16) SF_FAIL(SAMFAST_E_UNSUPPORTED, "preprocess: element type %d is neither SAMFAST_BF16 nor SAMFAST_F16", dtype);
  SF_REQUIRE(B >= 0 && h > 0 && w > 0 && S > 0 && S % 8 == 0 && h <= S && w <= S && S <= (1 << 16), "preprocess: bad shape B=%lld %dx%d in %d", (long long)B, h, w, S);
  if (B == 0) return SAMFAST_OK;
  SF_REQUIRE(x && mean && std && y && aligned16(y) && (x_is_u8 || (reinterpret_cast<uintptr_t>(x) & 3u) == 0), "preprocess: null or unaligned pointer");
  PreprocessArgs a = {x, mean, std, reinterpret_cast<unsigned short*>(y), B * 3 * S * (S / 8), h, w, S};
  SF_REQUIRE((a.chunks + 255) / 256 < (1ll << 31), "preprocess: too large");
  const dim3 grid((unsigned int)((a.chunks + 255) / 256)), block(256);
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  if (dtype == SAMFAST_F16) {
    if (x_is_u8) hipLaunchKernelGGL((preprocess_kernel<ElemF16, unsigned char>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((preprocess_kernel<ElemF16, float>), grid, block, 0, s, a);
  } else {
    if (x_is_u8) hipLaunchKernelGGL((preprocess_kernel<ElemBf16, unsigned char>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((preprocess_kernel<ElemBf16, float>), grid, block, 0, s, a);
  }
  return check_launch("preprocess_kernel");
}
