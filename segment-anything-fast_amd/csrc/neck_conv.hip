// The neck's two convolutions (1 x 1 and 3 x 3, stride 1, zero padding, no bias) over channels-last half-type images.
//
// One image is 4096 tokens and 256 output channels: 64 x 64 outputs a workgroup are exactly one workgroup per CU, and what bounds the
// launch is the time to stream 128 rows of every k tile through a CU's load path (3 x 3: 36 k tiles of 16 KB) and the launch itself.
// Operands go global -> LDS directly, six stages deep; a token outside the image is read from a page of zeros, so that
// nothing is padded or unfolded in memory.  Sums stay in fp32 over all of K in one fixed order.
// us, the whole neck with its LayerNorms, the library's kernels with their clearing and casting launches / these, recorded: one image of
// width 768 101 / 37, width 1280 102 / 40, eight images 287 / 176, 295 / 194; sixteen 230 / 329, where larger tiles are ahead.
//
// A 3 x 3 weight lies as (out, in, 3, 3); the products want its input channels next to each other.  The 1 x 1 launch in front of it
// carries that reordering along in workgroups of its own (1.2 MB, hidden by the products): nothing is kept between calls.
#include "gemm_pingpong.hpp"

namespace samfast {

struct ConvArgs {
  const unsigned char* x;    // (B, H, W, Cin)
  const unsigned char* w;    // TAPS == 1: (Cout, Cin); 9: (Cout, 9, Cin)
  unsigned short* y;         // (B, H, W, Cout)
  const unsigned short* relay_src;  // (R, S, 3, 3), may be null
  unsigned short* relay_dst;        // (R, 9, S)
  int relay_rows, relay_cin;
  int M, H, W, Cin, Cout;
  int tiles_n, tiles;
};

__device__ __attribute__((aligned(16))) const unsigned int conv_zeros[4] = {0, 0, 0, 0};

constexpr int CV = 64;                 // tokens and channels of a tile, and channels of a k tile
constexpr int CVSTAGE = 2 * CV * 128;  // 64 rows of X and of W, 128 bytes each
constexpr int CVNST = 6;

template <class E, int TAPS>
__global__ __launch_bounds__(256) void neck_conv_kernel(ConvArgs a) {
  typedef typename E::Out Out;
  __shared__ __attribute__((aligned(16))) unsigned char lds[CVNST * CVSTAGE];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  if ((int)blockIdx.x >= (a.tiles + 7) / 8 * 8) {
    // reordering: one output channel a workgroup, its S * 9 values through LDS
    const int n = (int)blockIdx.x - (a.tiles + 7) / 8 * 8;
    unsigned short* s = reinterpret_cast<unsigned short*>(lds);
    const int count = a.relay_cin * 9;
    const unsigned short* src = a.relay_src + (int64_t)n * count;
    for (int i = tid; i < count; i += 256) s[i] = src[i];
    __syncthreads();
    for (int i = tid; i < count; i += 256) {
      const int tap = i / a.relay_cin, c = i - tap * a.relay_cin;
      a.relay_dst[(int64_t)n * count + i] = s[c * 9 + tap];
    }
    return;
  }
  const unsigned int pid = xcd_contiguous_id(blockIdx.x, (unsigned int)a.tiles);
  if ((int)pid >= a.tiles) return;  // uniform over the workgroup
  const int m0 = (int)(pid / a.tiles_n) * CV, n0 = (int)(pid % a.tiles_n) * CV;
  const int wm = wave >> 1, wn = wave & 1, lr = lane & 15, lq = lane >> 4;

  // tile loads: an instruction fills eight LDS rows of 128 bytes, wavefront w takes rows 8 w .. and 32 + 8 w .. of either operand.
  // Chunk c of row r lies at c ^ ((r >> 1) & 7).  LDS row 16 j + r of a half of W (32 channels) is channel 2 r + j.
  typedef __attribute__((address_space(1))) const void* gptr_t;
  typedef __attribute__((address_space(3))) void* lptr_t;
  const int kc = a.Cin / CV, nk = TAPS * kc;
  int ty[2], tx[2];
  const unsigned char* xrow[2];
  const unsigned char* wrow[2];
  bool live[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = 32 * i + 8 * wave + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
    const int m = m0 + r, t = m % (a.H * a.W);
    live[i] = m < a.M;
    ty[i] = t / a.W;
    tx[i] = t - ty[i] * a.W;
    xrow[i] = a.x + (int64_t)m * a.Cin * 2 + c * 16;
    wrow[i] = a.w + (int64_t)(n0 + 32 * i + 2 * (r & 15) + ((r >> 4) & 1)) * TAPS * a.Cin * 2 + c * 16;
  }
  int tap = 0, cb = 0;  // of the k tile that is requested next
  auto fill = [&](int stage) __attribute__((always_inline)) {
    const int dy = TAPS == 9 ? tap / 3 - 1 : 0, dx = TAPS == 9 ? tap % 3 - 1 : 0;
    const int64_t xo = ((int64_t)(dy * a.W + dx) * a.Cin + cb * CV) * 2, wo = ((int64_t)tap * a.Cin + cb * CV) * 2;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const bool in = live[i] && (TAPS == 1 || ((unsigned int)(ty[i] + dy) < (unsigned int)a.H && (unsigned int)(tx[i] + dx) < (unsigned int)a.W));
      const unsigned char* src = in ? xrow[i] + xo : reinterpret_cast<const unsigned char*>(conv_zeros);
      __builtin_amdgcn_global_load_lds((gptr_t)src, (lptr_t)(lds + stage + (32 * i + 8 * wave) * 128), 16, 0, 0);
      __builtin_amdgcn_global_load_lds((gptr_t)(wrow[i] + wo), (lptr_t)(lds + stage + (CV + 32 * i + 8 * wave) * 128), 16, 0, 0);
    }
    if (++cb == kc) {
      cb = 0;
      ++tap;
    }
  };
  typename E::acc_t acc[2][2] = {};
#pragma unroll
  for (int p = 0; p < CVNST - 1; ++p)
    if (p < nk) fill(p * CVSTAGE);
  const int frag = (lq ^ ((lr >> 1) & 7)) * 16;
  int rd = 0, wr = (CVNST - 1) * CVSTAGE;
  for (int t = 0; t < nk; ++t) {
    // own loads of k tile t have landed (those of the CVNST - 2 behind it may be under way), then everybody's; the
    // stage of k tile t - 1 has been read by all
    if (t + CVNST - 2 < nk) pp_wait<4 * (CVNST - 2)>();
    else pp_wait<0>();
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    if (t + CVNST - 1 < nk) fill(wr);
    i32x4 fx[2][2], fw[2][2];
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        fx[k][i] = *reinterpret_cast<const i32x4*>(lds + rd + (wm * 32 + 16 * i + lr) * 128 + (frag ^ (64 * k)));
        fw[k][i] = *reinterpret_cast<const i32x4*>(lds + rd + (CV + wn * 32 + 16 * i + lr) * 128 + (frag ^ (64 * k)));
      }
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = E::mma(fx[k][i], fw[k][j], acc[i][j]);
    rd = rd == (CVNST - 1) * CVSTAGE ? 0 : rd + CVSTAGE;
    wr = wr == (CVNST - 1) * CVSTAGE ? 0 : wr + CVSTAGE;
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = m0 + wm * 32 + 16 * i + 4 * lq + r;
      if (m < a.M)
        *reinterpret_cast<unsigned int*>(a.y + (int64_t)m * a.Cout + n0 + wn * 32 + 2 * lr) = Out::pack2(acc[i][0][r], acc[i][1][r]);
    }
}

template <class E>
static int neck_conv_launch(const ConvArgs& a, int taps, hipStream_t stream) {
  const dim3 grid((unsigned int)((a.tiles + 7) / 8 * 8 + (a.relay_src ? a.relay_rows : 0)));
  if (taps == 1) hipLaunchKernelGGL((neck_conv_kernel<E, 1>), grid, dim3(256), 0, stream, a);
  else hipLaunchKernelGGL((neck_conv_kernel<E, 9>), grid, dim3(256), 0, stream, a);
  return check_launch("neck_conv_kernel");
}

}  // namespace samfast

extern "C" int samfast_neck_conv(const void* x, const void* w, void* y, int64_t B, int H, int W, int Cin, int Cout, int taps,
                                 int dtype, const void* relay_src, void* relay_dst, int relay_rows, int relay_cin, void* stream) {
  using namespace samfast;
  if (dtype != SAMFAST_BF16 && dtype != SAMFAST_F16) SF_FAIL(SAMFAST_E_UNSUPPORTED, "neck_conv: element type %d is neither SAMFAST_BF16 nor SAMFAST_F16", dtype);
  SF_REQUIRE(taps == 1 || taps == 9, "neck_conv: %d taps, 1 or 9 are built", taps);
  SF_REQUIRE(B >= 0 && H > 0 && W > 0 && Cin > 0 && Cout > 0 && Cin % CV == 0 && Cout % CV == 0,
             "neck_conv: bad shape B=%lld H=%d W=%d Cin=%d Cout=%d (channels must be multiples of %d)", (long long)B, H, W, Cin, Cout, CV);
  SF_REQUIRE((int64_t)H * W < (1ll << 30) && B * H * W < (1ll << 30) && Cin <= (1 << 16) && Cout <= (1 << 16), "neck_conv: too large");
  if (B == 0) return SAMFAST_OK;
  SF_REQUIRE(x && w && y && aligned16(x) && aligned16(w) && aligned16(y), "neck_conv: null or unaligned pointer");
  SF_REQUIRE((relay_src == nullptr) == (relay_dst == nullptr), "neck_conv: both ends of the reordered weight or none");
  SF_REQUIRE(!relay_src || (relay_rows > 0 && relay_rows <= (1 << 16) && relay_cin > 0 && relay_cin * 18 <= CVNST * CVSTAGE), "neck_conv: bad reordered weight");
  ConvArgs a = {};
  a.x = reinterpret_cast<const unsigned char*>(x);
  a.w = reinterpret_cast<const unsigned char*>(w);
  a.y = reinterpret_cast<unsigned short*>(y);
  a.relay_src = reinterpret_cast<const unsigned short*>(relay_src);
  a.relay_dst = reinterpret_cast<unsigned short*>(relay_dst);
  a.relay_rows = relay_rows;
  a.relay_cin = relay_cin;
  a.M = (int)(B * H * W);
  a.H = H;
  a.W = W;
  a.Cin = Cin;
  a.Cout = Cout;
  a.tiles_n = Cout / CV;
  const int64_t tiles = (int64_t)((a.M + CV - 1) / CV) * a.tiles_n;
  SF_REQUIRE(tiles < (1ll << 30), "neck_conv: too many tiles");
  a.tiles = (int)tiles;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  return dtype == SAMFAST_F16 ? neck_conv_launch<PPF16>(a, taps, s) : neck_conv_launch<PPBf16>(a, taps, s);
}
