// The neck's two convolutions (1 x 1 and 3 x 3, stride 1, zero padding, no bias) over channels-last half-type images.
//
// One image is 4096 tokens and 256 output channels: 64 x 64 outputs a workgroup are exactly one workgroup per CU.  What bounds the
// launch is the time from one barrier to the next - fragments from LDS (64 KB for two k tiles, 512 cycles), then sixteen products of a wavefront -
// and the launch itself, so two k tiles of 64 stand between two barriers, and five stages leave room for a second workgroup on a CU: from two images
// on another tile's, and in the launch that reorders weights (below) that work, which came behind the products on every CU.
// Operands go global -> LDS directly; a tap's 64 tokens are a buffer of their own, behind whose end a token outside the image is read as zeros, so that
// nothing is padded or unfolded in memory.  Sums stay in fp32 over all of K in one fixed order.
// us, the two launches recorded, six stages and a barrier per k tile / so: one image of width 768 24.5 / 20.9, 1280 26.9 / 22.9, two of 1024 46.3 / 29.7, four of 768 80.5 / 48.1, eight of
// 1280 172 / 99.6 (eight stages, 128 KB: 20.9, 22.7, 37.5, 64.5, 134; four: 22.5, 24.4, 28.5, 46.6, 97.7; a 64-bit address a lane and a page of zeros: the same).
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

constexpr int CV = 64;                 // tokens and channels of a tile, and channels of a k tile
constexpr int CVSTAGE = 2 * CV * 128;  // 64 rows of X and of W, 128 bytes each
constexpr int CVNST = 5;               // stages, of which two are read between two barriers; two workgroups' fit a CU

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
    const bool staged = count * 2 <= (int)sizeof(lds);  // (up to 4551 input channels)
    if (staged) {
      for (int i = tid; i < count; i += 256) s[i] = src[i];
      __syncthreads();
    }
    for (int i = tid; i < count; i += 256) {
      const int tap = i / a.relay_cin, c = i - tap * a.relay_cin;
      a.relay_dst[(int64_t)n * count + i] = staged ? s[c * 9 + tap] : src[c * 9 + tap];
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
  unsigned int xoff[2], woff[2];  // bytes, from the tile's first token of a tap / first channel
  bool live[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = 32 * i + 8 * wave + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
    const int m = m0 + r, t = m % (a.H * a.W);
    live[i] = m < a.M;
    ty[i] = t / a.W;
    tx[i] = t - ty[i] * a.W;
    xoff[i] = (unsigned int)(r * a.Cin * 2 + c * 16);
    woff[i] = (unsigned int)((32 * i + 2 * (r & 15) + ((r >> 4) & 1)) * TAPS * a.Cin * 2 + c * 16);
  }
  int tap = 0, cb = 0;  // of the k tile that is requested next
  const unsigned char* wk = a.w + (int64_t)n0 * TAPS * a.Cin * 2;
  __amdgpu_buffer_rsrc_t tokens;
  unsigned int xat[2];
  // The tap's 64 tokens as a buffer of their own: a lane whose token is outside the image reads behind its end, and gets zeros.
  auto aim = [&]() __attribute__((always_inline)) {
    const int dy = TAPS == 9 ? tap / 3 - 1 : 0, dx = TAPS == 9 ? tap % 3 - 1 : 0;
    tokens = __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned char*>(a.x) + ((int64_t)m0 + dy * a.W + dx) * a.Cin * 2, 0, CV * a.Cin * 2, 0x00027000);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const bool in = live[i] && (TAPS == 1 || ((unsigned int)(ty[i] + dy) < (unsigned int)a.H && (unsigned int)(tx[i] + dx) < (unsigned int)a.W));
      xat[i] = in ? xoff[i] : 0x80000000u;
    }
  };
  aim();
  auto fill = [&](int stage) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(tokens, (lptr_t)(lds + stage + (32 * i + 8 * wave) * 128), 16, (int)xat[i], cb * (2 * CV), 0, 0);
      const unsigned char* base = wk;
      unsigned int o = woff[i];
      asm volatile("" : "+s"(base));  // uniform base, 32-bit lane offset
      asm volatile("" : "+v"(o));
      __builtin_amdgcn_global_load_lds((gptr_t)(base + o), (lptr_t)(lds + stage + (CV + 32 * i + 8 * wave) * 128), 16, 0, 0);
    }
    wk += 2 * CV;  // (a tap's channels lie behind those of the tap before)
    if (++cb == kc) {
      cb = 0;
      ++tap;
      aim();
    }
  };
  typename E::acc_t acc[2][2] = {};
#pragma unroll
  for (int p = 0; p < CVNST - 2; ++p)
    if (p < nk) fill(p * CVSTAGE);
  const int frag = (lq ^ ((lr >> 1) & 7)) * 16;
  auto up = [](int stage) { return stage == (CVNST - 1) * CVSTAGE ? 0 : stage + CVSTAGE; };
  int rd = 0, wr = (CVNST - 2) * CVSTAGE;
  i32x4 fx[2][2][2], fw[2][2][2];
  auto read = [&](int d, int stage) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        fx[d][k][i] = *reinterpret_cast<const i32x4*>(lds + stage + (wm * 32 + 16 * i + lr) * 128 + (frag ^ (64 * k)));
        fw[d][k][i] = *reinterpret_cast<const i32x4*>(lds + stage + (CV + wn * 32 + 16 * i + lr) * 128 + (frag ^ (64 * k)));
      }
  };
  auto multiply = [&](int d) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = E::mma(fx[d][k][i], fw[d][k][j], acc[i][j]);
  };
  for (int t = 0; t < nk; t += 2) {
    // own loads of k tiles t and t + 1 have landed (those of the CVNST - 4 behind them may be under way), then everybody's; the
    // stages of the two before have been read by all
    if (t + CVNST - 2 <= nk) pp_wait<4 * (CVNST - 4)>();
    else pp_wait<0>();
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    const bool two = t + 1 < nk;  // uniform
    read(0, rd);
    rd = up(rd);
    if (two) read(1, rd);
    rd = up(rd);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int d = 0; d < 2; ++d)
      if (t + CVNST - 2 + d < nk) {
        fill(wr);
        wr = up(wr);
      }
    __builtin_amdgcn_sched_barrier(0);
    multiply(0);
    if (two) multiply(1);
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
  SF_REQUIRE(!relay_src || (relay_rows > 0 && relay_rows <= (1 << 16) && relay_cin > 0 && relay_cin * 18 <= 96 * 1024), "neck_conv: bad reordered weight");
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
