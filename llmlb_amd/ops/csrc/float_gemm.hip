// Products of 32-bit matrices on the matrix cores' bf16 instructions:
//
//   out[N, M] = act(x[N, K] W[M, K]^T)     float, summed in float
//
// A float is the sum of three bf16 numbers without a remainder, each the nearest
// to what the ones before leave (8 bits and a sign each), so a product of two is
// nine products of those, of which the three smallest are left out: 2^-24 of the
// product at most, to either side.  Six times the work at sixteen times the rate
// of the float instructions, and the sum is rounded once in 32 of the depth where
// theirs is in every four.  Errors against 64 bits, the library's -> here in tiles
// of eight waves, of four, which sum twice the depth each: normal numbers 32 deep
// 1.0e-7 -> 3.8e-8, 256 2.9e-7 -> 6.4e-8, 1.0e-7, 1024 5.8e-7 -> 1.6e-7, 2.3e-7, 3328
// 1.0e-6 -> 3.1e-7, 4.4e-7 (a piece's six products summed by themselves and added
// once would be 8.5e-8 and 1.3e-7 there, in 4 to 20% more time); numbers from 1 to
// 1.01 256 deep 2.1e-7 -> 5.2e-8, on average 9e-10 to one side.  Only rows with a
// single number that is not zero, which the library rounds once, are further off:
// 2.5e-8 -> 3.4e-8.  (Cutting bits off takes as many instructions and a few percent
// less time, but parts of one sign leave out up to 2^-21, always to the same side:
// 6.9e-8 of single numbers.)
//
// Bound by vector instructions, which take numbers apart and look for the largest
// (6 a number of a tile's edge), beside matrix instructions (a tile of 64 x 64, of
// 128 of the depth: 1780 and 1540 cycles a SIMD), and by how tiles fill the
// last round.  So waves have one stage in LDS, and two to four of them a SIMD cover
// each other (two stages at one wave a SIMD: 600 rows, 1024 x 1024 16 us, 14.2
// this way); a wave takes numbers apart between matrix instructions, each of which
// leaves room for two (3328 x 1024 35 -> 32.3, 4128 x 1024 40.3 -> 37.7); larger
// tiles take less apart (600 rows of 4096 x 2048 76 us with 64 x 64, 66 with 80 x
// 64).  us, the library -> here, weights from HBM:
//   600 rows: 1024 x 1024 16.7 -> 13.9, 3328 x 1024 37 -> 32, 4128 x 1024 53 ->
//       38, 1024 x 3328 41 -> 34; 64 rows: 8.5 -> 5.5, 12.5 -> 8.9, 13.3 ->
//       13.2, 11.7 -> 11.6; 16 rows of 4096 x 2048 12.3 -> 9.4; 1600 rows of
//       4096 x 2048 237 -> 156 (172 TFLOP/s)
// The largest numbers, which tell what may be lost (see the kernel), cost 2 to 5%.
#include "hybrid/float_tile.h"

template <int NT, int MT, int KW>
__global__ __launch_bounds__(KW * 64, KW == 4 ? 2 : 1) void float_gemm_kernel(
    float* __restrict__ out, int ld_out, const float* __restrict__ x,
    const float* __restrict__ w, int N, int M, int K, int ldx, int kind,
    bool narrow) {
  using Tile = FloatTile<NT, MT, KW>;
  extern __shared__ __align__(1024) char lds[];
  // One of eight XCDs has every eighth tile of W, and goes through them by
  // eight tiles of x at a time: what its workgroups read at once fits its L2.
  // Where W is narrow it has every eighth tile of x.
  const int across = (N + 16 * NT - 1) / (16 * NT);
  const int down = (M + 16 * MT - 1) / (16 * MT);
  const int xcd = blockIdx.x % 8, in = blockIdx.x / 8;
  int tile_x, tile_w, turn;
  if (narrow) {
    tile_x = in / down * 8 + xcd, tile_w = turn = in % down;
  } else {
    const int each = (down + 7) / 8, first = in / (8 * each) * 8;
    const int rest = in - first * each;
    const int wide = across - first < 8 ? across - first : 8;
    turn = rest / wide;
    tile_x = first + rest % wide, tile_w = turn * 8 + xcd;
  }
  const int n0 = tile_x * 16 * NT, m0 = tile_w * 16 * MT;
  if (n0 >= N || m0 >= M) return;
  x += (size_t)n0 * ldx, w += (size_t)m0 * K;
  const int last_x = N - 1 - n0, last_w = M - 1 - m0;
  Tile::run(
      lds, K, turn, x,
      [&](int r) {
        return (unsigned)(r < last_x ? r : last_x) * (unsigned)ldx;
      },
      w, [&](int r) { return (unsigned)(r < last_w ? r : last_w) * (unsigned)K; });
  Tile::finish(
      lds, K, kind, N - n0, M - m0,
      [&](int r) { return x + (size_t)r * ldx; },
      [&](int c) { return w + (size_t)c * K; },
      [&](int r) { return out + (size_t)(n0 + r) * ld_out + m0; });
}

// Whether tiles of x and not those of W are dealt to the XCDs
static bool narrow_w(long long across, long long down) {
  return across > down && down < 64;
}

struct FloatGemm {
  float* out;
  int ld_out;
  const float *x, *w;
  int N, M, K, ldx, kind;
  hipStream_t stream;
};

template <int NT, int MT, int KW>
static int float_gemm_launch(const FloatGemm& p) {
  auto* kernel = &float_gemm_kernel<NT, MT, KW>;
  constexpr int lds = FloatTile<NT, MT, KW>::LDS;
  static_assert(lds <= 160 * 1024, "LDS of a compute unit");
  // a lane's copies are at 32-bit offsets in bytes from the tile's first row
  if (64ll * NT * p.ldx > 1ll << 32 || 64ll * MT * p.K > 1ll << 32) return -2;
  static const hipError_t sized = hipFuncSetAttribute(
      reinterpret_cast<const void*>(kernel),
      hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (sized != hipSuccess) return -1;
  const long long down = (p.M + 16 * MT - 1) / (16 * MT);
  const long long across = (p.N + 16 * NT - 1) / (16 * NT);
  const bool narrow = narrow_w(across, down);
  const long long grid =
      narrow ? (across + 7) / 8 * 8 * down : (down + 7) / 8 * 8 * across;
  if (grid > 1 << 30) return -2;
  hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(KW * 64), lds,
                     p.stream, p.out, p.ld_out, p.x, p.w, p.N, p.M, p.K,
                     p.ldx, p.kind, narrow);
  HY_CHECK();
  return 0;
}

// Tiles that there are: how many a compute unit has at once, us of a tile 1024
// deep where each unit has one and where each has all of them, of the beginning
// and end, and of those of every round more.  Fitted to 348 products of 1 to 2000
// rows, 16 to 4128 outputs and 64 to 4700 deep, and 150 of up to 16 rows of 2048 to
// 8192 outputs.  Of 215 others the tile taken is 0.2% slower than the fastest on
// average, 4 are more than 5% slower, 7% at most (without the rounds' ends, and of
// 1024 deep and deeper alone, 2.6% up to 400 deep, 22% at most: 100 rows of 1024 x
// 256 3.7 -> 4.2 us).
struct FloatTileTime {
  int rows, cols, at_once;
  float one, all, ends, more;
};
static const FloatTileTime FLOAT_TILES[] = {
    {16, 16, 4, 2.6f, 7.8f, 3.48f, 0.6f},
    {32, 16, 3, 3.f, 8.61f, 3.5f, 1.9f},
    {32, 32, 2, 4.3f, 8.4f, 3.6f, 0.2f},
    {48, 32, 2, 5.5f, 11.52f, 3.5f, 3.f},
    {48, 64, 1, 8.5f, 10.6f, 4.8f, 4.6f},
    {48, 48, 3, 7.72f, 21.4f, 4.97f, 0.1f},
    {48, 64, 2, 9.6f, 17.9f, 4.7f, 3.7f},
    {64, 64, 2, 12.f, 21.2f, 5.36f, 2.1f},
    {80, 64, 2, 14.f, 26.3f, 5.4f, 0.1f},
    {64, 96, 2, 14.92f, 30.7f, 6.8f, 0.1f},
    {80, 80, 2, 15.3f, 29.3f, 7.9f, 0.4f}};

// The tile that is estimated to take least.  A last round takes as long as
// the units with most of its tiles.
static int float_tile(int N, int M, int K) {
  int best = 0;
  float least = 0.f;
  for (int t = 0; t < (int)(sizeof(FLOAT_TILES) / sizeof(FloatTileTime));
       ++t) {
    const FloatTileTime& at = FLOAT_TILES[t];
    const long long across = (N + at.rows - 1) / at.rows;
    const long long down = (M + at.cols - 1) / at.cols;
    // those of the XCD that has most, of 32 units
    const long long n = 8 * (narrow_w(across, down)
                                 ? (across + 7) / 8 * down
                                 : (down + 7) / 8 * across);
    const int round = 256 * at.at_once, rest = (int)(n % round);
    float tiles = (float)(n / round) * at.all;
    if (rest)
      tiles += at.one + (rest <= 256 ? 0.f
                                     : (at.all - at.one) *
                                           (float)((rest - 1) / 256) /
                                           (float)(at.at_once - 1));
    const float us = tiles * ((float)K / 1024.f) + at.ends +
                     at.more * (float)((n - 1) / round);
    if (t == 0 || us < least) least = us, best = t;
  }
  return best;
}

// Whether the library's product is the faster.  A tile's beginning and end are
// most of a shallow product, of which there are many tiles; deep products of fewer
// outputs than fill the chip it takes in shares of the depth.  The library's time
// over this one's, means of 7 to 14 sizes each by depth and outputs:
//   32: to 2^17.5 0.99, 2^18.5 0.93, 2^19 0.88, 2^20 0.65; 64: 1.04, 0.96, 0.86,
//   0.75; 128: 1.19, 1.21, 1.30, 0.94, then 0.77; 256: 2^19 1.01, then 0.88, 0.91
//   and to 2^22 0.96; 384: 1.02, 0.92, to 2^21 1.01; 512: 1.22, 0.94, 1.17; 640:
//   1.01, 0.96, 1.18; more than 512 rows 128 deep 0.72
//   4096: to 2^17 0.93, to 2^18 1.07; 8192 0.91, 1.08; 14336 0.88, 1.13; 3328 to
//   2^16 0.97; 18304 1.6
// The launch and pass of an activation's own kernel are more than that from 256 on.
static bool library_gains(int N, int M, int K, int kind) {
  const double outputs = (double)N * M;
  if (K < 256 && N > 512) return true;
  if (K >= 256 && kind != PLAIN) return false;
  if (K >= 4096 && K <= 16384 && outputs < 1 << 17) return true;
  return outputs > (K < 128 ? 1 << 18 : 1 << 19) &&
         outputs * K * K <= 0x1p38;
}

// Rows of x start ldx numbers apart, those of out ld_out.  tile: -1, or the
// one to take.  0: done, -2: not for this kernel.
extern "C" int ll_float_gemm(void* out, int ld_out, const void* x,
                             const void* w, int N, int M, int K, int ldx,
                             int kind, int tile, void* stream) {
  if (N <= 0 || M <= 0 || K <= 0 || M % 4 || K % 32 || ldx < K || ldx % 4 ||
      ld_out < M || ld_out % 4 || (uintptr_t)x % 16 || (uintptr_t)w % 16 ||
      (uintptr_t)out % 16 ||
      (kind != PLAIN && kind != RELU2 && kind != GELU))
    return -2;
  if (tile < 0 && library_gains(N, M, K, kind)) return -2;
  const FloatGemm p{(float*)out, ld_out, (const float*)x, (const float*)w,
                    N, M, K, ldx, kind, (hipStream_t)stream};
  switch (tile < 0 ? float_tile(N, M, K) : tile) {
    case 0: return float_gemm_launch<1, 1, 8>(p);
    case 1: return float_gemm_launch<2, 1, 8>(p);
    case 2: return float_gemm_launch<2, 2, 8>(p);
    case 3: return float_gemm_launch<3, 2, 8>(p);
    case 4: return float_gemm_launch<3, 4, 8>(p);
    case 5: return float_gemm_launch<3, 3, 4>(p);
    case 6: return float_gemm_launch<3, 4, 4>(p);
    case 7: return float_gemm_launch<4, 4, 4>(p);
    case 8: return float_gemm_launch<5, 4, 4>(p);
    case 9: return float_gemm_launch<4, 6, 4>(p);
    case 10: return float_gemm_launch<5, 5, 4>(p);
  }
  return -2;
}
