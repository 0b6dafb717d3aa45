// Products of many rows with a weight matrix, for prompts:
//
//   out[N, M] = act(x[N, K] W[M, K]^T)     bf16, summed in float
//
// Bound by the power of the matrix cores: at 1430 TFLOP/s they are busy 87% of
// the cycles, and the clock is down to 1.2 to 1.7 GHz (with how long the chip has
// been at it, swiglu of 16384 rows against 28672 x 4096 takes 2.55 to 2.65 ms,
// 1510 to 1450 TFLOP/s).  So what counts beside the cycles is the energy of a
// product: 16 x 16 x 32 (registers alone: 2060 TFLOP/s) and not 32 x 32 x 16
// (1790), LDS read without bank conflicts, each number once.  16384 rows of 4096 x
// 14336 take 1290 us without an activation; with copies all at once and two
// stages of 64 KB it was 1582, with the ring below and 32 x 32 products 1370.  The
// library's product takes 1200 to 1250 us, but a pass over its results more
// (swiglu of 16384 x 14336: 263 us).
//
// A tile's end is in no product's shadow: both waves of a SIMD come to it at the
// same time.  Sums rounded by hand -> by the hardware's conversion, and plain ones
// once and not twice, us, 16384 rows: gelu of 7168 x 2048 381 -> 369, plain 6416 x
// 2048 322 -> 318, clamped 11904 x 4096 1110 -> 1101, swiglu 28672 x 4096 2590 ->
// 2585.  (Results in registers whose stores follow through the next tile's steps
// gained nothing here.)
#include "hybrid/tile_product.h"

struct TileGemm {
  bf16_t* out;
  int ld_out;
  const bf16_t *x, *w;
  int N, M, K, ldx;
  RowAct act;
  hipStream_t stream;
};

// The rows of a matrix in order
template <int BM, int BN, int KIND>
struct Rows {
  static constexpr int OUT = KIND == SWIGLU || KIND == CLAMPED ? BN / 2 : BN;
  const bf16_t *x_, *w_;
  int N, ldx, down, across;
  struct At {
    int n0, m0;
  };
  __device__ __forceinline__ long long tiles() const {
    return (long long)down * across;
  }
  // tiles go through the outputs by four blocks of rows at a time
  __device__ __forceinline__ At at(int t) const {
    const int run = t / (4 * across), in = t - run * (4 * across);
    const int rows = down - run * 4 < 4 ? down - run * 4 : 4;
    return At{(run * 4 + in % rows) * BM, in / rows * OUT};
  }
  __device__ __forceinline__ void fetch(int) const {}
  __device__ __forceinline__ void fetched() const {}
  __device__ __forceinline__ const bf16_t* x(const At& a) const {
    return x_ + (size_t)a.n0 * ldx;
  }
  __device__ __forceinline__ const bf16_t* w(const At&) const { return w_; }
  __device__ __forceinline__ unsigned x_offset(const At& a, int r) const {
    const int last = N - 1 - a.n0;
    return (unsigned)(r < last ? r : last) * (unsigned)ldx;
  }
  __device__ __forceinline__ long long row(const At& a, int r) const {
    return a.n0 + r < N ? a.n0 + r : -1;
  }
  __device__ __forceinline__ bool whole(const At& a) const {
    return a.n0 + BM <= N;
  }
};

template <int BM, int BN, int WM, int WN, int D, int KIND>
__global__ __launch_bounds__(WM * WN * 64, WM * WN / 4)
void tile_gemm_kernel(Rows<BM, BN, KIND> rows, bf16_t* __restrict__ out,
                      int ld_out, int M, int K, RowAct act) {
  tile_product<BM, BN, WM, WN, D, KIND, true, false>(rows, out, ld_out, M, K,
                                                     act);
}

template <int BM, int BN, int WM, int WN, int D, int KIND>
static int tile_gemm_launch(const TileGemm& p) {
  auto* kernel = &tile_gemm_kernel<BM, BN, WM, WN, D, KIND>;
  constexpr int lds = ((D + 1) * BM + D * BN) * DEPTH * 2;
  static_assert(lds <= 160 * 1024, "LDS of a compute unit");
  static const hipError_t sized = hipFuncSetAttribute(
      reinterpret_cast<const void*>(kernel),
      hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (sized != hipSuccess) return -1;
  using R = Rows<BM, BN, KIND>;
  const int down = (p.N + BM - 1) / BM, across = (p.M + R::OUT - 1) / R::OUT;
  const long long per = ((long long)down * across + 7) / 8;
  if (per > 1 << 26) return -2;
  const int slots = per < 32 ? (int)per : 32;
  const R rows{p.x, p.w, p.N, p.ldx, down, across};
  hipLaunchKernelGGL(kernel, dim3(8 * slots), dim3(WM * WN * 64), lds,
                     p.stream, rows, p.out, p.ld_out, p.M, p.K, p.act);
  HY_CHECK();
  return 0;
}

// Tiles that there are: us of a step with all compute units at work and with
// half of them or fewer (then L2 and the clock give more), and of a tile's
// beginning and end, fitted to products 1024 and 8192 deep.
struct Tile {
  int rows, cols;
  float all, half, ends;
};
static const Tile TILES[] = {
    {256, 256, 1.38f, 0.98f, 11.f}, {192, 256, 1.14f, 0.89f, 7.f},
    {128, 256, 0.85f, 0.70f, 5.f},  {256, 128, 0.80f, 0.53f, 6.f},
    {192, 128, 0.69f, 0.48f, 5.5f}, {160, 128, 0.61f, 0.41f, 5.f},
    {128, 128, 0.55f, 0.37f, 4.5f}, {96, 128, 0.46f, 0.31f, 4.5f},
    {64, 128, 0.39f, 0.27f, 4.f}};

template <int KIND>
static int tile_gemm_go(const TileGemm& p, int tile) {
  switch (tile) {
    case 0: return tile_gemm_launch<256, 256, 2, 4, 2, KIND>(p);
    case 1: return tile_gemm_launch<192, 256, 2, 4, 2, KIND>(p);
    case 2: return tile_gemm_launch<128, 256, 2, 4, 3, KIND>(p);
    case 3: return tile_gemm_launch<256, 128, 4, 2, 2, KIND>(p);
    case 4: return tile_gemm_launch<192, 128, 2, 2, 3, KIND>(p);
    case 5: return tile_gemm_launch<160, 128, 2, 2, 3, KIND>(p);
    case 6: return tile_gemm_launch<128, 128, 2, 2, 4, KIND>(p);
    case 7: return tile_gemm_launch<96, 128, 2, 2, 5, KIND>(p);
    case 8: return tile_gemm_launch<64, 128, 2, 2, 5, KIND>(p);
  }
  return -2;
}

// The tile that is estimated to take least: a compute unit's time is that of
// its rounds, the last of which may be of few tiles.  (1355 rows of 6912 x
// 2048 are 162 tiles of 256 x 256, 42 us, 216 of 192 x 256, 39, or 297 of 128 x
// 256, 51.)
static int best_tile(int N, int rows, int K) {
  int best = 0;
  float least = 0.f;
  for (int t = 0; t < (int)(sizeof(TILES) / sizeof(Tile)); ++t) {
    const Tile& at = TILES[t];
    const long long n = ((long long)N + at.rows - 1) / at.rows *
                        ((rows + at.cols - 1) / at.cols);
    const float steps = (float)K / DEPTH;
    float us = (float)(n / 256) * (at.all * steps + at.ends);
    if (const int rest = (int)(n % 256)) {
      const float more = rest > 128 ? (rest - 128) / 128.f : 0.f;
      us += (at.half + (at.all - at.half) * more) * steps + at.ends;
    }
    if (t == 0 || us < least) least = us, best = t;
  }
  return best;
}

// Whether this is faster than the library's product and, with an activation,
// a kernel of its own.  us, the library -> here, rows: outputs x depth:
//  * always with an activation, but for few tiles of some depth.  swiglu 333:
//    2816 x 1024 26 -> 12; 1355: 5632 x 2048 72 -> 58, 14336 x 4096 282 -> 264;
//    16384: 2816 x 1024 228 -> 156, 14336 x 4096 2792 -> 2631.  gelu 16384: 7168 x
//    2048 429 -> 367, 19456 x 4096 1957 -> 1820.  clamped 16384: 4352 x 2048 522 ->
//    441, 11904 x 4096 2338 -> 2255.  squared relu 333: 6912 x 2048 25 -> 16; 1355:
//    43 -> 37, 18432 x 4096 179 -> 170.  From 129 to 320 rows by 1.03 to 1.9, but
//    for a last round of few tiles (320: 28672 x 4096 swiglu 86 -> 89)
//  * not for few tiles of some depth, which the library takes in shares: 333:
//    2048 x 2048 10.7 -> 12.9, 2048 x 7168 30 -> 43, 1024 x 3328 13 -> 18.  Of up
//    to 1024 deep fewer than 64 lose less than half a microsecond (129: 1024 x 1024
//    8.1 -> 8.4) or gain (129: 256 x 512 2.1 times), and the host, which prompts of
//    a few hundred rows wait for, is done 12 us earlier than with the library
//  * not for the widest that are not shallow, which memory bounds: 320: 32768 x
//    2048 50 -> 55, 57344 x 2048 90 -> 98; 2048: 349 -> 365
//  * outputs that are no whole tiles of 256: 333: 8224 x 2048 25 -> 21; 1355:
//    3216 x 1024 17.5 -> 13.2, 8224 x 2048 56 -> 52; 8200: 1808 x 1024 53 -> 34,
//    16448 x 4096 922 -> 834; 16384: 3600 x 2048 236 -> 200, 6416 x 2048 378 ->
//    338, but 16512 x 4096 1557 -> 1604.  From 129 to 1024 rows the library's
//    times go up and down by a fifth, and so do the gains: 129, 200, 256, 320,
//    400, 512, 700, 1024 rows of 8224 x 2048 0.94 (not taken), 1.24, 1.22, 1.04,
//    1.30, 0.95, 1.11, 1.04; of 10272 x 4096 0.95, 0.90, 1.16, 0.92, 1.18, 0.93,
//    1.03, 1.01
//  * shallow ones, or of medium depth and not too many rows: 1355: 1024 x 1024
//    10.8 -> 9.0, 2048 x 2048 18.6 -> 18.1, 3072 x 2048 24.6 -> 22.2; 12288:
//    1024 x 1024 28.4 -> 26.0, but 16384: 2048 x 2048 101 -> 104
//  * deep ones have the library's best rate (16384: 4096 x 14336 1250 -> 1296,
//    1355: 2048 x 7168 55 -> 59), but where its tiles of 256 x 256 leave a last
//    round of few (8200: 2048 x 7168 322 -> 216, 4096 x 4096 302 -> 216; 4100:
//    4096 x 18432 906 -> 614), and the deepest of medium rows (1355: 4096 x
//    18432 308 -> 227)
extern "C" int ll_tile_gemm_gains(int N, int rows, int K, int kind) {
  if (N <= 0 || rows <= 0 || K <= 0) return 0;
  const long long few = ((long long)N + 63) / 64 * ((rows + 127) / 128);
  if (K > 1024 && few < (kind == PLAIN ? 200 : 150)) return 0;
  if (kind != PLAIN) return 1;
  if (K <= 1024) return 1;
  if (rows % 256) return K < 3072 || N < 12288;
  if (K < 3072) return N < 4096 && rows < 32768;
  const long long large = ((long long)N + 255) / 256 * (rows / 256);
  const int last = (int)(large % 256);
  return (large > 256 && last > 0 && last <= 64) ||
         (K >= 16384 && N >= 256 && N <= 2048);
}

// Rows of x start ldx numbers apart, those of out ld_out.  tile: -1, or the one
// to take.  0: done, -2: not for this kernel.
extern "C" int ll_tile_gemm(void* out, int ld_out, const void* x,
                            const void* w, int N, int M, int K, int ldx,
                            int kind, int up, float a, float b, int tile,
                            void* stream) {
  if (N <= 0 || M <= 0 || K <= 0 || M % 8 || K % DEPTH || ldx < K ||
      ldx % 8 || ld_out < M || ld_out % 8 || up < 0 || (uintptr_t)x % 16 ||
      (uintptr_t)w % 16 || (uintptr_t)out % 16)
    return -2;
  // copies are at a lane's 32-bit offset
  if (((size_t)up + M) * K >= 1ull << 31 || (size_t)ldx >= 1u << 22)
    return -2;
  const TileGemm p{(bf16_t*)out, ld_out,           (const bf16_t*)x,
                   (const bf16_t*)w, N, M, K, ldx, RowAct{kind, up, a, b},
                   (hipStream_t)stream};
  const bool gated = kind == SWIGLU || kind == CLAMPED;
  if (tile < 0) tile = best_tile(N, gated ? 2 * M : M, K);
  switch (kind) {
    case PLAIN: return tile_gemm_go<PLAIN>(p, tile);
    case RELU2: return tile_gemm_go<RELU2>(p, tile);
    case GELU: return tile_gemm_go<GELU>(p, tile);
    case SWIGLU: return tile_gemm_go<SWIGLU>(p, tile);
    case CLAMPED: return tile_gemm_go<CLAMPED>(p, tile);
  }
  return -2;
}
