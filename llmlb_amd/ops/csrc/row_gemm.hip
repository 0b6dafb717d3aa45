// Products of few rows with a weight matrix, for decoding:
//
//   out[N, M] = x[N, K] W[M, K]^T     bf16, summed in float, N <= 128
//
// W is read once and nothing else is large, so the bound is memory for big
// matrices and latency for small ones; hybrid/row_tile.h says how a tile is
// computed.  Its result needs no second kernel.
//
// Sizes of a tile are ll_row_gemm's choice.  Against the library's
// products, us, weights from HBM (N rows: M x K, before -> now):
//   64: 1024 x 1024 8.8 -> 3.7,  1024 x 2816 9.7 -> 4.7, 2048 x 5632
//       18.5 -> 11.8, 4096 x 4096 15.5 -> 11.9, 6144 x 4096 17.4 -> 15.9,
//       4096 x 14336 40.7 -> 36.4, 28672 x 4096 48.9 -> 45.8 (5.1 TB/s)
//   16: 1024 x 1024 6.1 -> 3.5, 4096 x 4096 15.9 -> 8.2, 28672 x 4096
//       60.9 -> 37.0 (6.3 TB/s)
// With more rows the bound is what a compute unit takes in, about 50 GB/s:
// every tile reads all of its x and W.
#include "hybrid/row_tile.h"

template <int NT, int MT, int KW, int S>
__global__ __launch_bounds__(KW * 64, 2) void row_gemm_kernel(
    bf16_t* __restrict__ out, const bf16_t* __restrict__ x,
    const bf16_t* __restrict__ w, int N, int M, int K, int ldx) {
  using Tile = RowTile<NT, MT, KW, S>;
  extern __shared__ __align__(1024) char lds[];
  // tiles of the same rows of W are 8 apart: on one XCD
  const int across = (N + 16 * NT - 1) / (16 * NT);
  const int in = blockIdx.x % (8 * across);
  const int tile = blockIdx.x / (8 * across) * 8 + in % 8;
  const int m0 = tile * 16 * MT, n0 = in / 8 * 16 * NT;
  if (m0 >= M) return;
  Tile::run(
      lds, K, tile >> 3,
      [&](int r) {
        return x + (size_t)(n0 + r < N ? n0 + r : N - 1) * ldx;
      },
      [&](int r) { return w + (size_t)(m0 + r < M ? m0 + r : M - 1) * K; });
  Tile::each(lds, [&](int r, int c, f32x4 v) {
    if (n0 + r < N && m0 + c < M)
      *reinterpret_cast<uint2*>(out + (size_t)(n0 + r) * M + m0 + c) =
          make_uint2(to_bf16x2(v[0], v[1]), to_bf16x2(v[2], v[3]));
  });
}

template <int NT, int MT, int KW, int S>
static int row_gemm_launch(void* out, const void* x, const void* w, int N,
                           int M, int K, int ldx, hipStream_t stream) {
  constexpr int lds = RowTile<NT, MT, KW, S>::LDS;
  static_assert(lds <= 160 * 1024, "LDS of a compute unit");
  static const hipError_t sized = hipFuncSetAttribute(
      reinterpret_cast<const void*>(row_gemm_kernel<NT, MT, KW, S>),
      hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (sized != hipSuccess) return -1;
  const int down = (M + 16 * MT - 1) / (16 * MT);
  const int across = (N + 16 * NT - 1) / (16 * NT);
  hipLaunchKernelGGL((row_gemm_kernel<NT, MT, KW, S>),
                     dim3((down + 7) / 8 * 8 * across), dim3(KW * 64), lds,
                     stream, (bf16_t*)out, (const bf16_t*)x, (const bf16_t*)w,
                     N, M, K, ldx);
  HY_CHECK();
  return 0;
}

// 0: done, -2: not for this kernel.  Rows of x start ldx numbers apart.
extern "C" int ll_row_gemm(void* out, const void* x, const void* w, int N,
                           int M, int K, int ldx, void* stream) {
  if (N <= 0 || N > 128 || M <= 0 || K <= 0 || M % 4 || K % 8 || ldx % 8 ||
      (uintptr_t)x % 16 || (uintptr_t)w % 16 || (uintptr_t)out % 8)
    return -2;
  // The largest tile of which there are enough for the chip: a larger one
  // reads less (64 x 64 half of what 32 x 32 does), but under about 176 of
  // them, two thirds of the compute units, idle ones cost more than that
  // (64 rows against 6144 x 4096: 96 tiles of 64 x 64 17.0 us, 192 of
  // 32 x 64 15.9; against 11264 x 2048: 176 of 64 x 64 13.8, 352 of 32 x 64
  // 18).  Rows of x go in equal shares of up to 4 x 16.
  const int tiles = (N + 15) / 16, shares = (tiles + 3) / 4;
  const int nt = (tiles + shares - 1) / shares;
  auto enough = [&](int n, int m) {
    return (size_t)((M + 16 * m - 1) / (16 * m)) * ((tiles + n - 1) / n) >=
           176;
  };
  hipStream_t st = (hipStream_t)stream;
#define ROW_GEMM(NT, MT, KW, S) \
  return row_gemm_launch<NT, MT, KW, S>(out, x, w, N, M, K, ldx, st)
  if (nt == 4) {
    if (enough(4, 4)) ROW_GEMM(4, 4, 4, 2);
    if (enough(4, 2)) ROW_GEMM(4, 2, 4, 2);
  } else if (nt == 3) {
    if (enough(3, 4)) ROW_GEMM(3, 4, 4, 2);
    if (enough(3, 2)) ROW_GEMM(3, 2, 4, 2);
    if (enough(3, 1)) ROW_GEMM(3, 1, 4, 3);
  }
  if (nt >= 2) {
    if (enough(2, 4)) ROW_GEMM(2, 4, 4, 2);
    if (enough(2, 2)) ROW_GEMM(2, 2, 4, 2);
    if (enough(2, 1)) ROW_GEMM(2, 1, 4, 3);
  }
  // few rows, or a small matrix: all of a tile's depth is on its way at once
  if (enough(1, 2)) ROW_GEMM(1, 2, 4, 3);
  ROW_GEMM(1, 1, 8, 2);
#undef ROW_GEMM
}
