// Products of few rows with a weight matrix, for decoding:
//
//   out[N, M] = x[N, K] W[M, K]^T     bf16, summed in float, N <= 128
//
// W is read once and nothing else is large, so the bound is memory for big
// matrices and latency for small ones.  Both wanted the same things:
//  * W and x come by copies to LDS in rows of 128 bytes.  Loading MFMA
//    operands straight into registers asks for 16 bytes of 16 different
//    rows at a time, which the vector memory path serves one lane a cycle:
//    64 rows against 4096 x 14336 took 77 us that way.
//  * The waves of a workgroup share its tile and split the DEPTH, in pieces
//    of 64.  Each copies, waits for and multiplies its own pieces, without
//    a barrier until the sums meet in LDS at the end, and the result needs
//    no second kernel.
//  * Workgroups start at different depths: rows lie a multiple of 4 KB
//    apart, and in step they would all ask the same memory channel (3% to
//    10%).
//
// Sizes of a tile are row_gemm_launch's choice.  Against the library's
// products, us, weights from HBM (N rows: M x K, before -> now):
//   64: 1024 x 1024 8.8 -> 3.7,  1024 x 2816 9.7 -> 4.7, 2048 x 5632
//       18.5 -> 11.8, 4096 x 4096 15.5 -> 11.9, 6144 x 4096 17.4 -> 15.9,
//       4096 x 14336 40.7 -> 36.4, 28672 x 4096 48.9 -> 45.8 (5.1 TB/s)
//   16: 1024 x 1024 6.1 -> 3.5, 4096 x 4096 15.9 -> 8.2, 28672 x 4096
//       60.9 -> 37.0 (6.3 TB/s)
// With more rows the bound is what a compute unit takes in, about 50 GB/s:
// every tile reads all of its x and W.
#include "hybrid/lds_copy.h"
#include "hybrid/mfma.h"

// Tile: 16 MT rows of W, 16 NT rows of x.  KW waves; each has S stages of
// LDS, one piece of 64 of the depth of all the tile's rows a stage.
template <int NT, int MT, int KW, int S>
__global__ __launch_bounds__(KW * 64, 2) void row_gemm_kernel(
    bf16_t* __restrict__ out, const bf16_t* __restrict__ x,
    const bf16_t* __restrict__ w, int N, int M, int K, int ldx) {
  constexpr int ROWS = 16 * (NT + MT), C = ROWS / 8, STAGE = ROWS * 128;
  constexpr int RP = 16 * MT + 4;  // row of the sums
  extern __shared__ __align__(1024) char lds[];
  const int tid = threadIdx.x, lane = tid & 63, lo = lane & 15, hi = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
  // tiles of the same rows of W are 8 apart: on one XCD
  const int across = (N + 16 * NT - 1) / (16 * NT);
  const int in = blockIdx.x % (8 * across);
  const int tile = blockIdx.x / (8 * across) * 8 + in % 8;
  const int m0 = tile * 16 * MT, n0 = in / 8 * 16 * NT;
  if (m0 >= M) return;
  char* const own = lds + wave * (S * STAGE);
  const unsigned own_byte = lds_byte(own);

  // Copy j of a stage fills rows 8 j .. 8 j + 7, 8 lanes a row.  Piece c of
  // 16 bytes of row r lies at c ^ (r / 2 % 8): lanes reading one piece of
  // 16 rows meet every bank once.
  const bf16_t* src[C];
  int piece[C];
#pragma unroll
  for (int j = 0; j < C; ++j) {
    const int r = 8 * j + lane / 8;
    piece[j] = ((lane & 7) ^ ((r >> 1) & 7)) * 8;
    if (j < 2 * NT) {
      const int n = n0 + r;
      src[j] = x + (size_t)(n < N ? n : N - 1) * ldx + piece[j];
    } else {
      const int m = m0 + r - 16 * NT;
      src[j] = w + (size_t)(m < M ? m : M - 1) * K + piece[j];
    }
  }
  const int pieces = (K + 63) / 64;
  const int count = pieces > wave ? (pieces - wave + KW - 1) / KW : 0;
  const int turn = count ? (tile >> 3) % count : 0;
  auto copy = [&](int i) {
    const int at = i + turn;
    const int k0 = (wave + (at < count ? at : at - count) * KW) * 64;
    const unsigned to = own_byte + i % S * STAGE;
#pragma unroll
    for (int j = 0; j < C; ++j) {
      // past the depth both sides are zero
      const bf16_t* p = k0 + piece[j] < K
                            ? src[j] + k0
                            : reinterpret_cast<const bf16_t*>(zero_piece);
      if (j < 2 * NT)
        copy_to_lds(p, to + j * 1024);
      else
        stream_to_lds(p, to + j * 1024);
    }
  };

  f32x4 acc[MT][NT];
#pragma unroll
  for (int a = 0; a < MT; ++a)
#pragma unroll
    for (int b = 0; b < NT; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < S; ++i)
    if (i < count) copy(i);
  for (int i = 0; i < count; ++i) {
    const int newer = count - 1 - i;  // pieces, of which S - 1 are on the way
    if (newer >= S - 1)
      wait_copies<(S - 1) * C>();
    else if (S > 2 && newer == 1)
      wait_copies<(S > 2 ? C : 0)>();
    else
      wait_copies<0>();
    const char* st = own + i % S * STAGE;
    u32x4 wf[2][MT], xf[2][NT];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int at = lo * 128 + ((s * 4 + hi) ^ (lo >> 1)) * 16;
#pragma unroll
      for (int b = 0; b < NT; ++b)
        xf[s][b] = *reinterpret_cast<const u32x4*>(st + b * 2048 + at);
#pragma unroll
      for (int a = 0; a < MT; ++a)
        wf[s][a] = *reinterpret_cast<const u32x4*>(st + (NT + a) * 2048 + at);
    }
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int b = 0; b < NT; ++b)
#pragma unroll
        for (int a = 0; a < MT; ++a)
          acc[a][b] = mfma(wf[s][a], xf[s][b], acc[a][b]);
    // the stage has been read before its next copy starts
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (i + S < count) copy(i + S);
  }

  __syncthreads();  // the sums lie where the stages were
  float* const sums = reinterpret_cast<float*>(lds);
#pragma unroll
  for (int b = 0; b < NT; ++b)
#pragma unroll
    for (int a = 0; a < MT; ++a)
      *reinterpret_cast<f32x4*>(
          &sums[(wave * 16 * NT + b * 16 + lo) * RP + a * 16 + hi * 4]) =
          acc[a][b];
  __syncthreads();
  for (int i = tid; i < 64 * NT * MT; i += KW * 64) {
    const int r = i / (4 * MT), c = i % (4 * MT) * 4;
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int v = 0; v < KW; ++v)
      s += *reinterpret_cast<const f32x4*>(&sums[(v * 16 * NT + r) * RP + c]);
    if (n0 + r < N && m0 + c < M)
      *reinterpret_cast<uint2*>(out + (size_t)(n0 + r) * M + m0 + c) =
          make_uint2(to_bf16x2(s[0], s[1]), to_bf16x2(s[2], s[3]));
  }
}

template <int NT, int MT, int KW, int S>
static int row_gemm_launch(void* out, const void* x, const void* w, int N,
                           int M, int K, int ldx, hipStream_t stream) {
  constexpr int stages = KW * S * 16 * (NT + MT) * 128;
  constexpr int sums = KW * 16 * NT * (16 * MT + 4) * 4;
  constexpr int lds = stages > sums ? stages : sums;
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
