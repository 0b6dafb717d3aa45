// Products of tokens with their experts' matrices, any sizes and either
// type: for every pair of an expert's list (experts.h)
//   out[pair] = act(w[expert] in[pair / div])
// with act(z) = max(z, 0)^2 or none.
//  * expert_float_kernel  32 bits by float_tile.h
//  * expert_rows_kernel   other sizes, tiles of 32 pairs x 64 outputs
#include <math.h>

#include "experts.h"
#include "float_tile.h"

#define BM 32
#define BN 64
#define BK 32

template <typename T>
__global__ __launch_bounds__(256) void expert_rows_kernel(
    T* __restrict__ out, const T* __restrict__ in, const T* __restrict__ w,
    const int* __restrict__ counts, const int* __restrict__ pairs, int E,
    int N, int K, int div, int act, int n_tok) {
  __shared__ float la[BM][BK + 1], lb[BN][BK + 1];
  __shared__ ExpertTiles<BM> tiles;
  if (threadIdx.x < WAVE) tiles.count(counts, E);
  __syncthreads();
  const int i = blockIdx.x, whole = tiles.whole[E - 1];
  if (i >= whole + tiles.rest[E - 1]) return;
  const ExpertTile t =
      tiles.get(counts, E, i < whole ? i : i - whole, i >= whole);
  const int* list = pairs + (size_t)t.expert * n_tok + t.first;
  const T* we = w + (size_t)t.expert * N * K;
  const int n0 = blockIdx.y * BN;
  const int tid = threadIdx.x, r = tid / 8, c = tid % 8;
  const int kr = tid % BK, rr = tid / BK;  // staging: column, first row
  float acc[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) acc[i] = 0.f;
  for (int k0 = 0; k0 < K; k0 += BK) {
    const bool in_k = k0 + kr < K;
#pragma unroll
    for (int i = 0; i < BM; i += 256 / BK)
      la[rr + i][kr] =
          in_k && rr + i < t.n
              ? to_f(in[(size_t)(list[rr + i] / div) * K + k0 + kr])
              : 0.f;
#pragma unroll
    for (int i = 0; i < BN; i += 256 / BK)
      lb[rr + i][kr] = in_k && n0 + rr + i < N
                           ? to_f(we[(size_t)(n0 + rr + i) * K + k0 + kr])
                           : 0.f;
    __syncthreads();
    for (int k = 0; k < BK; ++k) {
      const float a = la[r][k];
#pragma unroll
      for (int i = 0; i < 8; ++i) acc[i] += a * lb[c + i * 8][k];
    }
    __syncthreads();
  }
  if (r >= t.n) return;
  T* dst = out + (size_t)list[r] * N + n0;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    float x = acc[i];
    if (act) {
      x = fmaxf(x, 0.f);
      x *= x;
    }
    if (n0 + c + i * 8 < N) dst[c + i * 8] = from_f<T>(x);
  }
}

struct ExpertRows {
  const void *in, *w;
  void* out;
  const int *counts, *pairs;
  int E, N, K, div, act, n_tok, n_pairs;
  hipStream_t stream;
};

// 16 NT pairs of an expert against 16 MT rows of its matrix.
template <int NT, int MT, int KW>
__global__ __launch_bounds__(KW * 64, KW == 4 ? 2 : 1)
void expert_float_kernel(float* __restrict__ out, const float* __restrict__ in,
                         const float* __restrict__ w,
                         const int* __restrict__ counts,
                         const int* __restrict__ pairs, int E, int N, int K,
                         int div, int act, int n_tok) {
  using Tile = FloatTile<NT, MT, KW>;
  extern __shared__ __align__(1024) char lds[];
  __shared__ ExpertTiles<16 * NT> tiles;
  if (threadIdx.x < WAVE) tiles.count(counts, E);
  __syncthreads();
  const int i = blockIdx.y, whole = tiles.whole[E - 1];
  if (i >= whole + tiles.rest[E - 1]) return;
  const ExpertTile t =
      tiles.get(counts, E, i < whole ? i : i - whole, i >= whole);
  const int* list = pairs + (size_t)t.expert * n_tok + t.first;
  const int n0 = blockIdx.x * 16 * MT, last = N - 1 - n0;
  if (last < 0) return;
  const float* const we = w + ((size_t)t.expert * N + n0) * K;
  auto row = [&](int r) { return list[r < t.n ? r : t.n - 1]; };
  Tile::run(
      lds, K, blockIdx.x + t.expert, in,
      [&](int r) { return (unsigned)(row(r) / div) * (unsigned)K; }, we,
      [&](int r) { return (unsigned)(r < last ? r : last) * (unsigned)K; });
  Tile::finish(
      lds, K, act ? RELU2 : PLAIN, t.n, N - n0,
      [&](int r) { return in + (size_t)(row(r) / div) * K; },
      [&](int c) { return we + (size_t)c * K; },
      [&](int r) { return out + (size_t)row(r) * N + n0; });
}

template <int NT, int MT, int KW>
static int expert_float(const ExpertRows& p) {
  auto* kernel = &expert_float_kernel<NT, MT, KW>;
  constexpr int lds = FloatTile<NT, MT, KW>::LDS;
  static const hipError_t sized = hipFuncSetAttribute(
      reinterpret_cast<const void*>(kernel),
      hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (sized != hipSuccess) return -1;
  const int tiles =
      p.n_pairs / (16 * NT) + (p.E < p.n_pairs ? p.E : p.n_pairs);
  hipLaunchKernelGGL(kernel, dim3((p.N + 16 * MT - 1) / (16 * MT), tiles),
                     dim3(KW * 64), lds, p.stream, (float*)p.out,
                     (const float*)p.in, (const float*)p.w, p.counts, p.pairs,
                     p.E, p.N, p.K, p.div, p.act, p.n_tok);
  HY_CHECK();
  return 0;
}

// Sizes that FloatTile's copies take: whole pieces of 32 of the depth, offsets of
// 32 bits, whole vectors of outputs.
static bool expert_float_ok(const ExpertRows& p) {
  const long long rows = (p.n_pairs + p.div - 1ll) / p.div;
  return p.K % 32 == 0 && p.N % 4 == 0 &&
         ((uintptr_t)p.in | (uintptr_t)p.w | (uintptr_t)p.out) % 16 == 0 &&
         4 * rows * p.K <= 1ll << 32 && 256ll * p.K <= 1ll << 32 &&
         p.n_pairs / 16 + p.E < 65536;
}

// Tiles that there are: how many a compute unit is taken to have at once, us of
// one 1024 deep where each unit has one and where each has all of them, of the
// beginning and end, and of every full round more.  Fitted to 328 products: 4 to 256
// experts, 1 to 8 a token, 1 to 4096 tokens, 96 to 4096 outputs and as deep, weights
// from HBM.  Of 234 others the tile taken is 2.2% slower than the fastest on average
// and 20 are more than 10% slower, 28% at most (by pairs an expert and the depth
// alone, from 16 experts of 1024 x 256, 5.4%, 47 and 46%).  us, expert_rows_kernel ->
// these, 16 experts, 4 a token, up (256 outputs, 1024 deep) and down (1024, 256 deep):
// 20 tokens 138 -> 8.4, 38 -> 7.9; 100 155 -> 10.9, 46 -> 10.4; 300 172 -> 20, 90 ->
// 17.5; 1200 376 -> 27, 231 -> 37.
struct ExpertTileTime {
  int rows, cols, at_once;
  float one, all, ends, more;
};
static const ExpertTileTime EXPERT_TILES[] = {
    {16, 32, 3, 2.3f, 6.5f, 6.8f, 1.f},  {32, 32, 2, 3.2f, 6.4f, 6.8f, 3.3f},
    {48, 32, 2, 4.3f, 10.4f, 7.f, 1.f},  {48, 64, 2, 6.9f, 13.5f, 6.9f, 0.f},
    {64, 64, 2, 6.5f, 13.5f, 8.2f, 0.f}};

// The tile that is estimated to take least.  An expert has its share of the pairs
// and as many more as their root, by which shares differ.
static int expert_float_tile(const ExpertRows& p) {
  const int experts = p.E < p.n_pairs ? p.E : p.n_pairs;
  const float each = (float)p.n_pairs / experts, most = each + sqrtf(each);
  int best = 0;
  float least = 0.f;
  for (int t = 0; t < 5; ++t) {
    const ExpertTileTime& at = EXPERT_TILES[t];
    const float tiles = each < 4.f * at.rows ? ceilf(most / at.rows)
                                             : each / at.rows + 0.5f;
    const long long n =
        (long long)(experts * tiles) * ((p.N + at.cols - 1ll) / at.cols);
    const int round = 256 * at.at_once, rest = (int)(n % round);
    const float full = (float)(n / round);
    float us = full * at.all;
    if (rest)
      us += at.one + (at.all - at.one) * (float)((rest - 1) / 256) /
                         (float)(at.at_once - 1);
    us = us * ((float)p.K / 1024.f) + at.ends + full * at.more;
    if (t == 0 || us < least) least = us, best = t;
  }
  return best;
}

static int expert_float_pick(const ExpertRows& p) {
  switch (expert_float_tile(p)) {
    case 0: return expert_float<1, 2, 8>(p);
    case 1: return expert_float<2, 2, 8>(p);
    case 2: return expert_float<3, 2, 8>(p);
    case 3: return expert_float<3, 4, 4>(p);
    default: return expert_float<4, 4, 4>(p);
  }
}

extern "C" int hy_expert_rows(void* out, const void* in, const void* w,
                              const void* counts, const void* pairs, int E,
                              int N, int K, int div, int act, int n_tok,
                              int n_pairs, int dtype, void* stream) {
  if (E <= 0 || E > EXPERTS_MAX || N <= 0 || K <= 0 || div <= 0 || N > 65535 * BN) return -2;
  if (n_tok <= 0 || n_pairs <= 0) return 0;
  const ExpertRows p{in, w, out, (const int*)counts, (const int*)pairs, E, N,
                     K, div, act, n_tok, n_pairs, (hipStream_t)stream};
  if (dtype == 1 && expert_float_ok(p)) return expert_float_pick(p);
  const int tiles = n_pairs / BM + (E < n_pairs ? E : n_pairs);
  HY_DTYPE(dtype, hipLaunchKernelGGL(
      expert_rows_kernel<T>, dim3(tiles, (N + BN - 1) / BN), dim3(256), 0,
      (hipStream_t)stream, (T*)out, (const T*)in, (const T*)w,
      (const int*)counts, (const int*)pairs, E, N, K, div, act, n_tok));
  HY_CHECK();
  return 0;
}
