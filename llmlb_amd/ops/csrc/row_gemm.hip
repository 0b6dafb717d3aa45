// Products of few rows with a weight matrix, for decoding:
//
//   out[N, M] = x[N, K] W[M, K]^T     bf16, summed in float, N <= 128
//
// W is read once and nothing else is large, so the bound is memory for big
// matrices and latency for small ones; hybrid/row_tile.h says how a tile is
// computed.  Deep matrices of more than 31 rows take the depth in shares, and
// a second kernel that adds them up, or the norm that follows does, for which
// matrices of few tiles are taken in shares too.
//
// Sizes of a tile are ll_row_gemm's choice.  Against the library's
// products, us, weights from HBM (N rows: M x K, before -> now):
//   64: 1024 x 1024 8.8 -> 3.7,  1024 x 2816 9.7 -> 4.7, 2048 x 5632
//       18.5 -> 11.8, 4096 x 4096 15.5 -> 11.9, 6144 x 4096 17.4 -> 15.9,
//       4096 x 14336 40.7 -> 30.0 (in shares; 36.4 in one), 28672 x 4096
//       48.9 -> 40.0 (5.9 TB/s)
//   16: 1024 x 1024 6.1 -> 3.5, 4096 x 4096 15.9 -> 8.2, 28672 x 4096
//       60.9 -> 37.0 (6.3 TB/s)
// With more rows it is what a compute unit takes in, as every tile reads all of
// its x and W: about 50 GB/s here, of 115 that copies alone reach from the L2.
// A wave waits for its pieces, and deeper rings, eight waves or fetching W in
// the kernel before gained 0.3 to 1.4 us.
#include "hybrid/norm_tile.h"
#include "hybrid/row_act.h"
#include "hybrid/row_tile.h"

// What becomes of the sums of a tile's row n of x: put(.., n, m, ..) stores
// those of outputs m .. m + 3.  PAIRED: a tile's rows of W are first(m) and, as
// many, second(m) of the same outputs.  What put will need that does not depend
// on the sums is asked for before they are made: token(n) at once, early(token,
// m), which takes a token's position to its table, with the last piece.
struct PlainEnd {
  static constexpr bool PAIRED = false;
  struct Token {};
  struct Early {};
  RowAct act;
  __device__ __forceinline__ Token token(int) const { return {}; }
  __device__ __forceinline__ Early early(Token, int) const { return {}; }
  __device__ __forceinline__ int first(int m) const { return m; }
  __device__ __forceinline__ int second(int m) const { return m; }
  // CAPPED results are floats, all others bf16
  __device__ __forceinline__ void put(void* out, int ld_out, int n, int m,
                                      Early, f32x4 v, f32x4) const {
    if (act.kind != PLAIN) {
      v = rounded(v);
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = row_act(act, v[i]);
    }
    const size_t at = (size_t)n * ld_out + m;
    if (act.kind == CAPPED)
      *reinterpret_cast<f32x4*>(static_cast<float*>(out) + at) = v;
    else
      *reinterpret_cast<uint2*>(static_cast<bf16_t*>(out) + at) =
          make_uint2(to_bf16x2(v[0], v[1]), to_bf16x2(v[2], v[3]));
  }
};
// gate and up
struct GatedEnd {
  static constexpr bool PAIRED = true;
  struct Token {};
  struct Early {};
  RowAct act;
  __device__ __forceinline__ Token token(int) const { return {}; }
  __device__ __forceinline__ Early early(Token, int) const { return {}; }
  __device__ __forceinline__ int first(int m) const { return m; }
  __device__ __forceinline__ int second(int m) const { return act.up + m; }
  __device__ __forceinline__ void put(void* out, int ld_out, int n, int m,
                                      Early, f32x4 v, f32x4 u) const {
    v = rounded(v);
    u = rounded(u);
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = row_gate(act, v[i], u[i]);
    *reinterpret_cast<uint2*>(static_cast<bf16_t*>(out) +
                              (size_t)n * ld_out + m) =
        make_uint2(to_bf16x2(v[0], v[1]), to_bf16x2(v[2], v[3]));
  }
};
// Queries, keys and values: the first two are rotated (halves of a head
// together), and with caches keys and values are copied to the page slot of
// their token as well; a slot below 0 has no place.  What rope_kv_append does
// in a launch of its own, to the bit: decoding pays for launches.  us a step
// with both, with this: one sequence of a small model 135.2, 127.9; 64 of four
// layers of an 8B model 650.1, 644.2; 32 with 8-bit caches (rotation only)
// 551.2, 546.7.
struct RotaryEnd {
  static constexpr bool PAIRED = true;
  struct Token {
    int position, slot;
  };
  struct Early {
    float4 c, s;
    int slot;
  };
  const float* cos_sin;        // [position][cosines, sines]
  const int *positions, *slots;
  bf16_t *kcache, *vcache;     // null: no caches
  int shift, n_q, n_kv, page;  // half a head is 1 << shift numbers
  __device__ __forceinline__ Token token(int n) const {
    return {positions[n], kcache ? slots[n] : -1};
  }
  __device__ __forceinline__ Early early(Token t, int m) const {
    const int half = 1 << shift, head = m >> shift, j = m & (half - 1);
    Early e{};
    if (head < n_q + n_kv) {
      const float* cs = cos_sin + (size_t)t.position * (2 * half) + j;
      e.c = *reinterpret_cast<const float4*>(cs);
      e.s = *reinterpret_cast<const float4*>(cs + half);
    }
    e.slot = head >= n_q ? t.slot : -1;
    return e;
  }
  __device__ __forceinline__ int first(int m) const {
    return m + (m >> shift << shift);
  }
  __device__ __forceinline__ int second(int m) const {
    return first(m) + (1 << shift);
  }
  __device__ __forceinline__ void put(void* out, int ld_out, int n, int m,
                                      const Early& e, f32x4 v, f32x4 u) const {
    const int half = 1 << shift, head = m >> shift, j = m & (half - 1);
    v = rounded(v);
    u = rounded(u);
    if (head < n_q + n_kv) {
      const float c[4] = {e.c.x, e.c.y, e.c.z, e.c.w};
      const float s[4] = {e.s.x, e.s.y, e.s.z, e.s.w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float a = v[i], b = u[i];
        v[i] = fmaf(a, c[i], -(b * s[i]));
        u[i] = fmaf(b, c[i], a * s[i]);
      }
    }
    const uint2 lo = make_uint2(to_bf16x2(v[0], v[1]), to_bf16x2(v[2], v[3]));
    const uint2 hi = make_uint2(to_bf16x2(u[0], u[1]), to_bf16x2(u[2], u[3]));
    bf16_t* to = static_cast<bf16_t*>(out) + (size_t)n * ld_out + first(m);
    *reinterpret_cast<uint2*>(to) = lo;
    *reinterpret_cast<uint2*>(to + half) = hi;
    if (e.slot < 0) return;
    const bool is_v = head >= n_q + n_kv;
    to = (is_v ? vcache : kcache) +
         (((size_t)(e.slot / page) * n_kv + head - n_q - (is_v ? n_kv : 0)) *
              page +
          e.slot % page) *
             (2 * half) +
         j;
    *reinterpret_cast<uint2*>(to) = lo;
    *reinterpret_cast<uint2*>(to + half) = hi;
  }
};

// The order in which a sum is made differs with the number of rows, as with
// any product: tiles, waves and shares follow from it.  M outputs, of PAIRED
// ends pairs; block: of the product's workgroups.
template <int NT, int MT, int KW, int S, class End>
__device__ __forceinline__ void row_gemm_block(
    char* lds, int block, void* __restrict__ out, int ld_out,
    const bf16_t* __restrict__ x, const bf16_t* __restrict__ w, int N, int M,
    int K, int ldx, const End& end) {
  using Tile = RowTile<NT, MT, KW, S>;
  constexpr int OUT = End::PAIRED ? 8 * MT : 16 * MT;  // outputs a tile
  constexpr int ITEMS = 16 * NT * (OUT / 4);
  // tiles of the same rows of W are 8 apart: on one XCD
  const int across = (N + 16 * NT - 1) / (16 * NT);
  const int in = block % (8 * across);
  const int tile = block / (8 * across) * 8 + in % 8;
  const int m0 = tile * OUT, n0 = in / 8 * 16 * NT;
  if (m0 >= M) return;
  auto here = [&](int i, int& n, int& m) {
    n = n0 + i / (OUT / 4), m = m0 + i % (OUT / 4) * 4;
    return i < ITEMS && n < N && m < M;
  };
  int n, m;
  typename End::Token token{};
  typename End::Early early{};
  const bool some = here(threadIdx.x, n, m);
  if (some) token = end.token(n);
  Tile::run(
      lds, K, tile >> 3,
      [&](int r) {
        return x + (size_t)(n0 + r < N ? n0 + r : N - 1) * ldx;
      },
      [&](int r) {
        const bool other = End::PAIRED && r >= OUT;
        int m = m0 + (other ? r - OUT : r);
        m = m < M ? m : M - 1;
        return w + (size_t)(other ? end.second(m) : end.first(m)) * K;
      },
      0,
      [&] {
        if (some) early = end.early(token, m);
      });
  for (int i = threadIdx.x; i < ITEMS; i += KW * 64) {
    if (!here(i, n, m)) continue;
    if (i != (int)threadIdx.x) early = end.early(end.token(n), m);
    const f32x4 v = Tile::sum(lds, n - n0, m - m0);
    const f32x4 u = End::PAIRED ? Tile::sum(lds, n - n0, m - m0 + OUT) : v;
    end.put(out, ld_out, n, m, early, v, u);
  }
}

template <int NT, int MT, int KW, int S, class End>
__global__ __launch_bounds__(KW * 64, NT * MT > 24 ? 1 : 2)
void row_gemm_kernel(
    void* __restrict__ out, int ld_out, const bf16_t* __restrict__ x,
    const bf16_t* __restrict__ w, int N, int M, int K, int ldx, End end) {
  extern __shared__ __align__(1024) char lds[];
  row_gemm_block<NT, MT, KW, S>(lds, blockIdx.x, out, ld_out, x, w, N, M, K,
                                ldx, end);
}

// Two products of equally many rows and equal depth, of which neither needs
// the other: the first ``blocks`` workgroups do one, the others the other.
// A launch less, and one beginning, last round and end for both.
struct RowOperands {
  void* out;
  const bf16_t *x, *w;
  int ld_out, M, ldx;
};
template <int NT, int MT, int KW, int S>
__global__ __launch_bounds__(KW * 64, NT * MT > 24 ? 1 : 2)
void row_gemm_two_kernel(RowOperands a, PlainEnd a_end, RowOperands b,
                         GatedEnd b_end, int blocks, int N, int K) {
  extern __shared__ __align__(1024) char lds[];
  if ((int)blockIdx.x < blocks)
    row_gemm_block<NT, MT, KW, S>(lds, blockIdx.x, a.out, a.ld_out, a.x, a.w,
                                  N, a.M, K, a.ldx, a_end);
  else
    row_gemm_block<NT, MT, KW, S>(lds, blockIdx.x - blocks, b.out, b.ld_out,
                                  b.x, b.w, N, b.M, K, b.ldx, b_end);
}

// The same of a few normed rows: out = norm(x) W^T
template <int MT, int KW, int S, class End>
__global__ __launch_bounds__(KW * 64, 2) void row_gemm_normed_kernel(
    void* __restrict__ out, int ld_out, const bf16_t* __restrict__ x,
    const bf16_t* __restrict__ w, int N, int M, int K, int ldx, RowNorm norm,
    End end) {
  using Tile = NormTile<MT, KW, S>;
  constexpr int OUT = End::PAIRED ? 8 * MT : 16 * MT;
  constexpr int ITEMS = 16 * (OUT / 4);
  extern __shared__ __align__(1024) char lds[];
  const int tile = blockIdx.x, m0 = tile * OUT;
  auto here = [&](int i, int& n, int& m) {
    n = i / (OUT / 4), m = m0 + i % (OUT / 4) * 4;
    return i < ITEMS && n < N && m < M;
  };
  int n, m;
  typename End::Token token{};
  typename End::Early early{};
  const bool some = here(threadIdx.x, n, m);
  if (some) token = end.token(n);
  Tile::run(
      lds, N, K, tile >> 3, x, ldx, norm, tile == 0,
      [&](int r) {
        const bool other = End::PAIRED && r >= OUT;
        int m = m0 + (other ? r - OUT : r);
        m = m < M ? m : M - 1;
        return w + (size_t)(other ? end.second(m) : end.first(m)) * K;
      },
      [&] {
        if (some) early = end.early(token, m);
      });
  for (int i = threadIdx.x; i < ITEMS; i += KW * 64) {
    if (!here(i, n, m)) continue;
    if (i != (int)threadIdx.x) early = end.early(end.token(n), m);
    const f32x4 v = Tile::sum(lds, n, m - m0);
    const f32x4 u = End::PAIRED ? Tile::sum(lds, n, m - m0 + OUT) : v;
    end.put(out, ld_out, n, m, early, v, u);
  }
}

// A share of the depth, ``depth`` numbers from blockIdx.y * depth on, into
// ws [shares][N][M] floats.
template <int NT, int MT, int KW, int S>
__global__ __launch_bounds__(KW * 64, 2) void row_gemm_share_kernel(
    float* __restrict__ ws, const bf16_t* __restrict__ x,
    const bf16_t* __restrict__ w, int N, int M, int K, int ldx, int depth) {
  using Tile = RowTile<NT, MT, KW, S>;
  extern __shared__ __align__(1024) char lds[];
  const int across = (N + 16 * NT - 1) / (16 * NT);
  const int in = blockIdx.x % (8 * across);
  const int tile = blockIdx.x / (8 * across) * 8 + in % 8;
  const int m0 = tile * 16 * MT, n0 = in / 8 * 16 * NT;
  if (m0 >= M) return;
  const int k0 = blockIdx.y * depth;
  Tile::run(
      lds, K - k0 < depth ? K - k0 : depth, tile >> 3,
      [&](int r) {
        return x + (size_t)(n0 + r < N ? n0 + r : N - 1) * ldx + k0;
      },
      [&](int r) {
        return w + (size_t)(m0 + r < M ? m0 + r : M - 1) * K + k0;
      });
  Tile::each(4 * MT, [&](int r, int c) {
    if (n0 + r >= N || m0 + c >= M) return;
    *reinterpret_cast<f32x4*>(
        ws + ((size_t)blockIdx.y * N + n0 + r) * M + m0 + c) =
        Tile::sum(lds, r, c);
  });
}

// out = the sum of the shares, four outputs a thread.  Four shares are asked
// for at a time: what bounds this is a chain of loads.  us with the product, one
// after the other -> now: 64 rows of 4096 x 14336 28.5 -> 28.1, 32 25.1 -> 24.4.
__global__ __launch_bounds__(256) void row_gemm_join_kernel(
    bf16_t* __restrict__ out, int ld_out, const float* __restrict__ ws, int N,
    int M, int shares) {
  const int i = blockIdx.x * 256 + threadIdx.x, n = i / (M / 4);
  if (n >= N) return;
  const int m = (i - n * (M / 4)) * 4;
  f32x4 v = {0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < shares; s0 += 4) {
    f32x4 part[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int s = s0 + i < shares ? s0 + i : shares - 1;
      part[i] =
          *reinterpret_cast<const f32x4*>(ws + ((size_t)s * N + n) * M + m);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (s0 + i < shares) v += part[i];
  }
  *reinterpret_cast<uint2*>(out + (size_t)n * ld_out + m) =
      make_uint2(to_bf16x2(v[0], v[1]), to_bf16x2(v[2], v[3]));
}

// residual += the sum of the shares, rounded to bf16 first, out = its RMS norm,
// as rmsnorm (kernels.hip) of the joined product.  A row has a thread for every
// vector, which asks for all that it needs at once.
template <int THREADS>
__global__ __launch_bounds__(THREADS) void rmsnorm_join_kernel(
    bf16_t* __restrict__ out, const float* __restrict__ ws, int shares,
    const bf16_t* __restrict__ weight, bf16_t* __restrict__ residual, int width,
    float eps) {
  __shared__ float red[THREADS / WAVE];
  const int i = threadIdx.x * 8;
  const size_t at = (size_t)blockIdx.x * width + i;
  const bool own = i < width;
  float f[8], r[8], w[8], ssq = 0.f;
  if (own) {
    load8(weight + i, w);
    load8(residual + at, r);
    join8(ws + at, shares, (size_t)gridDim.x * width, f);
#pragma unroll
    for (int j = 0; j < 8; ++j) f[j] += r[j];
#pragma unroll
    for (int j = 0; j < 8; j += 2) {
      round_bf16x2(f[j], f[j + 1]);
      ssq += f[j] * f[j];
      ssq += f[j + 1] * f[j + 1];
    }
    store8(residual + at, f);
  }
  const float scale = rsqrtf(block_sum<THREADS>(ssq, red) / width + eps);
  if (!own) return;
#pragma unroll
  for (int j = 0; j < 8; ++j) f[j] = f[j] * scale * w[j];
  store8(out + at, f);
}

template <class End>
struct RowGemm {
  void* out;
  int ld_out;
  const bf16_t *x, *w;
  int N, M, K, ldx;
  End end;
  hipStream_t stream;
};

template <int MT, int KW, int S, class End>
static int row_gemm_normed_launch(const RowGemm<End>& p, const RowNorm& norm) {
  auto* kernel = &row_gemm_normed_kernel<MT, KW, S, End>;
  using Tile = NormTile<MT, KW, S>;
  static const hipError_t sized = hipFuncSetAttribute(
      reinterpret_cast<const void*>(kernel),
      hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
  const int lds = Tile::lds(p.N, p.K);
  if (sized != hipSuccess) return -1;
  if (p.K > Tile::DEEPEST || lds > 160 * 1024) return -2;
  constexpr int OUT = End::PAIRED ? 8 * MT : 16 * MT;
  hipLaunchKernelGGL(kernel, dim3((p.M + OUT - 1) / OUT), dim3(KW * 64), lds,
                     p.stream, p.out, p.ld_out, p.x, p.w, p.N, p.M, p.K,
                     p.ldx, norm, p.end);
  HY_CHECK();
  return 0;
}

template <int NT, int MT, int KW, int S, class End>
static int row_gemm_launch(const RowGemm<End>& p) {
  auto* kernel = &row_gemm_kernel<NT, MT, KW, S, End>;
  constexpr int lds = RowTile<NT, MT, KW, S>::LDS;
  static_assert(lds <= 160 * 1024, "LDS of a compute unit");
  static const hipError_t sized = hipFuncSetAttribute(
      reinterpret_cast<const void*>(kernel),
      hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (sized != hipSuccess) return -1;
  constexpr int OUT = End::PAIRED ? 8 * MT : 16 * MT;
  const int down = (p.M + OUT - 1) / OUT;
  const int across = (p.N + 16 * NT - 1) / (16 * NT);
  hipLaunchKernelGGL(kernel, dim3((down + 7) / 8 * 8 * across), dim3(KW * 64),
                     lds, p.stream, p.out, p.ld_out, p.x, p.w, p.N, p.M, p.K,
                     p.ldx, p.end);
  HY_CHECK();
  return 0;
}

// The tile of which a compute unit takes in least.  What bounds all but the
// fewest rows is the busiest compute unit's intake (see above): the tiles
// that it gets, of 256 at a time, times the rows of a tile, of x and of W.  So
// what counts is that a last round is full, or that there is none.  64 rows,
// us, the largest tile with 176 of its kind before -> now: 19456 x 4096 43.4 (64
// outputs a tile, two rounds) -> 30.1 (80, one), 16512 x 4096 42.3 -> 28.0,
// 10272 x 4096 30.3 -> 21.2 (48), gate and up of 11904 x 4096 45.2 -> 35.3 (96),
// 8224 x 2048 16.4 -> 11.7; 16 rows: 12576 x 4096 21.0 -> 17.5; 128 rows: 10272 x
// 4096 38.3 -> 27.6, gate and up of 5632 x 2048 23.2 -> 16.5.  112 outputs a
// tile are for what they fit into one round, or two: 64 rows, from tiles of 64
// on, gate and up of 14336 x 4096 47.6 -> 39.8, 26000 x 2048 27.8 -> 22.1,
// 57344 x 1024 (two) 31.5 -> 29.9; with five rounds they lose (40 rows, 128256
// x 4096 170 -> 178: the card's memory is the bound).  One 16 of rows is mostly
// bound by memory, and small tiles, of which a unit has two, are less uneven
// than whole rounds say: another than 32 outputs has to take in 15% less (one
// row of 20480 x 1024 11.0 with 48, 10.1 with 32; 16512 x 1024 9.2 with 32, 8.6
// with 80).
// takes_in: rows that the busiest unit takes in, in 16s
static int row_gemm_tile(int N, long long rows, int K, bool paired,
                         long long beside = 0, float* takes_in = nullptr) {
  const int tiles = (N + 15) / 16;
  // what memory takes for W, in the same unit: 16 rows at 50 GB/s
  const float floor = (rows + beside) / 2500.f;
  int nt = 0, mt = 0;
  float least = 0.f;
  auto look = [&](int n, int m) {
    // tiles of the same rows of W are on one of eight XCDs of 32 units
    const long long down = (rows + 16 * m - 1) / (16 * m);
    const long long other = (beside + 16 * m - 1) / (16 * m);
    const long long count =
        ((down + 7) / 8 + (other + 7) / 8) * ((tiles + n - 1) / n);
    const long long rounds = (count + 31) / 32;
    if (m == 7 && rounds > 2) return;  // memory bounds these, of any tile
    const float takes = fmaxf((float)(rounds * (n + m)), floor);
    const float by = n == 1 ? 0.85f : 0.95f;
    if (!nt || takes < by * least) least = takes, nt = n, mt = m;
  };
  // what is as good: more rows of x, which read W less often, then the sizes
  // that memory likes best
  static const int OF_MANY[] = {4, 5, 6, 3, 2, 1, 7};
  static const int OF_ONE[] = {2, 3, 4, 1, 5, 5, 5};
  for (int n = tiles < 4 ? tiles : 4; n >= 1; --n)
    for (int i = 0; i < 7; ++i) {
      const int m = n == 1 ? OF_ONE[i] : OF_MANY[i];
      // (3, 1) and (4, 1) take in no less; of gate and up, tiles of 8 outputs
      // by eight waves are for what they share (1024 x 128, one row: 3.0 with
      // them, 2.8 with 16; 1024 x 768 3.4, 3.7)
      if ((n < 3 || m > 1) && (!paired || m > 1 || K > 256)) look(n, m);
    }
  if (takes_in) *takes_in = least;
  return nt * 8 + mt;
}

// all tiles: waves that share the depth, and pieces of it on their way, fit LDS
#define ROW_GEMM_TILES(GO) \
  GO(1, 1, 8, 2)           \
  GO(1, 2, 4, 3)           \
  GO(1, 3, 4, 3)           \
  GO(1, 4, 4, 3)           \
  GO(1, 5, 4, 3)           \
  GO(2, 1, 4, 3)           \
  GO(2, 2, 4, 2)           \
  GO(2, 3, 4, 2)           \
  GO(2, 4, 4, 2)           \
  GO(2, 5, 4, 2)           \
  GO(2, 6, 4, 2)           \
  GO(2, 7, 4, 2)           \
  GO(3, 2, 4, 2)           \
  GO(3, 3, 4, 2)           \
  GO(3, 4, 4, 2)           \
  GO(3, 5, 4, 2)           \
  GO(3, 6, 4, 2)           \
  GO(3, 7, 4, 2)           \
  GO(4, 2, 4, 2)           \
  GO(4, 3, 4, 2)           \
  GO(4, 4, 4, 2)           \
  GO(4, 5, 4, 2)           \
  GO(4, 6, 4, 2)           \
  GO(4, 7, 3, 2)

template <class End>
static int row_gemm_pick(const RowGemm<End>& p) {
  const long long rows = End::PAIRED ? 2ll * p.M : p.M;
  switch (row_gemm_tile(p.N, rows, p.K, End::PAIRED)) {
#define GO(NT, MT, KW, S) \
  case NT * 8 + MT: return row_gemm_launch<NT, MT, KW, S>(p);
    ROW_GEMM_TILES(GO)
#undef GO
  }
  return -2;
}

// The tile is chosen for the tiles of both.  us, a layer's input projection and
// its gate and up, one after the other -> together (rows: outputs, pairs, depth):
//   1: 4160, 2176 of 1024 9.0 -> 6.3, 8320, 4352 of 2048 15.8 -> 13.1, 16512,
//       11904 of 4096 52.4 -> 48.1; 64: 12.0 -> 8.2, 24.1 -> 17.2, 61.6 -> 60.2;
//       128: 14.5 -> 10.1, 29.5 -> 27.9, 103.4 -> 99.4
// Where one tile for both takes in so much more than each product's own that the
// launch is not worth it (3 us at 50 GB/s, of up to 16 rows, which memory bounds,
// 3.6), they stay apart: 72, 100 and 128 rows of 8192, 6144 of 4096 47.1 -> 50.8,
// 51.3 -> 55.2, 50.6 -> 54.4, of 6144, 4096 of 6144 57.6 -> 60.9, 62.9 -> 65.0, 60.6
// -> 62.6; 64 of 1024, 14336 of 4096 46.5 -> 48.2; 1 and 16 of 16384, 5632 of 6144
// 56.0 -> 56.6, 57.5 -> 59.3, but of 10240, 11904 of 4096, which take in just less,
// 48.4 -> 47.5, 49.6 -> 49.2.  Of 150 other sizes three lose in one launch, 0.2 to
// 2.5%, which all lie beyond this line, as do two that gain 0.1 and 1.7%.
struct RowGemmTwo {
  RowOperands a, b;
  PlainEnd a_end;
  GatedEnd b_end;
  int N, K;
  hipStream_t stream;
};
template <int NT, int MT, int KW, int S>
static int row_gemm_two_launch(const RowGemmTwo& p) {
  auto* kernel = &row_gemm_two_kernel<NT, MT, KW, S>;
  constexpr int lds = RowTile<NT, MT, KW, S>::LDS;
  static const hipError_t sized = hipFuncSetAttribute(
      reinterpret_cast<const void*>(kernel),
      hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (sized != hipSuccess) return -1;
  const int across = (p.N + 16 * NT - 1) / (16 * NT);
  auto blocks = [&](int M, int out) {
    return ((M + out - 1) / out + 7) / 8 * 8 * across;
  };
  const int first = blocks(p.a.M, 16 * MT), second = blocks(p.b.M, 8 * MT);
  hipLaunchKernelGGL(kernel, dim3(first + second), dim3(KW * 64), lds,
                     p.stream, p.a, p.a_end, p.b, p.b_end, first, p.N, p.K);
  HY_CHECK();
  return 0;
}

// Of a few normed rows, see norm_gains.
template <class End>
static int row_gemm_normed(const RowGemm<End>& p, const RowNorm& norm) {
  const long long rows = End::PAIRED ? 2ll * p.M : p.M;
  switch (row_gemm_tile(p.N, rows, p.K, End::PAIRED)) {
    case 9: return row_gemm_normed_launch<1, 8, 2>(p, norm);
    case 10: return row_gemm_normed_launch<2, 4, 3>(p, norm);
    case 11: return row_gemm_normed_launch<3, 4, 3>(p, norm);
    case 12: return row_gemm_normed_launch<4, 4, 3>(p, norm);
    case 13: return row_gemm_normed_launch<5, 4, 3>(p, norm);
  }
  return -2;
}

// In how many shares the depth is taken.  A deep matrix of so few rows that
// only small tiles fill the chip is bound by what these read of x, not by
// its own size: larger tiles of a part of the depth read half, for a second
// launch that adds the parts up.  us, weights from HBM, in one -> in shares:
//   64 rows: 4096 x 14336 40.2 -> 30.0, 4096 x 19456 54.2 -> 38.6,
//       4096 x 8192 22.8 -> 20.3, 6144 x 8192 32.2 -> 29.2
//   32 rows: 4096 x 14336 33.9 -> 25.9, 4096 x 8192 18.2 -> 17.6
//   128 rows: 4096 x 14336 50.7 -> 45.8, 2048 x 8192 18.8 -> 17.8
// Not gained by it: 17 rows (4096 x 8192 15.2 -> 16.9), 128 rows of 4096 x
// 4096 (15.5 -> 16.8), 64 of 2048 x 8192 in shares of 1024 (14.8 -> 16.9 at
// best).
extern "C" int ll_row_gemm_shares(int N, int M, int K) {
  if (N < 32 || N > 128 || K < 8192 || M <= 0 || M % 4) return 1;
  const int tiles = (N + 15) / 16, across = (tiles + 3) / 4;
  const int large = (M + 63) / 64 * across;
  if (large >= 176) return 1;
  const int most = K / 2048, shares = 256 / large < most ? 256 / large : most;
  return shares >= 2 && large * shares >= 176 ? shares : 1;
}

// Tiles of rows: from 33 rows on two where the shares of both are still no more
// workgroups than compute units.
static int share_across(int N, int M, int shares) {
  return N > 64 || (N > 32 && (M + 31ll) / 32 * 2 * shares <= 256) ? 2 : 1;
}
// Workgroups that shares of tiles of 16 mt outputs make, and the tile: the larger
// where there are enough of it for most compute units.
static long long share_blocks(int N, int M, int mt, int shares) {
  return (M + 16ll * mt - 1) / (16 * mt) * share_across(N, M, shares) * shares;
}
static int share_tile(int N, int M, int shares) {
  return share_blocks(N, M, 4, shares) >= 176 ? 4 : 2;
}

template <int NT, int MT, int KW, int S>
static int row_gemm_share_launch(float* ws, const bf16_t* x, const bf16_t* w,
                                 int shares, int N, int M, int K, int ldx,
                                 hipStream_t stream) {
  auto* kernel = &row_gemm_share_kernel<NT, MT, KW, S>;
  constexpr int lds = RowTile<NT, MT, KW, S>::LDS;
  static_assert(lds <= 160 * 1024, "LDS of a compute unit");
  static const hipError_t sized = hipFuncSetAttribute(
      reinterpret_cast<const void*>(kernel),
      hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (sized != hipSuccess) return -1;
  const int depth = ((K + shares - 1) / shares + 63) / 64 * 64;
  const int parts = (K + depth - 1) / depth;
  const int across = (N + 16 * NT - 1) / (16 * NT);
  const int down = (M + 16 * MT - 1) / (16 * MT);
  hipLaunchKernelGGL(kernel, dim3((down + 7) / 8 * 8 * across, parts),
                     dim3(KW * 64), lds, stream, ws, x, w, N, M, K, ldx,
                     depth);
  return hipGetLastError() == hipSuccess ? parts : -1;
}

// The shares alone, ws [shares][N][M] floats; > 0: as many as there are (with
// rounding to pieces of 64, up to ``shares``), -2: not for this kernel.
extern "C" int ll_row_gemm_parts(const void* x, const void* w, void* ws,
                                 int shares, int N, int M, int K, int ldx,
                                 void* stream) {
  if (N <= 0 || N > 128 || M <= 0 || K <= 0 || M % 4 || K % 8 || ldx % 8 ||
      (uintptr_t)x % 16 || (uintptr_t)w % 16 || (uintptr_t)ws % 16 ||
      shares < 1 || shares > 256)
    return -2;
  const int tiles = (N + 15) / 16, across = share_across(N, M, shares);
  switch ((tiles + across - 1) / across * 8 +
          share_tile(N, M, shares) - 1) {
#define GO(NT, MT, KW, S)                                                  \
  case NT * 8 + MT - 1:                                                    \
    return row_gemm_share_launch<NT, MT, KW, S>(                           \
        (float*)ws, (const bf16_t*)x, (const bf16_t*)w, shares, N, M, K,   \
        ldx, (hipStream_t)stream);
    GO(1, 2, 8, 3)
    GO(1, 4, 4, 4)
    GO(2, 2, 8, 2)
    GO(2, 4, 4, 2)
    GO(3, 2, 4, 3)
    GO(3, 4, 4, 2)
    GO(4, 2, 4, 3)
    GO(4, 4, 4, 2)
#undef GO
  }
  return -2;
}

// In how many shares a product whose shares the norm after it adds up, which
// reads them in the launch that it needs anyway.  So more gain than of those that
// need a launch to join: all whose outputs make few tiles, which leave compute units
// idle (up to 16 rows of 2048 outputs are 128 workgroups) or read x that much more
// often.  What bounds it: a second round of workgroups costs more than shares gain
// (48 rows of 2560 x 4096 in two shares, 160 workgroups, 3% faster, in four, 320,
// 13% slower), so there is at most one for every compute unit; and sums are more to
// write and read, so that each share needs some depth, more of it the more sums
// there are.  Product and norm, whole -> shares, us, weights from HBM (by
// post_norm_add; add_norms and the Llama norm are alike to 3%):
//   1024 outputs, 2816 deep, four: 1 row 7.0 -> 6.6, 16 8.3 -> 7.3, 64 8.4 -> 7.9,
//       128 9.5 -> 9.4; 2048 deep: 6.4 -> 6.2, 7.1 -> 6.7, 7.3 -> 7.4, 8.5 -> 8.6
//   2048 outputs, 3584 deep, four: 1 row 8.1 -> 7.8, 16 9.6 -> 8.2, 64 11.2 -> 10.5;
//       2816 deep: 7.3 -> 7.5, 8.7 -> 7.8, 10.0 -> 9.9 (Llama's norm 9.7 -> 9.7);
//       96 rows, two: 2816 deep 11.7 -> 10.5, 4096 14.0 -> 11.8 (four 11.9), 6400
//       19.6 -> 15.5, four 14.6
//   4096 outputs, two: 32 rows, 3584 deep 12.8 -> 11.8, 64 15.0 -> 14.1; 4096 deep
//       14.1 -> 12.4, 15.6 -> 14.8 (four 12.7, 15.3), 96 rows 17.5 -> 16.2; 2816 deep
//       11.5 -> 10.9, 13.1 -> 12.8; 24 rows, 6144 deep two and four alike (-9%),
//       14336 30.4 -> 27.3, four 25.4
//   4096 outputs, up to 16 rows, which memory bounds: 8 rows gain 3% at most,
//       16 with two 4096 deep 1%, 6144 6%, 14336 5%, with four 3 and 8%
//   1280 outputs, whose own tiles of 48 and 80 rows are one round of workgroups:
//       36 rows, 3136 deep 8.2 -> 8.7, 4608 9.7 -> 9.5, 70 and 90 rows 1 to 4% and
//       0 to 2% slower to 6016 deep; 60 and 110 rows gain as beside it
// Five shares or more of 2048 x 4096 lose (16 rows 8.4 with four, 9.3 with eight).
// Of 2900 products of 1 to 128 rows, 768 to 5120 outputs and 2048 to 19456 deep
// three are more than 2% slower by it, 4% at most (70 rows of 768 x 3136).
extern "C" int ll_row_gemm_joined(int N, int M, int K) {
  const int more = ll_row_gemm_shares(N, M, K);
  if (more > 1 || N <= 0 || N > 128 || M < 768 || M > 4096 || M % 4)
    return more;
  int shares = 1;
  if (M <= 2048) {
    if (K >= (M > 1536 && N <= 64 ? 3072 : 2816))
      shares = N > 64 && M > 1024 && K <= 4096 ? 2 : 4;
  } else if (N > 64) {
    shares = K >= 4096 ? 2 : 1;
  } else if (N > 16) {
    shares = K >= 6144 ? 4 : (K >= 3072 ? 2 : 1);
  } else if (N >= 12) {
    shares = K >= 12288 ? 4 : (K >= 6144 ? 2 : 1);
  }
  if (M > 1024 && M < 1408 &&
      ((N > 32 && N <= 48 && K < 4608) || (N > 64 && N <= 96)))
    shares = 1;
  while (shares > 1 &&
         share_blocks(N, M, share_tile(N, M, shares), shares) > 256)
    shares /= 2;
  return shares;
}

extern "C" int ll_rmsnorm_join(void* out, const void* ws, int shares,
                               const void* weight, void* residual, int rows,
                               int width, float eps, void* stream) {
  if (shares < 1 || rows <= 0 || width <= 0 || width % 8 || width > 8192 ||
      ((uintptr_t)out | (uintptr_t)ws | (uintptr_t)weight |
       (uintptr_t)residual) % 16)
    return -2;
#define GO(THREADS)                                                         \
  hipLaunchKernelGGL(rmsnorm_join_kernel<THREADS>, dim3(rows),              \
                     dim3(THREADS), 0, (hipStream_t)stream, (bf16_t*)out,   \
                     (const float*)ws, shares, (const bf16_t*)weight,       \
                     (bf16_t*)residual, width, eps)
  if (width <= 2048) GO(256);
  else if (width <= 4096) GO(512);
  else GO(1024);
#undef GO
  HY_CHECK();
  return 0;
}

// The same product in shares, which a second kernel adds up.
extern "C" int ll_row_gemm_split(void* out, int ld_out, const void* x,
                                 const void* w, void* ws, int shares, int N,
                                 int M, int K, int ldx, void* stream) {
  if (ld_out % 4 || (uintptr_t)out % 8) return -2;
  const int parts =
      ll_row_gemm_parts(x, w, ws, shares, N, M, K, ldx, stream);
  if (parts < 0) return parts;
  hipLaunchKernelGGL(row_gemm_join_kernel,
                     dim3((unsigned)(((size_t)N * (M / 4) + 255) / 256)),
                     dim3(256), 0, (hipStream_t)stream, (bf16_t*)out, ld_out,
                     (const float*)ws, N, M, parts);
  HY_CHECK();
  return 0;
}

// Whether the library's product is the faster one: more than 64 rows read W
// twice, and of the largest matrices the second time from memory.  us, here
// and the library, 72, 96, 128 rows: 32000 x 4096 77, 78, 86 and 103, 101,
// 101; 128256 x 2048 159, 165, 184 and 185, 186, 189; 96000 x 4096 227, 224,
// 245 and 230, 221, 234; 128256 x 4096 304, 298, 325 and 285, 280, 289; 57344
// x 8192 298, 256, 274 and 228, 228, 233.
static bool read_twice(int N, size_t rows, int K) {
  return N > 64 && rows * K > (384u << 20);
}

// Rows of x start ldx numbers apart, those of out ld_out.  0: done, -2: not
// for this kernel.
extern "C" int ll_row_gemm(void* out, int ld_out, const void* x,
                           const void* w, int N, int M, int K, int ldx,
                           int kind, int up, float a, float b, void* stream) {
  if (N <= 0 || N > 128 || M <= 0 || K <= 0 || M % 4 || K % 8 || ldx % 8 ||
      ld_out % 4 || (uintptr_t)x % 16 || (uintptr_t)w % 16 ||
      (uintptr_t)out % (kind == CAPPED ? 16 : 8) || kind < PLAIN ||
      kind > CAPPED)
    return -2;
  const bool gated = kind == SWIGLU || kind == CLAMPED;
  if (read_twice(N, (size_t)M * (gated ? 2 : 1), K)) return -2;
  const RowAct act{kind, up, a, b};
  if (gated)
    return row_gemm_pick(RowGemm<GatedEnd>{
        out, ld_out, (const bf16_t*)x, (const bf16_t*)w, N, M, K, ldx,
        GatedEnd{act}, (hipStream_t)stream});
  return row_gemm_pick(RowGemm<PlainEnd>{
      out, ld_out, (const bf16_t*)x, (const bf16_t*)w, N, M, K, ldx,
      PlainEnd{act}, (hipStream_t)stream});
}

// out1 = x1 W1^T and out2 = gated(x2 W2^T) of N rows, both K deep, as
// ll_row_gemm makes them (kind: SWIGLU or CLAMPED).  0: done, -2: not for this
// kernel.
extern "C" int ll_row_gemm_two(void* out1, int ld_out1, const void* x1,
                               int ldx1, const void* w1, int M1, void* out2,
                               int ld_out2, const void* x2, int ldx2,
                               const void* w2, int M2, int kind, int up,
                               float a, float b, int N, int K, void* stream) {
  auto fits = [&](const void* out, int ld_out, const void* x, int ldx,
                  const void* w, int M, int rows) {
    return M > 0 && M % 4 == 0 && ldx % 8 == 0 && ld_out % 4 == 0 &&
           (uintptr_t)x % 16 == 0 && (uintptr_t)w % 16 == 0 &&
           (uintptr_t)out % 8 == 0 && !read_twice(N, rows, K);
  };
  if (N <= 0 || N > 128 || K <= 0 || K % 8 ||
      (kind != SWIGLU && kind != CLAMPED) ||
      !fits(out1, ld_out1, x1, ldx1, w1, M1, M1) ||
      !fits(out2, ld_out2, x2, ldx2, w2, M2, 2 * M2) ||
      ll_row_gemm_shares(N, M1, K) > 1)
    return -2;
  const RowGemmTwo p{
      {out1, (const bf16_t*)x1, (const bf16_t*)w1, ld_out1, M1, ldx1},
      {out2, (const bf16_t*)x2, (const bf16_t*)w2, ld_out2, M2, ldx2},
      PlainEnd{RowAct{PLAIN, 0, 0.f, 0.f}},
      GatedEnd{RowAct{kind, up, a, b}},
      N,
      K,
      (hipStream_t)stream};
  float both, first, second;
  const int tile = row_gemm_tile(N, M1, K, true, 2ll * M2, &both);
  row_gemm_tile(N, M1, K, false, 0, &first);
  row_gemm_tile(N, 2ll * M2, K, true, 0, &second);
  if ((both - first - second) * K > (N <= 16 ? 5700.f : 4700.f)) return -2;
  switch (tile) {
#define GO(NT, MT, KW, S) \
  case NT * 8 + MT: return row_gemm_two_launch<NT, MT, KW, S>(p);
    ROW_GEMM_TILES(GO)
#undef GO
  }
  return -2;
}

// Whether a product norms its rows itself: every workgroup does all of them, so
// few, and not where workgroups come in rounds (of one row, in several, unless
// its norm is next to nothing).  us, both launches -> this:
//   1 row: 1536 x 1024 5.5 -> 4.9, gate and up of 5632 x 1024 6.9 -> 5.8, 32000 x
//       1024 14.6 -> 13.9, 3072 x 2048 7.0 -> 6.6, gate and up of 11264 x 2048
//       11.7 -> 11.2, 6144 x 4096 13.0 -> 13.7
//   1 row of many outputs: 49152 x 1024 20.4 -> 20.1, 98304 34.6 -> 35.4, 152064
//       49.8 -> 51.0; 49152 x 1536 27.2 -> 27.1, 65536 34.5 -> 35.1, 152064 72.3 ->
//       74.4; 49152 x 2048 34.3 -> 34.2, 98304 63.2 -> 64.0; 152064 x 512 32.2 ->
//       31.2; between rounds 22528 x 2048 18.6 -> 19.4
//   2 rows: 5.8 -> 4.9, 7.0 -> 6.2, 14.4 -> 14.7, 6.9 -> 7.3, 11.8 -> 11.6
//   4 rows: 5.8 -> 5.3, 7.1 -> 6.5, 14.6 -> 15.2; 6: 6.0 -> 5.8, 7.3 -> 7.8
// rows: of W.  ops.norms_rows is the same rule.
static bool norm_gains(int N, int rows, int K) {
  if (N == 1) return K <= 512 || (K <= 2048 && rows <= 48 * 1024);
  return N <= 4 && K <= 1024 && rows <= 16 * 1024;
}

static bool norm_fits(const void* x, const void* residual, const void* sum,
                      const void* weight, int N, int rows, int K) {
  return norm_gains(N, rows, K) && K % 64 == 0 && weight &&
         (uintptr_t)weight % 16 == 0 && (uintptr_t)residual % 16 == 0 &&
         (uintptr_t)sum % 16 == 0 && !residual == !sum &&
         (!sum || (sum != residual && sum != x));
}

// out = act(norm(x) W^T), of x + residual where there is one, which is left in
// ``sum`` (dense rows both).
extern "C" int ll_row_gemm_normed(void* out, int ld_out, const void* x,
                                  const void* w, const void* residual,
                                  void* sum, const void* norm_weight,
                                  float eps, int N, int M, int K, int ldx,
                                  int kind, int up, void* stream) {
  if (N <= 0 || M <= 0 || K <= 0 || M % 4 || ldx % 8 || ld_out % 4 ||
      (uintptr_t)x % 16 || (uintptr_t)w % 16 || (uintptr_t)out % 8 ||
      (kind != PLAIN && kind != SWIGLU) ||
      !norm_fits(x, residual, sum, norm_weight, N,
                 kind == SWIGLU ? 2 * M : M, K))
    return -2;
  const RowNorm norm{(const bf16_t*)residual, (bf16_t*)sum,
                     (const bf16_t*)norm_weight, eps};
  const RowAct act{kind, up, 0.f, 0.f};
  if (kind == SWIGLU)
    return row_gemm_normed(
        RowGemm<GatedEnd>{out, ld_out, (const bf16_t*)x, (const bf16_t*)w, N,
                          M, K, ldx, GatedEnd{act}, (hipStream_t)stream},
        norm);
  return row_gemm_normed(
      RowGemm<PlainEnd>{out, ld_out, (const bf16_t*)x, (const bf16_t*)w, N, M,
                        K, ldx, PlainEnd{act}, (hipStream_t)stream},
      norm);
}

// Queries, keys and values of N rows, rotated, and with caches appended: see
// RotaryEnd.  W holds n_q + 2 n_kv heads of D rows, D a power of two, in that
// order; caches are [page][head][page slot][D].  With norm_weight of normed
// rows, as above.
extern "C" int ll_row_gemm_rotary(
    void* out, const void* x, const void* w, const void* cos_sin,
    const void* positions, void* kcache, void* vcache, const void* slots,
    const void* residual, void* sum, const void* norm_weight, float eps, int N,
    int n_q, int n_kv, int D, int K, int ldx, int page, void* stream) {
  if (N <= 0 || N > 128 || n_q <= 0 || n_kv <= 0 || D < 8 || (D & (D - 1)) ||
      n_q > 1 << 16 || n_kv > 1 << 16 || D > 1 << 10 || K <= 0 || K % 8 ||
      ldx % 8 || page <= 0 || (uintptr_t)x % 16 || (uintptr_t)w % 16 ||
      (uintptr_t)out % 8 || (uintptr_t)cos_sin % 16 ||
      (uintptr_t)kcache % 8 || (uintptr_t)vcache % 8 || !cos_sin ||
      !positions || !kcache != !vcache || (kcache && !slots))
    return -2;
  const int M = (n_q + 2 * n_kv) * D;
  const RowGemm<RotaryEnd> p{
      out, M, (const bf16_t*)x, (const bf16_t*)w, N, M / 2, K, ldx,
      RotaryEnd{(const float*)cos_sin, (const int*)positions,
                (const int*)slots, (bf16_t*)kcache, (bf16_t*)vcache,
                __builtin_ctz(D) - 1, n_q, n_kv, page},
      (hipStream_t)stream};
  if (norm_weight) {
    if (!norm_fits(x, residual, sum, norm_weight, N, M, K)) return -2;
    return row_gemm_normed(p, RowNorm{(const bf16_t*)residual, (bf16_t*)sum,
                                      (const bf16_t*)norm_weight, eps});
  }
  if (read_twice(N, M, K) || ll_row_gemm_shares(N, M, K) > 1) return -2;
  return row_gemm_pick(p);
}

// The same for H pairs of rows and matrices at once, as latent attention needs
// for its heads: out[h] = x[h] W[h]^T, W [H][M][K], or out[h] = x[h] W[h], W
// [H][K][M] (DOWN).  x's and out's heads lie xs and os numbers apart; with w2
// there are two matrices, which lie anywhere.  With a gate, out = bf16(sum)
// sigmoid(gate), the gate of output m of head h being column h M + m of the row.
// A launch and two dependent loads; us, the library's batched product -> here,
// captured, weights from HBM (the first is DOWN, the second joins the heads in
// one row, which was a copy of torch's):
//   64 rows: 32 heads, 128 deep to 512 6.2 -> 4.3, 512 to 128 13.5 -> 3.9;
//       16 heads, 64 to 256 5.2 -> 2.7, 256 to 64 9.0 -> 2.9
//   128 rows: 32 heads, 128 to 512 6.9 -> 5.2, 512 to 128 15.4 -> 4.7
//   4 rows: 16 heads, 128 to 512 4.1 -> 2.9, 512 to 128 14.0 -> 3.3
template <int NT, int MT, int KW, int S, bool GATED, bool DOWN>
__global__ __launch_bounds__(KW * 64, 2) void head_gemm_kernel(
    bf16_t* __restrict__ out, int ld_out, int os,
    const bf16_t* __restrict__ x, int ldx, int xs,
    const bf16_t* __restrict__ w, const bf16_t* __restrict__ w2,
    const bf16_t* __restrict__ gate, int ld_gate, int N, int M, int K) {
  using Tile = RowTile<NT, MT, KW, S>;
  constexpr int OUT = 16 * MT;
  extern __shared__ __align__(1024) char lds[];
  const int h = blockIdx.y, n0 = blockIdx.z * 16 * NT;
  const int m0 = blockIdx.x * OUT;
  const bf16_t* wh = w2 && h ? w2 : w + (size_t)h * M * K;
  const bf16_t* xh = x + (size_t)h * xs;
  // DOWN: M is a multiple of 8, and so are columns
  Tile::template run<DOWN>(
      lds, K, blockIdx.x + h,
      [&](int r) {
        return xh + (size_t)(n0 + r < N ? n0 + r : N - 1) * ldx;
      },
      [&](int r) {
        return DOWN ? wh + (m0 + r < M ? m0 + r : M - 8)
                    : wh + (size_t)(m0 + r < M ? m0 + r : M - 1) * K;
      },
      M);
  Tile::each(OUT / 4, [&](int r, int c) {
    if (n0 + r >= N || m0 + c >= M) return;
    f32x4 v = Tile::sum(lds, r, c);
    if (GATED) {
      const uint2 z = *reinterpret_cast<const uint2*>(
          gate + (size_t)(n0 + r) * ld_gate + (size_t)h * M + m0 + c);
      const float g[4] = {
          __uint_as_float(z.x << 16), __uint_as_float(z.x & 0xffff0000u),
          __uint_as_float(z.y << 16), __uint_as_float(z.y & 0xffff0000u)};
      v = rounded(v);
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] *= sigmoid_f(g[i]);
    }
    *reinterpret_cast<uint2*>(out + (size_t)h * os +
                              (size_t)(n0 + r) * ld_out + m0 + c) =
        make_uint2(to_bf16x2(v[0], v[1]), to_bf16x2(v[2], v[3]));
  });
}

struct HeadGemm {
  bf16_t* out;
  int ld_out, os;
  const bf16_t* x;
  int ldx, xs;
  const bf16_t *w, *w2, *gate;
  int ld_gate, H, N, M, K;
  hipStream_t stream;
};
template <int NT, int MT, int KW, int S, bool GATED, bool DOWN>
static int head_gemm_launch(const HeadGemm& p) {
  auto* kernel = &head_gemm_kernel<NT, MT, KW, S, GATED, DOWN>;
  constexpr int lds = RowTile<NT, MT, KW, S>::LDS;
  static_assert(lds <= 160 * 1024, "LDS of a compute unit");
  static const hipError_t sized = hipFuncSetAttribute(
      reinterpret_cast<const void*>(kernel),
      hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (sized != hipSuccess) return -1;
  hipLaunchKernelGGL(kernel,
                     dim3((p.M + 16 * MT - 1) / (16 * MT), p.H,
                          (p.N + 16 * NT - 1) / (16 * NT)),
                     dim3(KW * 64), lds, p.stream, p.out, p.ld_out, p.os, p.x,
                     p.ldx, p.xs, p.w, p.w2, p.gate, p.ld_gate, p.N, p.M, p.K);
  HY_CHECK();
  return 0;
}
// Waves for the pieces of 64 of the depth that there are; 16 rows a tile, from
// 49 rows on 32 (us, 16 and 32: 64 rows, 32 heads of 128 x 512 4.1 and 3.9, 128
// rows 6.3 and 4.7; 16 heads of 64 x 256 2.9 and 3.1).  64 rows or outputs a
// tile are too few workgroups (4.5).
template <bool GATED>
static int head_gemm_pick(const HeadGemm& p) {
  if (p.K <= 128)
    return p.N <= 48 ? head_gemm_launch<1, 2, 2, 1, GATED, false>(p)
                     : head_gemm_launch<2, 2, 2, 1, GATED, false>(p);
  return p.N <= 48 ? head_gemm_launch<1, 2, 4, 2, GATED, false>(p)
                   : head_gemm_launch<2, 2, 4, 2, GATED, false>(p);
}
// Columns of W: 64 outputs are whole lines of memory (us, 32 and 64: 64 rows, 32
// heads of 128 x 512 5.0 and 4.3, one row 3.8 and 3.4), but too few workgroups
// for small matrices (one row, 16 heads of 64 x 256 2.5 and 2.6); 32 rows a tile
// only past 1024 workgroups (128 rows, 32 heads 5.5 and 5.2; 64 rows 4.3 and 4.4).
template <int KW, int S>
static int head_gemm_down(const HeadGemm& p) {
  if (p.H * (long long)p.M < 8192)
    return head_gemm_launch<1, 2, KW, S, false, true>(p);
  if ((p.N + 15) / 16 * (long long)p.H * ((p.M + 63) / 64) <= 1024)
    return head_gemm_launch<1, 4, KW, S, false, true>(p);
  return head_gemm_launch<2, 4, KW, S, false, true>(p);
}

// w2: null, or the second of two matrices.  0: done, -2: not for this kernel
extern "C" int ll_head_gemm(void* out, int ld_out, int os, const void* x,
                            int ldx, int xs, const void* w, const void* w2,
                            int down, const void* gate, int ld_gate, int H,
                            int N, int M, int K, void* stream) {
  if (H <= 0 || H > 65535 || N <= 0 || N > 128 || M <= 0 || K <= 0 || M % 4 ||
      K % 8 || ldx % 8 || xs % 8 || ld_out % 4 || os % 4 ||
      (uintptr_t)x % 16 || (uintptr_t)w % 16 || (uintptr_t)out % 8 ||
      (w2 && (H != 2 || (uintptr_t)w2 % 16)) || (down && (M % 8 || gate)) ||
      (gate && (ld_gate % 4 || (uintptr_t)gate % 8)))
    return -2;
  const HeadGemm p{(bf16_t*)out,     ld_out,  os, (const bf16_t*)x, ldx, xs,
                   (const bf16_t*)w, (const bf16_t*)w2, (const bf16_t*)gate,
                   ld_gate, H, N, M, K, (hipStream_t)stream};
  if (down) return K <= 128 ? head_gemm_down<2, 1>(p) : head_gemm_down<4, 2>(p);
  return gate ? head_gemm_pick<true>(p) : head_gemm_pick<false>(p);
}
