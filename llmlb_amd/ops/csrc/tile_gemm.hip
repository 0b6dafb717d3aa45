// Products of many rows with a weight matrix, for prompts:
//
//   out[N, M] = act(x[N, K] W[M, K]^T)     bf16, summed in float
//
// Bound by the power of the matrix cores: at 1430 TFLOP/s they are busy 87% of
// the cycles, and the clock is down to 1.2 to 1.7 GHz.  So what counts beside
// the cycles is the energy of a product: 16 x 16 x 32 (registers alone: 2060
// TFLOP/s) and not 32 x 32 x 16 (1790), LDS read without bank conflicts, each
// number once.  16384 rows of 4096 x 14336 take 1296 us without an
// activation; with copies all at once and two stages of 64 KB it was 1582, with
// the ring below and 32 x 32 products 1370.  The library's product takes 1250
// us, but a pass over its results more (swiglu of 16384 x 14336: 263 us).
#include <type_traits>

#include "hybrid/lds_copy.h"
#include "row_act.h"

template <int N, int I = 0, class F>
__device__ __forceinline__ void times(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    times<N, I + 1>(static_cast<F&&>(f));
  }
}

constexpr int DEPTH = 64;  // of a step: a row's part is a line of memory

// Workgroup: tiles of BM rows of x and BN rows of W, by WM x WN waves, one
// after the other.
//
// LDS holds D steps of W's rows and D + 1 of x's.  A step is computed in two
// halves of 32 of its depth; while one is multiplied, the operands of the
// next are read, each into the registers of one that is no longer needed
// (W's, which all of a wave's rows need, have two sets).  The step's only
// barrier stands BP groups of products into its second half: past it every
// wave has read all of the step, whose places the next copies take, and the
// step after is there.  Rows of x are on their way for D - 1/2 steps then,
// those of W for D - 1: small tiles, whose steps are short, need more (48
// tiles of 128 x 128: 0.74 us a step with D = 2, 0.43 with 4).  A tile's first
// steps are fetched while the last of the one before are computed, and its
// results are stored while the next one is.
//
// LDS rows are 8 pieces of 16 bytes; piece c of row r lies at c ^ swizzle(r),
// so that lanes reading one piece of the rows of an operand meet different
// banks.  W's rows enter the matrix cores in an order in which a lane gets 8
// consecutive outputs of each of its rows.
template <int BM, int BN, int WM, int WN, int D, int KIND>
__global__ __launch_bounds__(WM * WN * 64, WM * WN / 4)
void tile_gemm_kernel(bf16_t* __restrict__ out, int ld_out,
                      const bf16_t* __restrict__ x,
                      const bf16_t* __restrict__ w, int N, int M, int K,
                      int ldx, RowAct act, int down, int across) {
  constexpr int NW = WM * WN;
  constexpr int TX = BM / WM / 16, TW = BN / WN / 16;  // 16-row tiles a wave
  constexpr int CX = BM / 8 / NW, CW = BN / 8 / NW;    // copies a wave
  constexpr bool GATED = KIND == SWIGLU || KIND == CLAMPED;
  constexpr int OUT = GATED ? BN / 2 : BN;             // outputs a tile
  constexpr int GROUPS = GATED ? TW / 4 : TW / 2;      // of 32 outputs
  constexpr int STORES = GROUPS * TX;
  constexpr int UX = BM * DEPTH, UW = BN * DEPTH;      // a step's rows
  constexpr int BP = TX < 8 ? 1 : 2;
  static_assert(BM % (8 * NW) == 0 && BN % (8 * NW) == 0, "whole copies");
  static_assert(GROUPS >= 1 && D >= 2, "a wave's outputs, steps ahead");
  extern __shared__ __align__(1024) unsigned short lds[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  // an XCD (every eighth workgroup) has a run of neighbouring tiles
  const int xcd = blockIdx.x & 7, slots = gridDim.x >> 3;
  const long long all = (long long)down * across;
  const int end = (int)(all * (xcd + 1) / 8);
  int tile = (int)(all * xcd / 8) + (blockIdx.x >> 3);
  if (tile >= end) return;

  // first row of x and first output of a tile; tiles go through the outputs
  // by FOUR blocks of rows at a time
  auto place = [&](int t, int& n0, int& m0) {
    constexpr int FOUR = 4;
    const int run = t / (FOUR * across), in = t - run * (FOUR * across);
    const int rows = down - run * FOUR < FOUR ? down - run * FOUR : FOUR;
    n0 = (run * FOUR + in % rows) * BM;
    m0 = in / rows * OUT;
  };
  auto swizzle_x = [](int r) { return r & 7; };
  auto swizzle_w = [](int r) { return (r & 3) | ((r >> 1) & 4); };

  // -- copies: tile and depth they are at, the lane's offsets in bytes
  unsigned xo[CX], wo[CW];
  const bf16_t* xt;
  int xk = 0, wk = 0, x_tile = tile, w_tile = tile, to_x = 0, to_w = 0;
  auto aim_x = [&] {
    int n0, m0;
    place(x_tile, n0, m0);
    xt = x + (size_t)n0 * ldx;
    const int last = N - 1 - n0;
#pragma unroll
    for (int i = 0; i < CX; ++i) {
      const int r = (wave * CX + i) * 8 + (lane >> 3);
      const int c = ((lane & 7) ^ swizzle_x(r)) * 8;
      xo[i] = ((unsigned)(r < last ? r : last) * (unsigned)ldx + c) * 2;
    }
  };
  auto aim_w = [&] {
    int n0, m0;
    place(w_tile, n0, m0);
#pragma unroll
    for (int i = 0; i < CW; ++i) {
      const int r = (wave * CW + i) * 8 + (lane >> 3);
      const int c = ((lane & 7) ^ swizzle_w(r)) * 8;
      // with gate and up, 32 rows of the one and 32 of the other in turn
      const int m = m0 + (GATED ? (r >> 6) * 32 + (r & 31) : r);
      const int row =
          (m < M ? m : M - 1) + (GATED && (r & 32) ? act.up : 0);
      wo[i] = ((unsigned)row * (unsigned)K + c) * 2;
    }
  };
  auto next_x = [](int u) { return u == D ? 0 : u + 1; };
  auto next_w = [](int u) { return u == D - 1 ? 0 : u + 1; };
  const unsigned base = lds_byte(lds);
  auto copy_x = [&](int i) {
    copy_to_lds(xt + xk, xo[i], base + to_x * UX * 2 + (wave * CX + i) * 1024);
  };
  auto copy_w = [&](int i) {
    copy_to_lds(w + wk, wo[i],
                base + ((D + 1) * UX + to_w * UW) * 2 +
                    (wave * CW + i) * 1024);
  };
  // past the last tile its beginning is copied again: every step has as
  // many copies
  auto step_x = [&] {
    to_x = next_x(to_x);
    if ((xk += DEPTH) < K) return;
    xk = 0;
    if (x_tile + slots < end) {
      x_tile += slots;
      aim_x();
    }
  };
  auto step_w = [&] {
    to_w = next_w(to_w);
    if ((wk += DEPTH) < K) return;
    wk = 0;
    if (w_tile + slots < end) {
      w_tile += slots;
      aim_w();
    }
  };
  aim_x();
  aim_w();
#pragma unroll
  for (int s = 0; s < D; ++s) {
#pragma unroll
    for (int i = 0; i < CX; ++i) copy_x(i);
    step_x();
#pragma unroll
    for (int i = 0; i < CW; ++i) copy_w(i);
    step_w();
  }

  // -- operands and sums
  const int wm = wave / WN * (BM / WM), wn = wave % WN * (BN / WN);
  const int l = lane & 15, g = lane >> 4;
  const int rx = wm + l, rw = wn + 8 * (l >> 2) + (l & 3);
  const int sx = swizzle_x(rx), sw = swizzle_w(rw);
  u32x4 fx[TX], fw[2][TW];
  f32x4 acc[TX][TW];
  int ux = 0, uw = 0;  // where the step lies
  auto at_x = [&](int half) {
    return lds + ux * UX + rx * DEPTH + ((half * 4 + g) ^ sx) * 8;
  };
  auto at_w = [&](int half) {
    return lds + (D + 1) * UX + uw * UW + rw * DEPTH +
           ((half * 4 + g) ^ sw) * 8;
  };
  auto read_x = [&](const unsigned short* p, int i) {
    fx[i] = *reinterpret_cast<const u32x4*>(p + i * 16 * DEPTH);
  };
  auto read_w = [&](int set, const unsigned short* p, int i) {
    fw[set][i] = *reinterpret_cast<const u32x4*>(
        p + ((i >> 1) * 32 + (i & 1) * 4) * DEPTH);
  };
  // The products of half H of the step; the order alternates, so that one
  // operand stays from each to the next.
  auto half = [&](auto H, auto&& barrier) {
    constexpr int h = H, first = h ? BP : 0;  // where the next reads begin
    constexpr int C = h ? CW : CX, PER = (C + TX - first - 1) / (TX - first);
    const unsigned short *px = at_x(h), *nx, *nw;
    if (!h) nx = at_x(1), nw = at_w(1);
    times<TX>([&](auto IA) {
      constexpr int a = IA;
      if constexpr (h && a == BP) {
        barrier();
        nx = at_x(0), nw = at_w(0);
      }
      times<TW>([&](auto IB) {
        constexpr int i = IB, b = a % 2 ? TW - 1 - i : i;
        // W's reads: every second product, or where groups are few all
        constexpr int LEFT = (TW + TX - first - 1) / (TX - first);
        constexpr int RW = LEFT > TW / 2 ? LEFT : TW / 2;
        constexpr int IS = RW > TW / 2 ? i : (i % 2 ? i / 2 : RW);
        acc[a][b] = mfma(fw[h][b], fx[a], acc[a][b]);
        if constexpr (i == 0 && a == 0) read_x(px, TX - 1);
        if constexpr (i == 0 && a > first) read_x(nx, a - 1);
        if constexpr (h && a == BP && i < BP) read_x(nx, i);
        if constexpr (a >= first && IS < RW && (a - first) * RW + IS < TW)
          read_w(h ^ 1, nw, (a - first) * RW + IS);
        if constexpr (a >= first && i == 2 % TW)
          times<PER>([&](auto IC) {
            constexpr int c = (a - first) * PER + IC;
            if constexpr (c < C) {
              if constexpr (h) copy_w(c);
              else copy_x(c);
            }
          });
        __builtin_amdgcn_sched_barrier(0);
      });
    });
  };
  constexpr std::integral_constant<int, 0> H0{};
  constexpr std::integral_constant<int, 1> H1{};

  bool stored = false;  // STORES of each wave's may be under way
  wait_barrier<(D - 1) * (CX + CW)>();
#pragma unroll
  for (int b = 0; b < TW; ++b) read_w(0, at_w(0), b);
#pragma unroll
  for (int a = 0; a < TX - 1; ++a) read_x(at_x(0), a);
  for (;;) {
#pragma unroll
    for (int a = 0; a < TX; ++a)
#pragma unroll
      for (int b = 0; b < TW; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
    int s = 0;
    do {
      half(H0, [] {});
      step_x();
      half(H1, [&] {
        // all but the copies of the steps past the next one, and what the
        // tile before stored behind the next one's
        constexpr int COPIES = (D - 2) * (CX + CW) + CX;
        if (s < (D - 1) * DEPTH && stored) wait_barrier<COPIES + STORES>();
        else wait_barrier<COPIES>();
        ux = next_x(ux);
        uw = next_w(uw);
      });
      step_w();
    } while ((s += DEPTH) < K);

    int n0, m0;
    place(tile, n0, m0);
    // edges store less, and the wait is for all of it
    stored = n0 + BM <= N && m0 + OUT <= M;
    RowAct as = act;
    as.kind = KIND;
    times<TX>([&](auto IA) {
      constexpr int a = IA;
      const int n = n0 + wm + a * 16 + l;
      bf16_t* row = out + (size_t)n * ld_out;
      times<GROUPS>([&](auto IB) {
        constexpr int b = GATED ? 4 * IB : 2 * IB;
        const int m = m0 + (GATED ? wn / 2 : wn) + IB * 32 + g * 8;
        unsigned p[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float v[2];
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            const int e = 2 * i + j;
            const float z = to_f(from_f<bf16_t>(acc[a][b + e / 4][e % 4]));
            if constexpr (GATED)
              v[j] = row_gate(
                  as, z, to_f(from_f<bf16_t>(acc[a][b + 2 + e / 4][e % 4])));
            else
              v[j] = row_act(as, z);
          }
          p[i] = to_bf16x2(v[0], v[1]);
        }
        if (n < N && m < M)
          *reinterpret_cast<u32x4*>(row + m) = u32x4{p[0], p[1], p[2], p[3]};
      });
    });
    tile += slots;
    if (tile >= end) break;
  }
  // no copy is under way when the workgroup's LDS is given back
  wait_barrier<0>();
}

struct TileGemm {
  bf16_t* out;
  int ld_out;
  const bf16_t *x, *w;
  int N, M, K, ldx;
  RowAct act;
  hipStream_t stream;
};

template <int BM, int BN, int WM, int WN, int D, int KIND>
static int tile_gemm_launch(const TileGemm& p) {
  auto* kernel = &tile_gemm_kernel<BM, BN, WM, WN, D, KIND>;
  constexpr int lds = ((D + 1) * BM + D * BN) * DEPTH * 2;
  static_assert(lds <= 160 * 1024, "LDS of a compute unit");
  static const hipError_t sized = hipFuncSetAttribute(
      reinterpret_cast<const void*>(kernel),
      hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (sized != hipSuccess) return -1;
  constexpr int OUT = KIND == SWIGLU || KIND == CLAMPED ? BN / 2 : BN;
  const int down = (p.N + BM - 1) / BM, across = (p.M + OUT - 1) / OUT;
  const long long per = ((long long)down * across + 7) / 8;
  if (per > 1 << 26) return -2;
  const int slots = per < 32 ? (int)per : 32;
  hipLaunchKernelGGL(kernel, dim3(8 * slots), dim3(WM * WN * 64), lds,
                     p.stream, p.out, p.ld_out, p.x, p.w, p.N, p.M, p.K,
                     p.ldx, p.act, down, across);
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
//    2816 x 1024 18 -> 11; 1355: 5632 x 2048 79 -> 65, 14336 x 4096 291 -> 275;
//    16384: 2816 x 1024 233 -> 160, 14336 x 4096 2891 -> 2691 (1430 TFLOP/s).
//    gelu 16384: 7168 x 2048 440 -> 374, 19456 x 4096 2025 -> 1902.  clamped
//    16384: 4352 x 2048 547 -> 449, 11904 x 4096 2405 -> 2267.  squared relu
//    333: 6912 x 2048 29 -> 20; 1355: 50 -> 44, 18432 x 4096 193 -> 183
//  * not for few tiles of some depth, which the library takes in shares: 333:
//    2048 x 2048 10.7 -> 12.9, 2048 x 7168 30 -> 43, 1024 x 3328 13 -> 18
//  * outputs that are no whole tiles of 256: 333: 8224 x 2048 25 -> 21; 1355:
//    3216 x 1024 17.5 -> 13.2, 8224 x 2048 56 -> 52; 8200: 1808 x 1024 53 -> 34,
//    16448 x 4096 922 -> 834; 16384: 3600 x 2048 236 -> 200, 6416 x 2048 378 ->
//    338, but 16512 x 4096 1557 -> 1604
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
  if (kind != PLAIN || K <= 1024) return 1;
  if (rows % 256) return K < 3072 || N < 12288;
  if (K < 3072) return N < 4096;
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
