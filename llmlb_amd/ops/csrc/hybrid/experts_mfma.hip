// Matrix-core products of tokens with their experts' matrices, bf16: for
// every (token, choice) pair p = token * top + choice
//   out[p] = act(w[expert] in[p / div]),  act(z) = max(z, 0)^2 or none.
//
//  * expert_tile_kernel  prompts: tiles of an expert's list (experts.h)
//    against tiles of its matrix, both copied to LDS directly
//  * expert_product_kernel  the same by tile_product.h, where there are tiles
//    of 192 x 256 for the compute units
//  * expert_few_kernel   few pairs: a workgroup finds its expert's pairs
//    among all choices and streams some rows of its matrix once
//
// Both compute (w in^T) tiles: a lane holds outputs 4g..4g+3 (g = lane/16)
// of pair n = lane % 16.
#include "few_experts.h"
#include "tile_product.h"

// LDS rows are P pieces of 16 bytes; piece c of row r lies at
// c ^ swizzle(r), so that lanes reading one piece of the rows of an
// operand meet different banks.
template <int P>
__device__ __forceinline__ int swizzle_in(int r) {
  return P == 8 ? r & 7 : (r >> 1) & 3;
}
template <int P>
__device__ __forceinline__ int swizzle_w(int r) {
  return P == 8 ? (r & 3) | ((r >> 1) & 4) : ((r >> 1) & 1) | ((r >> 2) & 2);
}

// Workgroup: BM pairs x BN outputs, WM x WN waves; BK of the depth a step.
// LDS holds ST steps, the copies of a step start ST - 1 steps ahead.
// Within 32 outputs of a wave, row g * 8 + t * 4 + i of the matrix is row
// 4 g + i of MFMA tile t: a lane then holds 8 consecutive outputs of each
// of its pairs.
// WHOLE: the depth is whole steps, and all rows lie within 4 GB of each
// other: copies are at one scalar address and a lane's own offset, which
// takes no vector instruction a step (63 a wave before, a quarter of the
// time).  16384 tokens with 4 of 16 experts, us: 4096 to 1280 wide 668 ->
// 612, back 752 -> 687; 2048 to 512 169 -> 153, back 174 -> 166.  A
// compute unit takes in 42 GB/s then; copies alone reach 115.
// Results are stored by way of the caches: the next kernel reads them, and
// past the caches (nontemporal) they wait for what these write back (2048
// wide in a model: back 222 -> 193).
template <int BM, int BN, int WM, int WN, int BK, int ST, bool WHOLE>
__global__ __launch_bounds__(WM * WN * 64, WM * WN == 4 ? 2 : 1)
void expert_tile_kernel(
    bf16_t* __restrict__ out, const bf16_t* __restrict__ in,
    const bf16_t* __restrict__ w, const int* __restrict__ counts,
    const int* __restrict__ pairs, int E, int N, int K, int div, int act,
    int n_tok, int n_blocks) {
  constexpr int NW = WM * WN, TM = BM / WM / 16, TN = BN / WN / 64;
  constexpr int P = BK / 8, RC = 64 / P;  // pieces of a row, rows of a copy
  constexpr int CA = BM / RC / NW, CB = BN / RC / NW;  // copies a wave
  constexpr int C = CA + CB, SIZE = (BM + BN) * BK;
  __shared__ __align__(1024) unsigned short lds[ST * SIZE];
  __shared__ ExpertTiles<BM> tiles;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int n = lane & 15, g = lane >> 4;
  if (wave == 0) tiles.count(counts, E);
  __syncthreads();
  // neighbouring tiles on one XCD, which gets every eighth workgroup
  const int whole = tiles.whole[E - 1] * n_blocks;
  const int rest = tiles.rest[E - 1] * n_blocks;
  const int per = (whole + 7) / 8, rest_per = (rest + 7) / 8;
  const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3;
  const bool is_rest = local >= per;
  const int id = is_rest ? xcd * rest_per + local - per : xcd * per + local;
  if (is_rest ? local - per >= rest_per || id >= rest : id >= whole) return;
  const ExpertTile t = tiles.get(counts, E, id / n_blocks, is_rest);
  const int n0 = id % n_blocks * BN;
  const int* list = pairs + (size_t)t.expert * n_tok + t.first;
  const bf16_t* we = w + (size_t)t.expert * N * K;

  const bf16_t *ap[WHOLE ? 1 : CA], *bp[WHOLE ? 1 : CB];
  int ac[WHOLE ? 1 : CA], bc[WHOLE ? 1 : CB];  // the lane's column in a row
  unsigned ao[WHOLE ? CA : 1], bo[WHOLE ? CB : 1];
#pragma unroll
  for (int i = 0; i < CA; ++i) {
    const int r = (wave * CA + i) * RC + lane / P;
    const int c = ((lane % P) ^ swizzle_in<P>(r)) * 8;
    const size_t at =
        (size_t)(list[r < t.n ? r : t.n - 1] / div) * K + c;
    if constexpr (WHOLE) {
      ao[i] = (unsigned)at * 2;
    } else {
      ac[i] = c;
      ap[i] = in + at;
    }
  }
#pragma unroll
  for (int i = 0; i < CB; ++i) {
    const int r = (wave * CB + i) * RC + lane / P;
    const int c = ((lane % P) ^ swizzle_w<P>(r)) * 8;
    const size_t at = (size_t)(n0 + r < N ? n0 + r : N - 1) * K + c;
    if constexpr (WHOLE) {
      bo[i] = (unsigned)at * 2;
    } else {
      bc[i] = c;
      bp[i] = we + at;
    }
  }
  const unsigned base = lds_byte(lds);
  const bf16_t* zero = reinterpret_cast<const bf16_t*>(zero_piece);
  // past the depth something is copied as well: every step has as many
  // copies
  auto fetch = [&](int k0, int place) {
    const unsigned to = base + place * SIZE * 2;
    if constexpr (WHOLE) {
      const int k = k0 < K ? k0 : 0;
#pragma unroll
      for (int i = 0; i < CA; ++i)
        copy_to_lds(in + k, ao[i], to + (wave * CA + i) * 1024);
#pragma unroll
      for (int i = 0; i < CB; ++i)
        copy_to_lds(we + k, bo[i],
                    to + BM * BK * 2 + (wave * CB + i) * 1024);
    } else {
#pragma unroll
      for (int i = 0; i < CA; ++i)
        copy_to_lds(k0 + ac[i] < K ? ap[i] + k0 : zero,
                    to + (wave * CA + i) * 1024);
#pragma unroll
      for (int i = 0; i < CB; ++i)
        copy_to_lds(k0 + bc[i] < K ? bp[i] + k0 : zero,
                    to + BM * BK * 2 + (wave * CB + i) * 1024);
    }
  };
  const int wm = wave / WN * (BM / WM), wn = wave % WN * (BN / WN);
  f32x4 acc[TM][TN][4];
#pragma unroll
  for (int a = 0; a < TM; ++a)
#pragma unroll
    for (int b = 0; b < TN; ++b)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[a][b][i] = f32x4{0.f, 0.f, 0.f, 0.f};

  // the lane's numbers of a place, before the row tile and MFMA step
  const int ra = wm + n, rb = wn + (n >> 2) * 8 + (n & 3);
#pragma unroll
  for (int s = 0; s < ST - 1; ++s) fetch(s * BK, s);
  // One barrier a step: past it, every wave has read the place of the step
  // before, which the newest copies take.
  int place = 0, free = ST - 1;
  for (int k0 = 0; k0 < K; k0 += BK) {
    wait_barrier<(ST - 2) * C>();
    fetch(k0 + (ST - 1) * BK, free);
    __builtin_amdgcn_sched_barrier(0);
    const unsigned short* st = lds + place * SIZE;
    free = place;
    place = place + 1 == ST ? 0 : place + 1;
    if (wm >= t.n || n0 + wn >= N) continue;  // nothing for this wave
#pragma unroll
    for (int s = 0; s < BK / 32; ++s) {
      const unsigned short* pa =
          st + ra * BK + ((s * 4 + g) ^ swizzle_in<P>(ra)) * 8;
      const unsigned short* pb =
          st + BM * BK + rb * BK + ((s * 4 + g) ^ swizzle_w<P>(rb)) * 8;
      // the pieces of rows 4 further lie elsewhere where P is 8
      const unsigned short* pb4 =
          st + BM * BK + (rb + 4) * BK +
          ((s * 4 + g) ^ swizzle_w<P>(rb + 4)) * 8;
      u32x4 af[TM], bf[TN][4];
#pragma unroll
      for (int a = 0; a < TM; ++a)
        af[a] = *reinterpret_cast<const u32x4*>(pa + a * 16 * BK);
#pragma unroll
      for (int b = 0; b < TN; ++b)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          bf[b][i] = *reinterpret_cast<const u32x4*>(
              (i & 1 ? pb4 : pb) + (b * 64 + (i >> 1) * 32) * BK);
#pragma unroll
      for (int a = 0; a < TM; ++a)
#pragma unroll
        for (int b = 0; b < TN; ++b)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            acc[a][b][i] = mfma(bf[b][i], af[a], acc[a][b][i]);
    }
  }
  // no copy is under way when the workgroup's LDS is given back
  wait_barrier<0>();
#pragma unroll
  for (int a = 0; a < TM; ++a) {
    const int r = wm + a * 16 + n;
    if (r >= t.n) continue;
    bf16_t* dst = out + (size_t)list[r] * N;
#pragma unroll
    for (int b = 0; b < TN; ++b) {
      const int c = n0 + wn + b * 64 + g * 8;
      unsigned x[8];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        f32x4 v = acc[a][b][i];
        if (act) {
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            v[j] = fmaxf(v[j], 0.f);
            v[j] *= v[j];
          }
        }
        x[2 * i] = to_bf16x2(v[0], v[1]);
        x[2 * i + 1] = to_bf16x2(v[2], v[3]);
      }
#pragma unroll
      for (int i = 0; i < 2; ++i)
        if (c + i * 32 < N)
          *reinterpret_cast<u32x4*>(dst + c + i * 32) =
              u32x4{x[4 * i], x[4 * i + 1], x[4 * i + 2], x[4 * i + 3]};
    }
  }
}

// The rows of experts' lists, for tile_product.  AHEAD: a tile's part of its
// list is in LDS before the copies of its rows begin; asked for there, it would
// have to wait for all copies under way.  It is on its way for a step at least,
// so tiles have two or more.
template <int BM, int BN, bool AHEAD>
struct ListRows {
  // of tiles that are fetched, copied, computed and stored at a time
  static constexpr int PARTS = 8;
  const bf16_t *in, *w_;
  const int *counts, *pairs;
  int E, N, K, div, n_tok, n_blocks;
  const ExpertTiles<BM>* found;
  int* parts;  // [PARTS][BM]
  struct At {
    ExpertTile t;
    const int* list;
    int m0;
  };
  __device__ __forceinline__ long long tiles() const {
    return (long long)(found->whole[E - 1] + found->rest[E - 1]) * n_blocks;
  }
  // a workgroup's tiles are as far apart as an XCD has workgroups
  __device__ __forceinline__ int* part(int i) const {
    return parts + i / (int)(gridDim.x >> 3) % PARTS * BM;
  }
  __device__ __forceinline__ ExpertTile tile(int i) const {
    const int whole = found->whole[E - 1], j = i / n_blocks;
    return found->get(counts, E, j < whole ? j : j - whole, j >= whole);
  }
  __device__ __forceinline__ At at(int i) const {
    const ExpertTile t = tile(i);
    return At{t,
              AHEAD ? part(i) : pairs + (size_t)t.expert * n_tok + t.first,
              i % n_blocks * BN};
  }
  // 64 numbers a wave; past the end the last one again
  __device__ __forceinline__ void fetch(int i) const {
    static_assert(BM % WAVE == 0, "whole waves");
    if (!AHEAD) return;
    const int at = __builtin_amdgcn_readfirstlane(threadIdx.x & ~63);
    if (at >= BM) return;
    const ExpertTile t = tile(i);
    const int r = threadIdx.x < t.n ? threadIdx.x : t.n - 1;
    copy_words_to_lds(pairs + (size_t)t.expert * n_tok + t.first + r,
                      lds_byte(part(i) + at));
  }
  __device__ __forceinline__ void fetched() const {
    if (AHEAD) wait_barrier<0>();
  }
  __device__ __forceinline__ const bf16_t* x(const At&) const { return in; }
  __device__ __forceinline__ const bf16_t* w(const At& a) const {
    return w_ + (size_t)a.t.expert * N * K;
  }
  __device__ __forceinline__ unsigned x_offset(const At& a, int r) const {
    const int i = AHEAD || r < a.t.n ? r : a.t.n - 1;
    return (unsigned)(a.list[i] / div) * (unsigned)K;
  }
  __device__ __forceinline__ long long row(const At& a, int r) const {
    return r < a.t.n ? a.list[r] : -1;
  }
  __device__ __forceinline__ bool whole(const At& a) const {
    return a.t.n == BM;
  }
};

// Bound by the matrix cores' power and, for shallow products, by what they
// write: 16384 tokens with 4 of 16 experts, us, the best of the tiles above
// -> here: 1024 to 256 wide 60 -> 46, back 61 -> 52; 2048 to 512 162 -> 117,
// back 211 -> 176.  Of that, lists asked for from memory and results stored at
// once -> lists in LDS -> results held, sides in turn: 2048 to 512 120 -> 118 ->
// 117, back 178 -> 180 -> 175; 4096 to 1280 555 -> 545 -> 538, back 677 -> 666 ->
// 645; 1024 to 256 46 -> 45 -> 46, back 54 -> 52 -> 52; back 128 deep to 2048 61.7 ->
// 57 -> 59; 4096 tokens back 2048 to 512 46 -> 46 -> 43.  One step deep both lose:
// 64 to 2048 73 -> 81.  Without any stores the way back of 512 deep takes 116 us;
// they alone take 41.  256 x 256 leaves no LDS for the tiles' numbers; 256 x 128 and
// 128 x 256 read more (2048 to 512: 146, 156).
template <int BM, int BN, int WM, int WN, int D, int KIND, bool DEEP>
__global__ __launch_bounds__(WM * WN * 64, WM * WN / 4)
void expert_product_kernel(bf16_t* __restrict__ out,
                           ListRows<BM, BN, DEEP> rows) {
  __shared__ ExpertTiles<BM> tiles;
  if (threadIdx.x < WAVE) tiles.count(rows.counts, rows.E);
  __syncthreads();
  __shared__ int parts[DEEP ? rows.PARTS * BM : 1];
  rows.found = &tiles;
  rows.parts = parts;
  tile_product<BM, BN, WM, WN, D, KIND, false, DEEP>(
      rows, out, rows.N, rows.N, rows.K, RowAct{KIND, 0, 0.f, 0.f});
}

struct ExpertProduct {
  bf16_t* out;
  const bf16_t *in, *w;
  const int *counts, *pairs;
  int E, N, K, div, n_tok, n_pairs;
  hipStream_t stream;
};
template <int BM, int BN, int WM, int WN, int D, int KIND, bool DEEP>
static int expert_product(const ExpertProduct& p) {
  auto* kernel = &expert_product_kernel<BM, BN, WM, WN, D, KIND, DEEP>;
  constexpr int lds = ((D + 1) * BM + D * BN) * DEPTH * 2;
  static_assert(lds + sizeof(ExpertTiles<BM>) +
                        ListRows<BM, BN, DEEP>::PARTS * BM * 4 <= 160 * 1024,
                "LDS of a compute unit");
  static const hipError_t sized = hipFuncSetAttribute(
      reinterpret_cast<const void*>(kernel),
      hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (sized != hipSuccess) return -1;
  const int nb = (p.N + BN - 1) / BN;
  // as many tiles as there can be, and a workgroup a compute unit at most
  const long long most =
      ((long long)p.n_pairs / BM + (p.E < p.n_pairs ? p.E : p.n_pairs)) * nb;
  if (most >= 1ll << 27) return -2;
  const long long per = (most + 7) / 8;
  const ListRows<BM, BN, DEEP> rows{p.in, p.w, p.counts, p.pairs, p.E, p.N,
                              p.K,  p.div, p.n_tok, nb, nullptr, nullptr};
  hipLaunchKernelGGL(kernel, dim3(8 * (unsigned)(per < 32 ? per : 32)),
                     dim3(WM * WN * 64), lds, p.stream, p.out, rows);
  HY_CHECK();
  return 0;
}

template <int MT>
__global__ __launch_bounds__(FEW_KW * 64, 2) void expert_few_kernel(
    FewExperts a) {
  extern __shared__ __align__(1024) char lds[];
  __shared__ FewList list;
  few_block<MT>(a, blockIdx.x, blockIdx.y, lds, list);
}

extern "C" {

// tile: 0 128 x 128, 1 256 x 256, 2 128 x 256, 3 192 x 256 by tile_product
// (pairs x outputs)
int hy_expert_tiles(void* out, const void* in, const void* w,
                    const void* counts, const void* pairs, int E, int N,
                    int K, int div, int act, int n_tok, int n_pairs,
                    int tile, void* stream) {
  if (E <= 0 || E > EXPERTS_MAX || N <= 0 || K <= 0 || N % 8 || K % 8 ||
      div <= 0)
    return -2;
  if (n_tok <= 0 || n_pairs <= 0) return 0;
#define RUN(BM, BN, WM, WN, BK, ST, WHOLE)                                   \
  hipLaunchKernelGGL((expert_tile_kernel<BM, BN, WM, WN, BK, ST, WHOLE>),    \
                     dim3((unsigned)groups * 8), dim3(WM * WN * 64), 0,      \
                     (hipStream_t)stream, (bf16_t*)out, (const bf16_t*)in,   \
                     (const bf16_t*)w, (const int*)counts,                   \
                     (const int*)pairs, E, N, K, div, act, n_tok, (int)nb)
#define GO(BM, BN, WM, WN, BK, ST)                                           \
  do {                                                                       \
    const long long nb = (N + BN - 1) / BN;                                  \
    const long long groups = (n_pairs / BM * nb + 7) / 8 +                   \
                             ((E < n_pairs ? E : n_pairs) * nb + 7) / 8;     \
    if (groups >= (1ll << 27)) return -2;                                    \
    if (K % BK == 0 && near) RUN(BM, BN, WM, WN, BK, ST, true);              \
    else RUN(BM, BN, WM, WN, BK, ST, false);                                 \
  } while (0)
  const long long rows = n_pairs / div + 1 > N ? n_pairs / div + 1 : N;
  const bool near = rows * K * 2 < (1ll << 32);
  switch (tile) {
    case 0: GO(128, 128, 2, 2, 64, 2); break;
    case 1: GO(256, 256, 4, 4, 64, 2); break;
    case 2: GO(128, 256, 2, 4, 32, 3); break;
    case 3:
      if (K % DEPTH == 0 && near) {
        const ExpertProduct p{(bf16_t*)out, (const bf16_t*)in,
                              (const bf16_t*)w, (const int*)counts,
                              (const int*)pairs, E, N, K, div, n_tok,
                              n_pairs, (hipStream_t)stream};
        // a tile of one step has none to fetch and to store in
        if (K == DEPTH)
          return act ? expert_product<192, 256, 2, 4, 2, RELU2, false>(p)
                     : expert_product<192, 256, 2, 4, 2, PLAIN, false>(p);
        return act ? expert_product<192, 256, 2, 4, 2, RELU2, true>(p)
                   : expert_product<192, 256, 2, 4, 2, PLAIN, true>(p);
      }
      GO(256, 256, 4, 4, 64, 2);
      break;
    default: return -2;
  }
#undef RUN
#undef GO
  HY_CHECK();
  return 0;
}

// Outputs a tile of hy_expert_few over 16, by what a compute unit takes in as
// for other products of few rows: rounds of 256 tiles of the experts that are
// likely used, times a tile's rows.  32, but 16 for small matrices and 80 for
// deep ones.  us, 32 outputs -> these, 61 tokens: 1024 to 256 wide 5.4 -> 4.9,
// 4096 to 1280 32.2 -> 29.4, 300 tokens 90 -> 62; 1280 deep 80 outputs lost (81.6
// -> 90.4).  16 are not for many experts, whose idle workgroups they double (one
// token, 64 of 2048 to 512 9.0 -> 9.8); of 80 a compute unit has one workgroup,
// which with 64 pairs a tile waits for every piece of the depth (128 tokens, 8 of
// 2048 to 4096 53.7 -> 58.5), and the last may be mostly empty (300 tokens, 64 of
// 2048 to 512 30.0 -> 32.9).
int hy_expert_few_tile(int E, int N, int K, int n_pairs) {
  const float used = E * (1.f - powf(1.f - 1.f / E, (float)n_pairs));
  const int each = (int)(n_pairs / used + 15.f) / 16;
  auto takes = [&](int mt) {
    const float tiles = (float)((N + 16 * mt - 1) / (16 * mt)) * used;
    return ceilf(tiles / 256.f) * ((each < 4 ? each : 4) + mt);
  };
  int mt = 2;
  if (K >= 1024 && E * (long long)N <= 8192 && takes(1) < 0.95f * takes(2))
    mt = 1;
  const float whole = (float)N / ((N + 79) / 80 * 80);
  const float waits = each > 2 ? 1.4f : 1.f;
  if (K >= 2048 && takes(5) * waits < 0.85f * whole * takes(mt)) mt = 5;
  return mt;
}

// tile: 1, 2 or 5 times 16 outputs; -1: the choice above
int hy_expert_few(void* out, const void* in, const void* w, const void* index,
                  int E, int N, int K, int div, int act, int n_pairs, int tile,
                  void* stream) {
  const FewExperts a{(bf16_t*)out, (const bf16_t*)in, (const bf16_t*)w,
                     (const int*)index, E, N, K, div, act, n_pairs};
  if (!few_ok(a)) return -2;
  if (n_pairs <= 0) return 0;
#define GO(MT)                                                               \
  do {                                                                       \
    static_assert(FEW_LDS<MT> + sizeof(FewList) <= 160 * 1024,               \
                  "LDS of a compute unit");                                  \
    static const hipError_t sized = hipFuncSetAttribute(                     \
        reinterpret_cast<const void*>(expert_few_kernel<MT>),                \
        hipFuncAttributeMaxDynamicSharedMemorySize, FEW_LDS<MT>);            \
    if (sized != hipSuccess) return -1;                                      \
    hipLaunchKernelGGL(expert_few_kernel<MT>,                                \
                       dim3((N + 16 * MT - 1) / (16 * MT), E),               \
                       dim3(FEW_KW * 64), FEW_LDS<MT>, (hipStream_t)stream,  \
                       a);                                                   \
  } while (0)
  switch (tile < 0 ? hy_expert_few_tile(E, N, K, n_pairs) : tile) {
    case 1: GO(1); break;
    case 2: GO(2); break;
    case 5: GO(5); break;
    default: return -2;
  }
#undef GO
  HY_CHECK();
  return 0;
}

}  // extern "C"
