// Products of few (token, choice) pairs with their experts' matrices.
#pragma once
#include "experts.h"
#include "row_tile.h"

// Few pairs: workgroup (expert, 16 MT outputs), tiles of up to 64 of the
// expert's pairs as in row_tile.h.  Bound by reading the matrices: both
// products of 16 experts of 4096 x 1280 took 105 us for 64 tokens with
// operands loaded straight into registers, 67 (5.0 TB/s) this way; 8 tokens
// 88 -> 60, 16 experts of 1024 x 256 13.1 -> 10.5.  hy_expert_few_tile
// has the outputs a tile.
#define FEW_PAIRS 2048  // most that fit a workgroup's list
// 16 NT pairs by 16 MT outputs; pieces of the depth on their way so that every
// NT fits the LDS of the first
#define FEW_KW 4
template <int NT, int MT>
using FewTile =
    RowTile<NT, MT, FEW_KW, NT == 1 ? 3 : (NT == 2 ? 2 : 1)>;
template <int MT>
constexpr int FEW_LDS = FewTile<1, MT>::LDS;

struct FewExperts {
  bf16_t* out;       // [pairs][N]
  const bf16_t* in;  // [pairs / div][K]
  const bf16_t* w;   // [E][N][K]
  const int* index;  // [pairs] experts
  int E, N, K, div, act, n_pairs;
};
struct FewList {
  unsigned short list[FEW_PAIRS];
  int len;
};
__host__ inline bool few_ok(const FewExperts& a) {
  return a.E > 0 && a.N > 0 && a.K > 0 && a.N % 8 == 0 && a.K % 8 == 0 &&
         a.div > 0 && a.E <= 65535 && a.n_pairs <= FEW_PAIRS;
}

template <int MT>
__device__ __forceinline__ void few_block(const FewExperts& a, int block,
                                          int e, char* lds, FewList& pairs) {
  static_assert(FewTile<2, MT>::LDS <= FEW_LDS<MT> &&
                    FewTile<4, MT>::LDS <= FEW_LDS<MT>,
                "one size of LDS for all tiles");
  const int n0 = block * 16 * MT, N = a.N, K = a.K;
  const bf16_t *in = a.in, *w = a.w;
  unsigned short* list = pairs.list;
  const int tid = threadIdx.x;
  if (tid == 0) pairs.len = 0;
  __syncthreads();
  for (int p = tid; p < a.n_pairs; p += FEW_KW * 64)
    if (a.index[p] == e)
      list[atomicAdd(&pairs.len, 1)] = (unsigned short)p;
  __syncthreads();
  const int count = pairs.len;
  auto tile = [&](auto t, int first) {
    using Tile = decltype(t);
    Tile::run(
        lds, K, block + e,
        [&](int r) {
          const int p = first + r < count ? first + r : count - 1;
          return in + (size_t)(list[p] / a.div) * K;
        },
        [&](int r) {
          return w + ((size_t)e * N + (n0 + r < N ? n0 + r : N - 1)) * K;
        });
    Tile::each(4 * MT, [&](int r, int c) {
      f32x4 v = Tile::sum(lds, r, c);
      if (a.act) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          v[j] = fmaxf(v[j], 0.f);
          v[j] *= v[j];
        }
      }
      if (first + r < count && n0 + c < N)
        *reinterpret_cast<uint2*>(a.out + (size_t)list[first + r] * N + n0 +
                                  c) =
            make_uint2(to_bf16x2(v[0], v[1]), to_bf16x2(v[2], v[3]));
    });
    __syncthreads();
  };
  for (int first = 0; first < count; first += 64) {
    const int left = count - first;
    if (left <= 16) tile(FewTile<1, MT>{}, first);
    else if (left <= 32) tile(FewTile<2, MT>{}, first);
    else tile(FewTile<4, MT>{}, first);
  }
}
