// The loop of prompt attention that its kernels share: 128 rows a workgroup
// of four waves, 32 a wave, a row being one head of one query; keys and
// values of one head in tiles of 64, bf16.
//
// S^T = K Q^T with 16x16x32 MFMAs: a lane holds, for ONE row n = lane % 16
// of each of its two sets, the scores of keys 4g .. 4g + 3 of each 16-key
// tile (g = lane / 16), so that sums and maxima are its own, and P^T is
// already the operand of O^T = V^T P^T.
//
// With 128 numbers a key the matrix cores need 1024 cycles for a wave's tile
// and LDS as many for the two waves of a SIMD, so what costs is all that
// comes on top.
//  * Tiles are copied to LDS by the memory path itself, one ahead, with one
//    barrier a tile; V is read transposed.
//  * A row's first tile with keys sets what its scores are taken relative
//    to, their maximum; after that it moves only when the weights grow out
//    of range (2^40), which the sum that is needed anyway shows.  Any such
//    number gives the same quotient, float and bf16 reach far enough, and
//    the common path has no maxima, no exchange between lanes and no
//    scaling of accumulators.
//  * Tiles before and after those that a wave sees are loops of their own,
//    so that accumulators stay in their registers.
// Times stand with the kernels.
#pragma once
#include "lds_copy.h"
#include "mfma.h"

// A tile's 64 rows of D numbers in LDS.
template <int D>
struct TileRows {
  static_assert(D == 64 || D == 96 || D == 128 || D == 192,
                "what turn() knows, in whole copies");
  static constexpr int ROW = 2 * D, PR = ROW / 16;  // bytes, pieces of 16
  static constexpr int BYTES = 64 * ROW;
  static constexpr int COPIES = 16 * PR / 64;  // of a wave, its 16 rows

  // Piece c of row r lies at c ^ turn(r): lanes reading one piece of 16
  // rows meet every bank once.
  static __device__ __forceinline__ int turn(int r) {
    return D == 128 ? r & 15 : D == 96 ? (r >> 2) & 3 : (r >> 1) & 7;
  }
  // row among the wave's 16 and its piece that a lane copies in copy c
  static __device__ __forceinline__ int row(int c, int lane) {
    return (c * 64 + lane) / PR;
  }
  static __device__ __forceinline__ int piece(int c, int lane) {
    return (c * 64 + lane) % PR ^ turn(row(c, lane));
  }
};

// where 16 neighbouring rows of keys and values begin
struct KeyRows {
  const bf16_t *k, *v;
};

// Rows of as many numbers for keys and values, ld apart among 16
// neighbours.  find(j): KeyRows of keys j .. j + 15, j a multiple of 16.
template <int D, class Find>
struct PagedRows {
  using Tile = TileRows<D>;
  Find find;
  int ld, last, lane;
  unsigned off[Tile::COPIES];

  __device__ __forceinline__ PagedRows(Find f, int ld_, int last_)
      : find(f), ld(ld_), last(last_), lane(threadIdx.x & 63) {
#pragma unroll
    for (int c = 0; c < Tile::COPIES; ++c) off[c] = place(c, 15);
  }
  __device__ __forceinline__ unsigned place(int c, int most) {
    const int r = Tile::row(c, lane);
    return (unsigned)((r < most ? r : most) * ld + Tile::piece(c, lane) * 8) *
           2;
  }
  // the wave's rows, from key j on; looked up a tile before they are copied
  __device__ __forceinline__ KeyRows look_up(int j) {
    return find((j < last ? j : last) & ~15);
  }
  __device__ __forceinline__ void copy(const KeyRows& s, int j, unsigned k_to,
                                       unsigned v_to) {
    if (j + 15 <= last) {
#pragma unroll
      for (int c = 0; c < Tile::COPIES; ++c) {
        copy_to_lds(s.k, off[c], k_to + c * 1024);
        copy_to_lds(s.v, off[c], v_to + c * 1024);
      }
    } else {
      // rows past the last one repeat it: their weights are zero, and
      // what they are multiplied with has to be a number
#pragma unroll
      for (int c = 0; c < Tile::COPIES; ++c) {
        const unsigned from = place(c, last & 15);
        copy_to_lds(s.k, from, k_to + c * 1024);
        copy_to_lds(s.v, from, v_to + c * 1024);
      }
    }
  }
};
template <int D, class Find>
__device__ __forceinline__ PagedRows<D, Find> paged_rows(Find f, int ld,
                                                         int last) {
  return PagedRows<D, Find>(f, ld, last);
}

// keys of DK numbers, values of DV
template <int DK, int DV = DK>
struct Flash {
  using K = TileRows<DK>;
  using V = TileRows<DV>;
  static constexpr int KD = DK / 32, VT = DV / 16;
  static constexpr int TILE = K::BYTES + V::BYTES, LDS = 2 * TILE;

  u32x4 qf[2][KD];
  f32x4 o[2][VT];
  float l[2];

  // Attention of the rows over keys lo .. last (lo a multiple of 16).
  //   rows: what brings a tile's rows, by wave (see PagedRows)
  //   pos, span: a row's position, and how far back it sees
  //   w_lo, w_hi: positions of the wave's first and last row; w_lo_key,
  //     w_hi_key: the first keys they see
  // scale: of scores, in powers of two; SCALED: it is not one
  // sink: a score (in powers of two) without key and value, if has_sink
  template <bool SCALED, class R>
  __device__ __forceinline__ void run(char* lds, R rows, int lo, int last,
                                      const int (&pos)[2],
                                      const int (&span)[2], int w_lo,
                                      int w_hi, int w_lo_key, int w_hi_key,
                                      float scale, float sink = 0.f,
                                      bool has_sink = false) {
    const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const unsigned at = lds_byte(lds) + wave * 16 * K::ROW;
    const unsigned at_v = lds_byte(lds) + K::BYTES + wave * 16 * V::ROW;
    auto look_up = [&](int j0) { return rows.look_up(j0 + wave * 16); };
    auto copy = [&](const auto& s, int j0, int buf) {
      rows.copy(s, j0 + wave * 16, at + buf * TILE, at_v + buf * TILE);
    };
    float m[2];
    bool seen[2];  // whether the row has met a key
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      m[a] = sink;
      l[a] = has_sink && g == 0 ? 1.f : 0.f;
      seen[a] = has_sink;
#pragma unroll
      for (int v = 0; v < VT; ++v) o[a][v] = f32x4{0.f, 0.f, 0.f, 0.f};
    }

    copy(look_up(lo), lo, 0);
    auto ahead = look_up(lo + 64);
    int buf = 0, j0 = lo;
    auto next = [&]() {  // the tile at j0 is there, the one after it comes
      wait_barrier<0>();
      if (j0 + 64 <= last) {
        copy(ahead, j0 + 64, buf ^ 1);
        ahead = look_up(j0 + 128);
      }
    };
    for (; j0 + 63 < w_lo_key && j0 <= last; j0 += 64, buf ^= 1) next();
    for (; j0 <= w_hi && j0 <= last; j0 += 64, buf ^= 1) {
      next();
      const char* kt = lds + buf * TILE;
      const char* vt = kt + K::BYTES;
      f32x4 s[2][4];
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        const float c = SCALED ? 0.f : -m[a];
#pragma unroll
        for (int t = 0; t < 4; ++t) s[a][t] = f32x4{c, c, c, c};
      }
#pragma unroll
      for (int k = 0; k < KD; ++k)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const u32x4 kf = *reinterpret_cast<const u32x4*>(
              kt + (t * 16 + n) * K::ROW + ((k * 4 + g) ^ K::turn(n)) * 16);
          s[0][t] = mfma(kf, qf[0][k], s[0][t]);
          s[1][t] = mfma(kf, qf[1][k], s[1][t]);
        }
      if (!(j0 + 63 <= w_lo && j0 >= w_hi_key)) {
#pragma unroll
        for (int a = 0; a < 2; ++a) {
          const int age = pos[a] - j0 - g * 4;
#pragma unroll
          for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i)
              s[a][t][i] =
                  (unsigned)(age - t * 16 - i) <= (unsigned)span[a]
                      ? s[a][t][i]
                      : -INFINITY;
        }
      }
      f32x4 w[2][4];
      float sum[2];
      // twice at most: rows whose weights are out of range are raised once
      for (bool raised = false;; raised = true) {
#pragma unroll
        for (int a = 0; a < 2; ++a) {
          sum[a] = 0.f;
#pragma unroll
          for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              w[a][t][i] = __builtin_amdgcn_exp2f(
                  SCALED ? fmaf(s[a][t][i], scale, -m[a]) : s[a][t][i]);
              sum[a] += w[a][t][i];
            }
        }
        if (raised || !__any(sum[0] > 0x1p40f || sum[1] > 0x1p40f ||
                             !(seen[0] && seen[1])))
          break;
#pragma unroll
        for (int a = 0; a < 2; ++a) {
          float mx = s[a][0][0];
#pragma unroll
          for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) mx = fmaxf(mx, s[a][t][i]);
          // above what the row's scores are relative to
          float over = SCALED ? mx * scale - m[a] : mx;
          over = fmaxf(over, __shfl_xor(over, 16, WAVE));
          over = fmaxf(over, __shfl_xor(over, 32, WAVE));
          float by = 0.f, keep = 1.f;
          if (over > 30.f || (!seen[a] && over > -INFINITY)) {
            by = over;
            keep = seen[a] ? __builtin_amdgcn_exp2f(-by) : 0.f;
            seen[a] = true;
          }
          m[a] += by;
          l[a] *= keep;
#pragma unroll
          for (int v = 0; v < VT; ++v) o[a][v] *= keep;
          if (!SCALED) {
#pragma unroll
            for (int t = 0; t < 4; ++t) s[a][t] -= by;
          }
        }
      }
      u32x4 pf[2][2];
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        l[a] += sum[a];
#pragma unroll
        for (int h = 0; h < 2; ++h)
          pf[a][h] = u32x4{to_bf16x2(w[a][2 * h][0], w[a][2 * h][1]),
                           to_bf16x2(w[a][2 * h][2], w[a][2 * h][3]),
                           to_bf16x2(w[a][2 * h + 1][0], w[a][2 * h + 1][1]),
                           to_bf16x2(w[a][2 * h + 1][2], w[a][2 * h + 1][3])};
      }
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const int r = p * 32 + g * 4 + (n >> 2);
#pragma unroll
        for (int v = 0; v < VT; ++v) {
          const int c = 2 * v + ((n >> 1) & 1);
          const u32x4 vf = load_columns(
              reinterpret_cast<const unsigned short*>(
                  vt + r * V::ROW + (c ^ V::turn(r)) * 16 + (n & 1) * 8),
              16 * DV);
          o[0][v] = mfma(vf, pf[0][p], o[0][v]);
          o[1][v] = mfma(vf, pf[1][p], o[1][v]);
        }
      }
    }
    for (; j0 <= last; j0 += 64, buf ^= 1) next();
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      l[a] += __shfl_xor(l[a], 16, WAVE);
      l[a] += __shfl_xor(l[a], 32, WAVE);
    }
  }
};
