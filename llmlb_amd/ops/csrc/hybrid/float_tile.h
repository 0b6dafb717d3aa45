// One tile of a product of 32-bit matrices on the matrix cores' bf16
// instructions; float_gemm.hip says how and why.
#pragma once
#include <float.h>

#include "lds_copy.h"
#include "row_act.h"

// the larger of ``most`` and the sizes of two numbers, in one instruction
__device__ __forceinline__ float larger(float most, float a, float b) {
  asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(most) : "v"(a), "v"(b));
  return most;
}

// A block of 16 x 16 outputs by the float instructions, where the sum of parts
// will not do; x, w: the lane's row (lane % 16) of each.  Bound by them and by
// waiting for rows: 600 rows of 4096 x 1024 take 44 us, 64 with one row that has
// no numbers (374 with a loop over the depth a lane), 176 (4711) with all of them.
static __device__ __forceinline__ f32x4 float_block(const float* x,
                                                    const float* w, int K) {
  x += threadIdx.x % WAVE / 16 * 4, w += threadIdx.x % WAVE / 16 * 4;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int k = 0; k < K; k += 128) {  // eight loads of each on their way
    f32x4 a[8], b[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int at = k + 16 * i < K ? k + 16 * i : k;
      a[i] = *reinterpret_cast<const f32x4*>(w + at);
      b[i] = *reinterpret_cast<const f32x4*>(x + at);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const bool more = k + 16 * i < K;
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(
            more ? a[i][j] : 0.f, more ? b[i][j] : 0.f, acc, 0, 0, 0);
      }
  }
  return acc;
}

// One tile, 16 NT rows of x against 16 MT of W; KW waves share it and split
// the depth in pieces of 32 (rows of 128 bytes), as RowTile's do.
template <int NT, int MT, int KW>
struct FloatTile {
  static constexpr int F = NT + MT, C = 2 * F;
  static constexpr int STAGE = F * 2048;  // one piece of all rows
  static constexpr int RP = 16 * MT + 4;  // row of the sums
  static constexpr int STAGES = KW * STAGE, SUMS = KW / 2 * 16 * NT * RP * 4;
  // behind the sums: the largest size in every 16th row of x, and of W, and a bit
  // for every block of 16 x 16 outputs
  static constexpr int ENDS = SUMS + 33 * 4;
  static constexpr int LDS = STAGES > ENDS ? STAGES : ENDS;

  // x_at(r), w_at(r): how many numbers behind x, w the tile's row r begins; each
  // row there is, for rows that there are not
  template <class X, class W>
  static __device__ __forceinline__ void run(char* lds, int K, int step,
                                             const float* x, X x_at,
                                             const float* w, W w_at) {
    const int tid = threadIdx.x, lane = tid & 63;
    const int lo = lane & 15, hi = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    char* const own = lds + wave * STAGE;
    const unsigned own_byte = lds_byte(own);
    // rows and pieces of 16 bytes lie as RowTile's
    unsigned at[C];
#pragma unroll
    for (int j = 0; j < C; ++j) {
      const int r = 8 * j + lane / 8, piece = ((lane & 7) ^ ((r >> 1) & 7)) * 4;
      at[j] = ((j < 2 * NT ? x_at(r) : w_at(r - 16 * NT)) + piece) * 4;
    }
    const int pieces = K / 32;
    const int count = pieces > wave ? (pieces - wave + KW - 1) / KW : 0;
    const int turn = count ? step % count : 0;
    auto copy = [&](int i) {
      const int turned = i + turn;
      const int k0 =
          (wave + (turned < count ? turned : turned - count) * KW) * 32;
#pragma unroll
      for (int j = 0; j < C; ++j)
        copy_to_lds(reinterpret_cast<const bf16_t*>((j < 2 * NT ? x : w) + k0),
                    at[j], own_byte + j * 1024);
    };
    f32x4 acc[MT][NT];
#pragma unroll
    for (int a = 0; a < MT; ++a)
#pragma unroll
      for (int b = 0; b < NT; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
    float most[2] = {0.f, 0.f};  // of the lane's rows of x, of W
    if (count) copy(0);
    for (int i = 0; i < count; ++i) {
      wait_copies<0>();
      u32x4 raw[F][2], part[F][3];
#pragma unroll
      for (int f = 0; f < F; ++f)
#pragma unroll
        for (int s = 0; s < 2; ++s)
          raw[f][s] = *reinterpret_cast<const u32x4*>(
              own + f * 2048 + lo * 128 + ((s * 4 + hi) ^ (lo >> 1)) * 16);
      // the stage has been read before its next copy starts
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      if (i + 1 < count) copy(i + 1);
      auto take_apart = [&](int f) {
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
          for (int c = 0; c < 2; ++c) {
            const float lo = __uint_as_float(raw[f][s][2 * c]);
            const float hi = __uint_as_float(raw[f][s][2 * c + 1]);
            most[f >= NT] = larger(most[f >= NT], lo, hi);
            unsigned p[3];
            split3(lo, hi, p[0], p[1], p[2]);
#pragma unroll
            for (int t = 0; t < 3; ++t) part[f][t][2 * s + c] = p[t];
          }
      };
      // the k-th 16 rows that are taken apart: of x and W in turn
      auto kth = [](int k) {
        constexpr int few = NT < MT ? NT : MT;
        const bool of_x = k < 2 * few ? k % 2 == 0 : NT > MT;
        const int i = k < 2 * few ? k / 2 : k - few;
        return of_x ? i : NT + i;
      };
      // products of the k-th with all before it
      auto products = [&](int k) {
        constexpr int WP[] = {2, 0, 1, 1, 0, 0}, XP[] = {0, 2, 1, 0, 1, 0};
        const int f = kth(k);
#pragma unroll
        for (int q = 0; q < 6; ++q)
#pragma unroll
          for (int j = 0; j < k; ++j) {
            const int g = kth(j);
            if ((f < NT) == (g < NT)) continue;
            const int b = f < NT ? f : g, a = (f < NT ? g : f) - NT;
            acc[a][b] =
                mfma(part[NT + a][WP[q]], part[b][XP[q]], acc[a][b]);
          }
      };
      take_apart(kth(0));
      take_apart(kth(1));
#pragma unroll
      for (int k = 1; k < F; ++k) {
        __builtin_amdgcn_sched_barrier(0);
        products(k);
        if (k + 1 < F) take_apart(kth(k + 1));
#pragma unroll
        for (int i = 0; i < 24; ++i) {
          __builtin_amdgcn_sched_group_barrier(8, 1, 0);  // a matrix product
          __builtin_amdgcn_sched_group_barrier(2, 2, 0);  // two of the others
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }

    // the sums lie where the stages were: first those of half of the waves,
    // then the others' with them
    auto at_of = [&](int w, int a, int b) {
      return reinterpret_cast<f32x4*>(
          reinterpret_cast<float*>(lds) + (w * 16 * NT + b * 16 + lo) * RP +
          a * 16 + hi * 4);
    };
    __syncthreads();
    if (tid < 33) ends(lds)[tid] = 0;
    if (wave >= KW / 2) {
#pragma unroll
      for (int b = 0; b < NT; ++b)
#pragma unroll
        for (int a = 0; a < MT; ++a) *at_of(wave - KW / 2, a, b) = acc[a][b];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2; ++i)  // sizes are in order as whole numbers too
      atomicMax(&ends(lds)[16 * i + lo], __float_as_uint(most[i]));
    if (wave < KW / 2) {
#pragma unroll
      for (int b = 0; b < NT; ++b)
#pragma unroll
        for (int a = 0; a < MT; ++a) {
          f32x4* const at = at_of(wave, a, b);
          *at = *at + acc[a][b];
        }
    }
    __syncthreads();
  }

  static __device__ __forceinline__ unsigned* ends(char* lds) {
    return reinterpret_cast<unsigned*>(lds + SUMS);
  }
  static __device__ __forceinline__ f32x4 sum(const char* lds, int r, int c) {
    const float* const sums = reinterpret_cast<const float*>(lds);
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < KW / 2; ++w)
      v += *reinterpret_cast<const f32x4*>(
          &sums[(w * 16 * NT + r) * RP + c]);
    return v;
  }

  // What becomes of the sums: out_row(r) is where those of the tile's row r go,
  // x_row(r) and w_row(c) are the rows themselves; rows, cols: as many as there
  // are, or more.  kind: PLAIN, RELU2 or GELU.
  template <class X, class W, class O>
  static __device__ __forceinline__ void finish(char* lds, int K, int kind,
                                                int rows, int cols, X x_row,
                                                W w_row, O out_row) {
    // Outputs c .. c + 3 of row r whose sum of parts will not do: the parts of an
    // infinite number are that and no number, and parts below 2^-126 may be lost,
    // of a product 2^-125 of the other number and 2^-123 of sums.  So a sum has to
    // be 2^25 of what K products can lose, where rows have numbers at all (those of
    // padding have not), as far as the largest numbers of every 16th row tell.
    const unsigned* const most = ends(lds);
    const float least = K * 0x1p-98f;
    auto lost = [&](int r, int c, f32x4 v) {
      const float of_x = __uint_as_float(most[r % 16]);
      const f32x4 of_ws = *reinterpret_cast<const f32x4*>(most + 16 + c % 16);
      unsigned bits = 0;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float of_w = of_ws[j];
        const float size = fabsf(v[j]);
        const bool zeros = of_x == 0.f || of_w == 0.f;
        bits |= (!(size <= FLT_MAX) ||
                 (!zeros && !(size >= least * (1.f + of_x + of_w))))
                << j;
      }
      return bits;
    };
    auto put = [&](int r, int c, f32x4 v, unsigned bits) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (kind == RELU2) {
          v[j] = fmaxf(v[j], 0.f);
          v[j] *= v[j];
        } else if (kind == GELU) {
          v[j] = gelu_tanh_f(v[j]);
        }
      }
      float* const to = out_row(r) + c;
      if (bits == 15)
        *reinterpret_cast<f32x4*>(to) = v;
      else
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (bits >> j & 1) to[j] = v[j];
    };
    // all of a thread's sums are asked for before the first is looked at
    constexpr int ITEMS = 16 * NT * 4 * MT;
    constexpr int OF_ONE = (ITEMS + KW * 64 - 1) / (KW * 64);
    f32x4 sums[OF_ONE];
#pragma unroll
    for (int e = 0; e < OF_ONE; ++e) {
      const int i = threadIdx.x + e * KW * 64;
      if (i < ITEMS) sums[e] = sum(lds, i / (4 * MT), i % (4 * MT) * 4);
    }
#pragma unroll
    for (int e = 0; e < OF_ONE; ++e) {
      const int i = threadIdx.x + e * KW * 64;
      const int r = i / (4 * MT), c = i % (4 * MT) * 4;
      if (i >= ITEMS || r >= rows || c >= cols) continue;
      const f32x4 v = sums[e];
      const unsigned bits = lost(r, c, v);
      if (bits)
        atomicOr(ends(lds) + 32, 1u << (r / 16 * MT + c / 16));
      put(r, c, v, 15 & ~bits);
    }
    __syncthreads();
    unsigned blocks = __builtin_amdgcn_readfirstlane(most[32]);
    const int lo = threadIdx.x & 15;
    int others = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    for (; blocks; blocks &= blocks - 1) {  // every KW-th is the wave's
      if (others--) continue;
      others = KW - 1;
      const int block = __builtin_ctz(blocks);
      const int r = block / MT * 16 + lo, c0 = block % MT * 16;
      const f32x4 v =
          float_block(x_row(r < rows ? r : rows - 1),
                      w_row(c0 + lo < cols ? c0 + lo : cols - 1), K);
      const int c = c0 + threadIdx.x % WAVE / 16 * 4;
      if (r < rows && c < cols)
        put(r, c, v, lost(r, c, sum(lds, r, c)));
    }
  }
};
