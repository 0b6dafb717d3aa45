// One tile of a product of a few normed rows with a weight matrix: RowTile with
// rows of x that the workgroup norms itself and keeps in LDS.
//
// The norm's own launch takes about 2 us where the product takes 4, and little
// of it is data.  Here every workgroup copies all rows to LDS, then the first
// pieces of its W, and norms while these are on their way.  (Rows loaded to
// registers make a wave wait for its pieces first: 1536 x 1024, one row 4.6 us,
// 5632 x 1024 gate and up 6.2; with copies 4.9 and 5.8.)
#pragma once
#include "row_tile.h"

// x = rows (+ residual), out = x rsqrt(mean(x^2) + eps) weight, as rmsnorm
struct RowNorm {
  const bf16_t* residual;  // null: none
  bf16_t* sum;             // rows + residual; null: nobody wants it
  const bf16_t* weight;
  float eps;
};

template <int MT, int KW, int S>
struct NormTile {
  static constexpr int C = 2 * MT, STAGE = MT * 2048;
  static constexpr int RP = 16 * MT + 4;
  static constexpr int STAGES = KW * S * STAGE, SUMS = KW * 16 * RP * 4;
  static constexpr int FIXED = STAGES > SUMS ? STAGES : SUMS;
  static constexpr int VECTORS = 4;  // of 8 numbers that a lane has of a row
  static constexpr int DEEPEST = VECTORS * 8 * WAVE;
  // Rows lie in whole copies of 1 KB, and begin on other banks
  static __host__ __device__ __forceinline__ int pitch(int K) {
    return (2 * K + 1023) / 1024 * 1024 + 16;
  }
  // rows of x, of the residual, and the norm's weight
  static __host__ __device__ __forceinline__ int lds(int N, int K) {
    return FIXED + (2 * N + 1) * pitch(K);
  }

  // K: a multiple of 64, DEEPEST at most; others as for RowTile
  template <class W, class L>
  static __device__ __forceinline__ void run(char* lds, int N, int K, int step,
                                             const bf16_t* x, int ldx,
                                             const RowNorm& norm, bool writes,
                                             W w_row, L last) {
    const int tid = threadIdx.x, lane = tid & 63;
    const int lo = lane & 15, hi = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    char* const own = lds + wave * (S * STAGE);
    char* const rows = lds + FIXED;
    const unsigned own_byte = lds_byte(own);
    const bf16_t* src[C];
#pragma unroll
    for (int j = 0; j < C; ++j) {
      const int r = 8 * j + lane / 8;
      src[j] = w_row(r) + ((lane & 7) ^ ((r >> 1) & 7)) * 8;
    }
    const int pieces = K / 64;
    const int count = pieces > wave ? (pieces - wave + KW - 1) / KW : 0;
    const int turn = count ? step % count : 0;
    auto depth = [&](int i) {
      const int at = i + turn;
      return (wave + (at < count ? at : at - count) * KW) * 64;
    };
    auto copy = [&](int i) {
      const int k0 = depth(i);
      const unsigned to = own_byte + i % S * STAGE;
#pragma unroll
      for (int j = 0; j < C; ++j) stream_to_lds(src[j] + k0, to + j * 1024);
    };
    // rows first: they are normed while the first pieces of W are on their way
    const int P = pitch(K), each = P / 1024;
    for (int i = wave; i < (2 * N + 1) * each; i += KW) {
      const int row = i / each, at = i % each * 512 + lane * 8;
      if (row >= N && row < 2 * N && !norm.residual) continue;
      const bf16_t* from = row < N ? x + (size_t)row * ldx
                           : row < 2 * N
                               ? norm.residual + (size_t)(row - N) * K
                               : norm.weight;
      copy_to_lds(at < K ? from + at
                         : reinterpret_cast<const bf16_t*>(zero_piece),
                  lds_byte(rows) + row * P + i % each * 1024);
    }
#pragma unroll
    for (int i = 0; i < S; ++i)
      if (i < count) copy(i);
    if (count >= S)
      wait_copies<S * C>();
    else
      wait_copies<0>();
    __syncthreads();

    const int vectors = K / 8;
    const u32x4* const gv = reinterpret_cast<const u32x4*>(rows + 2 * N * P);
    for (int n = wave; n < N; n += KW) {  // a row a wave
      u32x4 v[VECTORS];
      u32x4* const xv = reinterpret_cast<u32x4*>(rows + n * P);
      const u32x4* const rv =
          reinterpret_cast<const u32x4*>(rows + (N + n) * P);
      float squares = 0.f;
#pragma unroll
      for (int j = 0; j < VECTORS; ++j) {
        const int i = lane + j * WAVE;
        if (i >= vectors) continue;
        v[j] = xv[i];
        if (norm.residual) {
          const u32x4 r = rv[i];
#pragma unroll
          for (int c = 0; c < 4; ++c)
            v[j][c] = to_bf16x2(__uint_as_float(v[j][c] << 16) +
                                    __uint_as_float(r[c] << 16),
                                __uint_as_float(v[j][c] & 0xffff0000u) +
                                    __uint_as_float(r[c] & 0xffff0000u));
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const float a = __uint_as_float(v[j][c] << 16);
          const float b = __uint_as_float(v[j][c] & 0xffff0000u);
          squares += a * a;
          squares += b * b;
        }
      }
#pragma unroll
      for (int off = WAVE / 2; off; off >>= 1)
        squares += __shfl_xor(squares, off, WAVE);
      const float scale = rsqrtf(squares / K + norm.eps);
#pragma unroll
      for (int j = 0; j < VECTORS; ++j) {
        const int i = lane + j * WAVE;
        if (i >= vectors) continue;
        const u32x4 g = gv[i], sum = v[j];
#pragma unroll
        for (int c = 0; c < 4; ++c)
          v[j][c] = to_bf16x2(__uint_as_float(v[j][c] << 16) * scale *
                                  __uint_as_float(g[c] << 16),
                              __uint_as_float(v[j][c] & 0xffff0000u) * scale *
                                  __uint_as_float(g[c] & 0xffff0000u));
        xv[i] = v[j];
        if (writes && norm.residual)
          *reinterpret_cast<u32x4*>(norm.sum + (size_t)n * K + i * 8) = sum;
      }
    }
    __syncthreads();

    f32x4 acc[MT];
#pragma unroll
    for (int a = 0; a < MT; ++a) acc[a] = f32x4{0.f, 0.f, 0.f, 0.f};
    const char* const row = rows + (lo < N ? lo : N - 1) * P;
    for (int i = 0; i < count; ++i) {
      const int newer = count - 1 - i;
      if (newer >= S - 1)
        wait_copies<(S - 1) * C>();
      else if (S > 2 && newer == 1)
        wait_copies<(S > 2 ? C : 0)>();
      else
        wait_copies<0>();
      if (newer == 0) last();
      const char* st = own + i % S * STAGE;
      const int k0 = depth(i);
      u32x4 wf[2][MT], xf[2];
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        xf[s] = *reinterpret_cast<const u32x4*>(row + k0 * 2 +
                                                (s * 4 + hi) * 16);
#pragma unroll
        for (int a = 0; a < MT; ++a)
          wf[s][a] = *reinterpret_cast<const u32x4*>(
              st + a * 2048 + lo * 128 + ((s * 4 + hi) ^ (lo >> 1)) * 16);
      }
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int a = 0; a < MT; ++a) acc[a] = mfma(wf[s][a], xf[s], acc[a]);
      // the stage has been read before its next copy starts
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      if (i + S < count) copy(i + S);
    }
    if (count == 0) last();
    __syncthreads();  // the sums lie where the stages were
    float* const sums = reinterpret_cast<float*>(lds);
#pragma unroll
    for (int a = 0; a < MT; ++a)
      *reinterpret_cast<f32x4*>(
          &sums[(wave * 16 + lo) * RP + a * 16 + hi * 4]) = acc[a];
    __syncthreads();
  }

  // outputs c .. c + 3 of the tile's row r of x
  static __device__ __forceinline__ f32x4 sum(const char* lds, int r, int c) {
    const float* const sums = reinterpret_cast<const float*>(lds);
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < KW; ++w)
      v += *reinterpret_cast<const f32x4*>(&sums[(w * 16 + r) * RP + c]);
    return v;
  }
};
