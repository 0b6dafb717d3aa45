// Attention of float models to cached rows that several heads share, on the
// matrix cores in float (16x16x4 MFMAs, exact products): what the kernels of
// latent and of windowed attention have in common.
//
// A workgroup: one token and up to 16 heads that read the same keys and
// values; the waves take every NW-th 16 keys and meet at the end.
//   S^T = K Q^T: a lane holds the scores of keys 4g .. 4g + 3 (g = lane /
//   16) for head n = lane % 16, which is the operand of O^T = V^T P^T.
// A product's four numbers of a lane are neighbours in memory, in the
// contraction as among the 64 value columns of four products, so that keys
// and values are read 16 bytes a lane, straight from the cache.  A kernel of
// a head at a time read every row once per head, which was its bound.
#pragma once
#include "mfma.h"

#define ROWS_KEYS 16

// Numbers a row: W of them meet the query's, V from v_off on are values.
// E: weights are powers of e, not of two (a factor of log2(e) on the queries
// or the scores would cost their last bits).
template <int VT, int NW, bool E>
struct FloatRows {
  static_assert(VT % 4 == 0, "64 columns at a time");
  static __device__ __forceinline__ float power(float x) {
    return E ? expf(x) : exp2f(x);
  }
  // floats of LDS
  static constexpr int maxima = 2 * 16 * NW;
  static __host__ __device__ int pitch(int W) { return (W + 15) / 16 * 16 + 4; }
  static __host__ __device__ int floats(int W) {
    const int q = 16 * pitch(W), o = 16 * (16 * VT + 4);
    return maxima + (q > o ? q : o);
  }

  // lds: at ``maxima`` the queries [16][pitch], scaled, zeros past W and past the real heads (the caller has waited for them).
  //   row(j): where key j's row begins
  // Leaves there the sums of values [16][16 VT + 4] and returns the sum of
  // weights of head n, both relative to the returned maximum; all threads
  // may read them.
  template <class R>
  static __device__ __forceinline__ float run(float* lds, R row, int W,
                                              int v_off, int V, int first,
                                              int last, float& max_out) {
    const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    float* lq = lds + maxima;
    const int KP = pitch(W), blocks = (W + 15) / 16;
    f32x4 o[VT];
    float m = -1e30f, l = 0.f;
#pragma unroll
    for (int v = 0; v < VT; ++v) o[v] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int j0 = first + wave * ROWS_KEYS; j0 <= last;
         j0 += NW * ROWS_KEYS) {
      const float* key = row(j0 + n < last ? j0 + n : last);
      // 128 numbers at a time, in four parts: long sums lose digits
      f32x4 s = {0.f, 0.f, 0.f, 0.f};
      for (int b0 = 0; b0 < blocks; b0 += 8) {
        f32x4 part[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) part[i] = f32x4{0.f, 0.f, 0.f, 0.f};
        const int end = b0 + 8 < blocks ? b0 + 8 : blocks;
#pragma unroll 4
        for (int b = b0; b < end; ++b) {
          const int d = b * 16 + g * 4;
          const f32x4 k =
              *reinterpret_cast<const f32x4*>(key + (d < W ? d : 0));
          const f32x4 q = *reinterpret_cast<const f32x4*>(lq + n * KP + d);
#pragma unroll
          for (int i = 0; i < 4; ++i)
            part[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(k[i], q[i], part[i],
                                                           0, 0, 0);
        }
        s += (part[0] + part[1]) + (part[2] + part[3]);
      }
      const float* value[4];
      float mx = m;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int j = j0 + g * 4 + i;
        value[i] = row(j < last ? j : last) + v_off;
        s[i] = j <= last ? s[i] : -INFINITY;
        mx = fmaxf(mx, s[i]);
      }
      mx = fmaxf(mx, __shfl_xor(mx, 16, WAVE));
      mx = fmaxf(mx, __shfl_xor(mx, 32, WAVE));
      const float keep = power(m - mx);
      m = mx;
      l *= keep;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        s[i] = power(s[i] - m);
        l += s[i];
      }
#pragma unroll
      for (int v = 0; v < VT; ++v) o[v] *= keep;
#pragma unroll
      for (int v = 0; v < VT; v += 4) {
        const int c = v * 16 + n * 4;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const f32x4 x =
              *reinterpret_cast<const f32x4*>(value[i] + (c < V ? c : 0));
#pragma unroll
          for (int a = 0; a < 4; ++a)
            o[v + a] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[a], s[i],
                                                            o[v + a], 0, 0, 0);
        }
      }
    }
    l += __shfl_xor(l, 16, WAVE);
    l += __shfl_xor(l, 32, WAVE);
    if (g == 0) {
      lds[n * NW + wave] = m;
      lds[(16 + n) * NW + wave] = l;
    }
    __syncthreads();  // the queries have been read as well
    float mx = lds[n * NW];
#pragma unroll
    for (int w = 1; w < NW; ++w) mx = fmaxf(mx, lds[n * NW + w]);
    float sum = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w)
      sum += power(lds[n * NW + w] - mx) * lds[(16 + n) * NW + w];
    const float mine = power(m - mx);
    // register i of products v .. v + 3: columns 16 v + 16 g + 4 i .. + 3
    float* to = lq + n * (16 * VT + 4) + g * 16;
    for (int w = 0; w < NW; ++w) {
      if (w == wave)
#pragma unroll
        for (int v = 0; v < VT; v += 4)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            f32x4* x = reinterpret_cast<f32x4*>(to + v * 16 + i * 4);
            const f32x4 add = f32x4{o[v][i], o[v + 1][i], o[v + 2][i],
                                    o[v + 3][i]} * mine;
            *x = w == 0 ? add : *x + add;
          }
      __syncthreads();
    }
    max_out = mx;
    return sum;
  }
};

// GO(VT, NW) for V <= 512: sixteen waves where a workgroup a token and 16
// heads leaves the chip idle
#define FLOAT_ROWS_SIZES(groups, V)               \
  do {                                            \
    const bool many = (groups) < 256;             \
    if ((V) <= 64 && many) GO(4, 16);             \
    else if ((V) <= 64) GO(4, 4);                 \
    else if ((V) <= 128 && many) GO(8, 16);       \
    else if ((V) <= 128) GO(8, 4);                \
    else if ((V) <= 256 && many) GO(16, 16);      \
    else if ((V) <= 256) GO(16, 4);               \
    else GO(32, 4);                               \
  } while (0)
