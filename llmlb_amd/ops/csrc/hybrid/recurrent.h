// Pieces shared by the recurrent layers: short convolutions over packed
// tokens, runs of neighbouring elements, rows of a state.
//
// A state is [slots][H][V][D] float, value-major: 16 neighbouring lanes
// hold one value column, rows_per_lane(D) key channels each, and read it
// in one run.  A convolution's last inputs are a ring [slots][taps][C],
// position p in entry p % taps: the entry of the current token is never
// one that its own taps read.
#pragma once
#include "row_act.h"

// silu(conv + bias) of channel c at packed token t (bias null: none)
template <typename T>
__device__ __forceinline__ float conv_silu(
    const T* __restrict__ proj, int ld, const T* __restrict__ ring,
    const float* __restrict__ wconv, const float* __restrict__ bias, int C,
    int taps, int c, int t, int pos, int tstart, int slot) {
  float acc = to_f(proj[(size_t)t * ld + c]) *
                  wconv[(size_t)(taps - 1) * C + c] +
              (bias ? bias[c] : 0.f);
  for (int back = 1; back < taps; ++back) {
    const int p = pos - back;
    if (p < 0) break;
    const float in =
        t - back >= tstart
            ? to_f(proj[(size_t)(t - back) * ld + c])
            : to_f(ring[((size_t)slot * taps + p % taps) * C + c]);
    acc += in * wconv[(size_t)(taps - 1 - back) * C + c];
  }
  return silu_f(acc);
}

// N consecutive elements, as wide as alignment allows; VEC: the address
// is aligned to the whole run (or to 16 bytes).
template <int N, bool VEC>
__device__ __forceinline__ void load_run(const bf16_t* p, float* f) {
  if (VEC && N % 8 == 0) {
#pragma unroll
    for (int i = 0; i < N; i += 8) load8(p + i, f + i);
  } else if (VEC && N == 4) {
    load4(p, f);
  } else {
#pragma unroll
    for (int i = 0; i < N; ++i) f[i] = to_f(p[i]);
  }
}
template <int N, bool VEC>
__device__ __forceinline__ void load_run(const float* p, float* f) {
  if (VEC && N % 4 == 0) {
#pragma unroll
    for (int i = 0; i < N; i += 4) load4(p + i, f + i);
  } else {
#pragma unroll
    for (int i = 0; i < N; ++i) f[i] = p[i];
  }
}
template <int N, bool VEC>
__device__ __forceinline__ void store_run(float* p, const float* f) {
  if (VEC && N % 4 == 0) {
#pragma unroll
    for (int i = 0; i < N; i += 4) store4(p + i, f + i);
  } else {
#pragma unroll
    for (int i = 0; i < N; ++i) p[i] = f[i];
  }
}
template <int N, bool VEC>
__device__ __forceinline__ void store_run(bf16_t* p, const float* f) {
  if (VEC && N % 8 == 0) {
#pragma unroll
    for (int i = 0; i < N; i += 8) store8(p + i, f + i);
  } else if (VEC && N == 4) {
    store4(p, f);
  } else {
#pragma unroll
    for (int i = 0; i < N; ++i) p[i] = from_f<bf16_t>(f[i]);
  }
}
// only the first ``valid`` of N elements exist
template <int N, bool VEC, typename T>
__device__ __forceinline__ void load_some(const T* p, int valid, float* f) {
  if (VEC || valid >= N) {
    load_run<N, VEC>(p, f);
  } else {
#pragma unroll
    for (int i = 0; i < N; ++i) f[i] = i < valid ? to_f(p[i]) : 0.f;
  }
}
template <int N, bool VEC, typename T>
__device__ __forceinline__ void store_some(T* p, int valid, const float* f) {
  if (VEC || valid >= N) {
    store_run<N, VEC>(p, f);
  } else {
#pragma unroll
    for (int i = 0; i < N; ++i)
      if (i < valid) p[i] = from_f<T>(f[i]);
  }
}

// 16-bit models take the hardware's exponential and logarithm
template <typename T>
__device__ __forceinline__ float sigmoid_t(float x) {
  return sizeof(T) == 2 ? 1.f / (1.f + __expf(-x)) : sigmoid_f(x);
}
// (BOTH: log(1 + e) and its series are made and one is taken, which is less than
// a branch where nothing else hides it, and more where many numbers do.)
template <typename T, bool BOTH = false>
__device__ __forceinline__ float decay_t(float z, float rate) {
  if (sizeof(T) == 2) {
    const float e = __expf(-fabsf(z));
    // log(1 + e) by its series where 1 + e would lose e
    float lp;
    if (BOTH) {
      constexpr float LN2 = 0.6931471805599453f;
      const float l = LN2 * __builtin_amdgcn_logf(1.f + e);
      lp = e < 1e-3f ? e * (1.f - 0.5f * e) : l;
    } else {
      lp = e < 1e-3f ? e * (1.f - 0.5f * e) : __logf(1.f + e);
    }
    return __expf(-rate * (fmaxf(z, 0.f) + lp));
  }
  return expf(-rate * softplus_f(z));
}

// The convolution of N neighbouring channels over consecutive tokens,
// each input read once: ``hist`` holds the last taps - 1 inputs.
#define TAPS_MAX 4
template <typename T, int N, bool VEC>
struct ConvRun {
  float w[TAPS_MAX][N], hist[TAPS_MAX - 1][N], b0[N];
  const T* proj;
  const T* ring;
  int ld, C, taps, c, valid;

  __device__ __forceinline__ ConvRun(const T* proj_, int ld_, const T* ring_,
                                     const float* wconv, const float* bias,
                                     int C_, int taps_, int c_, int valid_)
      : proj(proj_), ring(ring_), ld(ld_), C(C_), taps(taps_), c(c_),
        valid(valid_) {
#pragma unroll
    for (int b = 0; b < TAPS_MAX; ++b)
      if (b < taps)
        load_some<N, VEC>(wconv + (size_t)(taps - 1 - b) * C + c, valid,
                          w[b]);
#pragma unroll
    for (int i = 0; i < N; ++i) b0[i] = 0.f;
    if (bias) load_some<N, VEC>(bias + c, valid, b0);
  }
  // inputs before token t, from the batch or the sequence's ring
  __device__ __forceinline__ void start(int t, int pos, int tstart,
                                        int slot) {
#pragma unroll
    for (int b = 1; b < TAPS_MAX; ++b) {
#pragma unroll
      for (int i = 0; i < N; ++i) hist[b - 1][i] = 0.f;
      if (b < taps && pos - b >= 0)
        load_some<N, VEC>(
            t - b >= tstart
                ? proj + (size_t)(t - b) * ld + c
                : ring + ((size_t)slot * taps + (pos - b) % taps) * C + c,
            valid, hist[b - 1]);
    }
  }
  __device__ __forceinline__ void load(int t, float* x) const {
    load_some<N, VEC>(proj + (size_t)t * ld + c, valid, x);
  }
  // the next token, whose inputs are x
  __device__ __forceinline__ void step(const float* x, float* y) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      float acc = x[i] * w[0][i] + b0[i];
#pragma unroll
      for (int b = 1; b < TAPS_MAX; ++b)
        if (b < taps) acc += hist[b - 1][i] * w[b][i];
#pragma unroll
      for (int b = TAPS_MAX - 1; b > 1; --b) hist[b - 1][i] = hist[b - 2][i];
      hist[0][i] = x[i];
      y[i] = sizeof(T) == 2 ? row_ratio(acc, __expf(-acc))
                            : acc * sigmoid_f(acc);
    }
  }
};

// A row's parts, a workgroup each, of runs of rows: side by side where
// ``together``, else a part of all runs after the other.
struct RunPart {
  int run, part;
};
__host__ inline dim3 run_parts(int runs, int parts, bool together) {
  return together ? dim3((unsigned)runs * (unsigned)parts)
                  : dim3((unsigned)runs, (unsigned)parts);
}
__device__ __forceinline__ RunPart run_part(int parts) {
  if (gridDim.y > 1) return RunPart{(int)blockIdx.x, (int)blockIdx.y};
  return RunPart{(int)blockIdx.x / parts, (int)blockIdx.x % parts};
}

// Tokens t0 .. t1 - 1 in order, some at a time: start(t, its sequence's first)
// where the tokens before t have not been walked, go(t, n) for the next n.  n,
// a constant, is GROUP where all of these are of one sequence, else 1.
template <int GROUP, class Start, class Go>
__device__ __forceinline__ void walk_tokens(const int* tstart, int t0, int t1,
                                            Start start, Go go) {
  constexpr std::integral_constant<int, 1> ONE{};
  for (int t = t0; t < t1;) {
    const int first = tstart[t];
    if (t == t0 || t == first) start(t, first);
    if constexpr (GROUP > 1) {
      if (t + GROUP <= t1 && tstart[t + GROUP - 1] <= t) {
        go(t, std::integral_constant<int, GROUP>{});
        t += GROUP;
        continue;
      }
    }
    go(t++, ONE);
  }
}

template <int RPL, bool EXACT>
__device__ __forceinline__ void load_rows(const float* __restrict__ p, int r0,
                                          int D, float* f) {
  if (EXACT && RPL % 4 == 0) {
#pragma unroll
    for (int i = 0; i < RPL / 4; ++i) {
      const float4 v = reinterpret_cast<const float4*>(p + r0)[i];
      f[i * 4] = v.x; f[i * 4 + 1] = v.y;
      f[i * 4 + 2] = v.z; f[i * 4 + 3] = v.w;
    }
  } else {
#pragma unroll
    for (int i = 0; i < RPL; ++i)
      f[i] = (EXACT || r0 + i < D) ? p[r0 + i] : 0.f;
  }
}

template <int RPL, bool EXACT>
__device__ __forceinline__ void store_rows(float* __restrict__ p, int r0,
                                           int D, const float* f) {
  if (EXACT && RPL % 4 == 0) {
#pragma unroll
    for (int i = 0; i < RPL / 4; ++i)
      reinterpret_cast<float4*>(p + r0)[i] =
          make_float4(f[i * 4], f[i * 4 + 1], f[i * 4 + 2], f[i * 4 + 3]);
  } else {
#pragma unroll
    for (int i = 0; i < RPL; ++i)
      if (EXACT || r0 + i < D) p[r0 + i] = f[i];
  }
}

// The same with a lane's numbers spread over the column by fours: number i is
// channel spread_at<RPL, EXACT>(lane, i).  16 lanes then read and write 256
// bytes in a row with each instruction, where every lane's own run leaves
// gaps that a later instruction fills.  They go past the caches: a step
// reads and writes every state once, and what it leaves dirty in them is
// written back under the products that follow.  64 sequences at 32 heads of
// 128 x 128, us a step of the model: Dibelix 1634 with runs by way of the
// caches, 1630 spread, 1617 with stores past the caches, 1615 with loads, 1540
// with both; Taletar 1596, 1592, 1564, 1570, 1526.
template <int RPL, bool EXACT>
__device__ __forceinline__ int spread_at(int lane, int i) {
  return EXACT && RPL % 4 == 0 ? i / 4 * 64 + lane * 4 + i % 4
                               : lane * RPL + i;
}
typedef __attribute__((ext_vector_type(4))) float fvec4;
template <int RPL, bool EXACT>
__device__ __forceinline__ void load_spread(const float* __restrict__ p,
                                            int lane, int D, float* f) {
  if (EXACT && RPL % 4 == 0) {
#pragma unroll
    for (int i = 0; i < RPL / 4; ++i) {
      const fvec4 v = __builtin_nontemporal_load(
          reinterpret_cast<const fvec4*>(p) + i * 16 + lane);
#pragma unroll
      for (int j = 0; j < 4; ++j) f[i * 4 + j] = v[j];
    }
  } else {
    load_rows<RPL, EXACT>(p, lane * RPL, D, f);
  }
}
template <int RPL, bool EXACT>
__device__ __forceinline__ void store_spread(float* __restrict__ p, int lane,
                                             int D, const float* f) {
  if (EXACT && RPL % 4 == 0) {
#pragma unroll
    for (int i = 0; i < RPL / 4; ++i) {
      const fvec4 v = {f[i * 4], f[i * 4 + 1], f[i * 4 + 2], f[i * 4 + 3]};
      __builtin_nontemporal_store(
          v, reinterpret_cast<fvec4*>(p) + i * 16 + lane);
    }
  } else {
    store_rows<RPL, EXACT>(p, lane * RPL, D, f);
  }
}

// key channels a lane holds when 16 lanes share a column of D
static int rows_per_lane(int D) {
  int r = 1;
  while (r * 16 < D) r *= 2;
  return r;
}

#define HY_RPL(D, ...)                                                  \
  do {                                                                  \
    const int rpl__ = rows_per_lane(D);                                 \
    const bool ex__ = rpl__ * 16 == (D);                                \
    if (rpl__ == 1) { constexpr int RPL = 1; HY_EX(__VA_ARGS__); }      \
    else if (rpl__ == 2) { constexpr int RPL = 2; HY_EX(__VA_ARGS__); } \
    else if (rpl__ == 4) { constexpr int RPL = 4; HY_EX(__VA_ARGS__); } \
    else if (rpl__ == 8) { constexpr int RPL = 8; HY_EX(__VA_ARGS__); } \
    else if (rpl__ == 16) { constexpr int RPL = 16; HY_EX(__VA_ARGS__); } \
    else { constexpr int RPL = 32; HY_EX(__VA_ARGS__); }                \
  } while (0)
#define HY_EX(...)                                        \
  if (ex__) { constexpr bool EXACT = true; __VA_ARGS__; } \
  else { constexpr bool EXACT = false; __VA_ARGS__; }
