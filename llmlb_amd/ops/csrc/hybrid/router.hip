// Routing kernels (router.h):
//  * route_kernel       bf16, 16 tokens a workgroup on the matrix cores
//  * route_rows_kernel  any size and either type, a workgroup a token
#include "router.h"

template <int NT>
__global__ __launch_bounds__(256) void route_kernel(Routing a) {
  extern __shared__ float lds[];
  route_block<NT>(a, blockIdx.x, lds);
}

// J experts of a wave at a time: their rows fly together (300 tokens of 1024
// columns, 16 experts, 32 bits, one by one 30.5 us, four 11), as many as a wave
// has, for each place is worked on (2000 tokens of 4100 columns, 4 experts, 16 bits,
// one by one 18 us, four 28).
template <typename T, int J>
__global__ __launch_bounds__(256) void route_rows_kernel(Routing a) {
  extern __shared__ float lds[];
  const int E = a.E, top = a.top;
  float* s = lds;                          // E logits
  float* best = s + E;                     // groups
  int* open = (int*)(best + a.groups);     // groups
  int* idx = open + a.groups;              // top
  float* wgt = (float*)(idx + top);        // top
  const int t = blockIdx.x, wave = threadIdx.x / WAVE;
  const int lane = threadIdx.x & (WAVE - 1);
  const T* x = (const T*)a.h + (size_t)t * a.width;
  // by vectors of four where all rows lie on whole ones
  const bool whole = a.width % 4 == 0 &&
                     ((uintptr_t)a.h | (uintptr_t)a.w) % (4 * sizeof(T)) == 0;
  for (int e0 = wave; e0 < E; e0 += 4 * J) {
    float acc[J] = {};
    const T* r[J];
#pragma unroll
    for (int j = 0; j < J; ++j)
      r[j] = (const T*)a.w +
             (size_t)(e0 + 4 * j < E ? e0 + 4 * j : e0) * a.width;
    if (whole) {
#pragma unroll 2
      for (int i = lane * 4; i < a.width; i += 4 * WAVE) {
        float f[4], g[J][4];
        load4(x + i, f);
#pragma unroll
        for (int j = 0; j < J; ++j) load4(r[j] + i, g[j]);
#pragma unroll
        for (int j = 0; j < J; ++j)
#pragma unroll
          for (int c = 0; c < 4; ++c) acc[j] += f[c] * g[j][c];
      }
    } else {
      for (int i = lane; i < a.width; i += WAVE)
#pragma unroll
        for (int j = 0; j < J; ++j) acc[j] += to_f(x[i]) * to_f(r[j][i]);
    }
#pragma unroll
    for (int j = 0; j < J; ++j) {
      acc[j] = wave_sum(acc[j]);
      if (lane == 0 && e0 + 4 * j < E) s[e0 + 4 * j] = acc[j];
    }
  }
  __syncthreads();
  if (wave != 0) return;
  choose_experts(s, best, open, E, top, a.groups, a.keep, a.scale, idx, wgt);
  __builtin_amdgcn_wave_barrier();
  for (int k = lane; k < top; k += WAVE) {
    a.index[(size_t)t * top + k] = idx[k];
    a.weight[(size_t)t * top + k] = wgt[k];
    if (a.counts)
      a.pairs[(size_t)idx[k] * a.n_tok + atomicAdd(&a.counts[idx[k]], 1)] =
          t * top + k;
  }
}

extern "C" int hy_route(void* index, void* weight, void* counts, void* pairs,
                        const void* h, const void* w, int width, int E,
                        int top, int groups, int keep, float scale, int n_tok,
                        int dtype, void* stream) {
  const Routing a{(int*)index, (float*)weight, (int*)counts, (int*)pairs, h,
                  w, width, E, top, groups, keep, scale, n_tok};
  if (!routing_ok(a)) return -2;
  if (n_tok <= 0) return 0;
  const hipStream_t st = (hipStream_t)stream;
  if (route_block_ok(a, dtype)) {
    const dim3 grid((n_tok + 15) / 16), block(256);
#define GO(NT)                                                            \
  hipLaunchKernelGGL(route_kernel<NT>, grid, block,                       \
                     4 * route_floats<NT>(E, top, groups), st, a)
    if (E <= 16) GO(1);
    else if (E <= 32) GO(2);
    else GO(4);
#undef GO
  } else {
#define GO(J)                                            \
  HY_DTYPE(dtype, hipLaunchKernelGGL(                    \
      (route_rows_kernel<T, J>), dim3(n_tok), dim3(256), \
      4 * (E + 2 * groups + 2 * top), st, a))
    if (E <= 4) GO(1);
    else if (E <= 8) GO(2);
    else GO(4);
#undef GO
  }
  HY_CHECK();
  return 0;
}
