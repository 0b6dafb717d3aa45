// Causal attention of whole prompts for the Llama family: queries, keys and
// values as the projection left them, rows of a wider matrix.
//
// A workgroup: all heads of one key/value head for neighbouring queries,
// 128 rows (hybrid/flash.h), so that a staged tile serves as many rows as
// there are.  8 x 2048 tokens, 32 heads on 8 of 128: the library's kernel
// took 808 us, this one
// 368 us (750 TFLOP/s).
#include "hybrid/flash.h"

struct PromptAttn {
  bf16_t* out;  // [B][Lq][H][D]
  const bf16_t *q, *k, *v;
  size_t q_batch, k_batch;  // numbers from one sequence to the next
  int ldq, ldk;             // from one token to the next
  int B, H, G, Lq, Lk;      // the last Lq of Lk tokens ask
  float scale;              // in powers of two
};

template <int D>
__global__ __launch_bounds__(256, 2) void prompt_attn_kernel(PromptAttn a,
                                                             int tiles) {
  using F = Flash<D>;
  __shared__ __align__(1024) char lds[F::LDS];
  const int R = a.H / a.G, per = 128 / R;  // queries a workgroup
  // Eight key/value heads of sequences at a time, one an XCD, which gets
  // every eighth workgroup: its L2 serves all tiles.  The tiles of the last
  // ones, fewer than eight, go to all XCDs (16 heads on one of 4096 tokens: on
  // one XCD 527 us, on all 123).  Last queries first: they see most.
  const int pairs = a.B * a.G, whole = (pairs & ~7) * tiles;
  int pair, tile;
  if ((int)blockIdx.x < whole) {
    const int r = blockIdx.x >> 3;
    pair = r / tiles * 8 + (blockIdx.x & 7);
    tile = r % tiles;
  } else {
    const int r = blockIdx.x - whole;
    pair = (pairs & ~7) + r % (pairs & 7);
    tile = r / (pairs & 7);
  }
  const int q0 = (tiles - 1 - tile) * per;
  const int b = pair / a.G, kv = pair % a.G;
  const int n_rows = (a.Lq - q0 < per ? a.Lq - q0 : per) * R;
  const int before = a.Lk - a.Lq + q0;  // position of the first query
  const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);

  F f;
  int qi[2], head[2], pos[2];
  const int span[2] = {a.Lk, a.Lk};
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    int row = wave * 32 + s * 16 + n;
    row = row < n_rows ? row : n_rows - 1;
    qi[s] = q0 + row / R;
    head[s] = kv * R + row % R;
    pos[s] = a.Lk - a.Lq + qi[s];
    const bf16_t* q = a.q + b * a.q_batch + (size_t)qi[s] * a.ldq +
                      (size_t)head[s] * D + g * 8;
#pragma unroll
    for (int k = 0; k < F::KD; ++k)
      f.qf[s][k] = *reinterpret_cast<const u32x4*>(q + k * 32);
  }
  const bf16_t* k0 = a.k + b * a.k_batch + (size_t)kv * D;
  const bf16_t* v0 = a.v + b * a.k_batch + (size_t)kv * D;
  const int last = before + (n_rows - 1) / R;
  const int w_lo = before + wave * 32 / R;
  const int w_hi = before + (wave * 32 + 31) / R;
  f.template run<true>(
      lds,
      paged_rows<D>(
          [&](int j) {
            const size_t at = (size_t)j * a.ldk;
            return KeyRows{k0 + at, v0 + at};
          },
          a.ldk, last),
      0, last, pos, span, w_lo, w_hi, 0, 0, a.scale);
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    if (wave * 32 + s * 16 + n >= n_rows) continue;
    const float by = 1.f / f.l[s];
    bf16_t* to = a.out +
                 (((size_t)b * a.Lq + qi[s]) * a.H + head[s]) * D + g * 4;
#pragma unroll
    for (int v = 0; v < F::VT; ++v)
      *reinterpret_cast<uint2*>(to + v * 16) =
          make_uint2(to_bf16x2(f.o[s][v][0] * by, f.o[s][v][1] * by),
                     to_bf16x2(f.o[s][v][2] * by, f.o[s][v][3] * by));
  }
}

// -2: not for this kernel
extern "C" int ll_prompt_attn(void* out, const void* q, const void* k,
                              const void* v, long long q_batch,
                              long long k_batch, int ldq, int ldk, int B,
                              int H, int G, int Lq, int Lk, int D,
                              float scale, void* stream) {
  if (B < 0 || G <= 0 || H <= 0 || H % G || H / G > 128 || Lq < 0 ||
      Lk < Lq || ldq % 8 || ldk % 8 || q_batch % 8 || k_batch % 8 ||
      !(scale > 0.f) ||
      (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v) % 16) ||
      (uintptr_t)out % 8)
    return -2;
  if (D != 64 && D != 128) return -2;
  if (B == 0 || Lq == 0) return 0;
  const int per = 128 / (H / G), tiles = (Lq + per - 1) / per;
  const long long groups = (long long)B * G * tiles;
  if (groups >= (1ll << 31)) return -2;
  const PromptAttn a{(bf16_t*)out, (const bf16_t*)q, (const bf16_t*)k,
                     (const bf16_t*)v, (size_t)q_batch, (size_t)k_batch, ldq,
                     ldk, B, H, G, Lq, Lk, scale * LOG2E};
  hipStream_t st = (hipStream_t)stream;
  if (D == 128)
    hipLaunchKernelGGL(prompt_attn_kernel<128>, dim3((unsigned)groups),
                       dim3(256), 0, st, a, tiles);
  else
    hipLaunchKernelGGL(prompt_attn_kernel<64>, dim3((unsigned)groups),
                       dim3(256), 0, st, a, tiles);
  HY_CHECK();
  return 0;
}
