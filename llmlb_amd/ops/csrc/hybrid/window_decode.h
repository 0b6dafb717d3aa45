// Attention of single tokens over their windows (window_mfma.hip).
#pragma once
#include "flash.h"
#include "paged_tiles.h"

struct WindowDecode {
  bf16_t* out;
  int ld_out;
  float* acc;  // parts > 1: [N][H][parts][V]
  float* ml;   // [N][H][parts] (maximum, sum)
  const bf16_t* proj;
  int ld, g_off;
  const bf16_t* cache;
  const int* pos;
  const int* row;
  const int* bt;
  int max_blocks, H, G, D, V;
  Mask mask;
  int parts;
};
// joins the parts where there are several (window_mfma.hip); 0: done
int window_merge(const WindowDecode& a, int n_rows, hipStream_t stream);
// operands of the kernels
__host__ inline bool window_ok(int ld, int ld_out, int H, int G, int D, int V,
                               int window) {
  return G > 0 && H > 0 && H % G == 0 && D > 0 && V > 0 && D % 8 == 0 &&
         V % 8 == 0 && D <= 256 && V <= 256 && ld % 8 == 0 &&
         ld_out % 8 == 0 && window >= 1;
}
#define PARTS_MAX 64
__host__ inline bool window_decode_ok(const WindowDecode& a) {
  return window_ok(a.ld, a.ld_out, a.H, a.G, a.D, a.V, a.mask.size) &&
         a.parts >= 1 && a.parts <= PARTS_MAX &&
         (a.parts == 1 || (a.acc && a.ml)) &&
         a.G * ((a.H / a.G + 15) / 16) <= 65535;
}

// Single tokens.  One workgroup: one query, up to 16 heads of one
// key/value head, one part of its window.  Each wave scores 16 of a
// tile's 64 keys, the weights go through LDS, and each wave accumulates a
// quarter of the value columns.
//   acc [N][H][parts][V], ml [N][H][parts] (maximum, sum); one part: the
//   output itself
// groups: how many workgroups there are
// ONCE: no other workgroup reads the head's keys, which then go past the
// caches and leave them to what the next kernels read: 8 layers of 61
// sequences from 777 tokens, 32 heads of 128, 1382 -> 1354 us a step of the
// model, of 64 sequences from 1024, 16 heads of 64, 507 -> 497.
// Two tiles are on their way while one is worked on, which is why tiles come
// in twos (loads that come and go are not waited for by count): one tile ahead
// 8 layers' attention beside their experts' first products, 61 sequences, took
// 78.8 us a layer, this way 74.9.  Heads of up to 64 gain by it only where units
// have several workgroups of four tiles or more, whose keys nobody else reads;
// larger ones than 128 have no registers for it.  us, one ahead, two ahead (of one
// tile, with a second one without weights) and as chosen:
//   heads     sequences, keys: 1, 64          1, 192         64, 192       64, 778
//   128 x 128, 4 a key's     4.9, 5.6, 4.4  7.8, 8.0, 6.8  8.7, 8.9, 7.7  18.8, 16.1, 15.4
//   64 x 64, 4 a key's       3.7, 5.2, 3.7  5.4, 7.0, 5.5  6.5, 7.6, 5.8  19.4, 17.2, 16.5
//   32 x 32, 1 a key's       3.5, 4.6, 3.5  5.1, 6.2, 5.1  6.3, 7.7, 6.0  18.9, 17.5, 17.1
//   256 x 256, 4 a key's     5.9, 8.1, 4.8  10.7, 12.1, 8.3  12.0, 14.3, 10.0  29.0, 29.0, 25.7
template <int DQ, int DV>
struct __align__(16) WindowLds {
  using St = Stage<1, DQ, DV>;
  unsigned short lk[64 * St::KP];
  unsigned short lv[64 * St::VP];
  unsigned short lp[16 * (64 + 8)];
  float lmax[16][4], lsum[16][4];
};
template <int DQ, int DV, bool ONCE>
__device__ __forceinline__ void window_decode_block(
    const WindowDecode& a, int q, int y, int part, int groups,
    WindowLds<DQ, DV>& lds) {
  constexpr int KD = DQ / 32, NV = DV / 64, PP = 64 + 8;
  using St = Stage<1, DQ, DV>;
  unsigned short *lk = lds.lk, *lv = lds.lv, *lp = lds.lp;
  auto &lmax = lds.lmax, &lsum = lds.lsum;
  const int H = a.H, G = a.G, D = a.D, V = a.V, parts = a.parts;
  const bf16_t* proj = a.proj;
  const Mask mask = a.mask;
  const int R = H / G, ht = (R + 15) / 16;
  const int kv = y / ht, h0 = y % ht * 16;
  const int tid = threadIdx.x, wave = tid / WAVE, lane = tid & 63;
  const int n = lane & 15, g = lane >> 4;
  const int pos = a.pos[q];
  const int h = kv * R + h0 + n;  // this lane's head
  const bool real = h0 + n < R;

  const int span = mask.span(pos);
  const int lo = mask.first(pos) & ~(PAGE - 1);
  const int tiles = (pos - lo) / 64 + 1;
  const int per = (tiles + parts - 1) / parts;
  const int t_lo = part * per;
  const int t_hi = t_lo + per < tiles ? t_lo + per : tiles;

  St st(a.cache, a.bt + (size_t)a.row[q] * a.max_blocks, G, kv, D, V, pos);
  u32x4 pk[2][St::KL], pv[2][St::VL];
  int pg[2][4];
  constexpr bool NEVER = DQ > 128 || DV > 128 || (!ONCE && DQ <= 64);
  constexpr bool WIDE = DQ > 64 && DV > 64;
  const int some = t_hi - t_lo;
  const bool two =
      !NEVER && (WIDE ? ONCE || some > 1 : groups >= 256 && some >= 4);
  auto ask = [&](int t, int s) {
    st.template ask<ONCE>(pg[s], pk[s], pv[s], t < t_hi);
  };
  st.fetch_pages(lo + t_lo * 64, pg[0]);
  if (two) {
    st.fetch_pages(lo + t_lo * 64 + 64, pg[1]);
    ask(t_lo, 0);
    ask(t_lo + 1, 1);
    st.fetch_pages(lo + t_lo * 64 + 128, pg[0]);
    st.fetch_pages(lo + t_lo * 64 + 192, pg[1]);
  } else {
    ask(t_lo, 0);
    st.fetch_pages(lo + t_lo * 64 + 64, pg[0]);
  }
  u32x4 qf[KD];
#pragma unroll
  for (int k = 0; k < KD; ++k) {
    const int d = k * 32 + g * 8;
    qf[k] = u32x4{0, 0, 0, 0};
    if (d < D && real)
      qf[k] = *reinterpret_cast<const u32x4*>(proj + (size_t)q * a.ld +
                                              (size_t)h * D + d);
  }
  // what the sum is multiplied with to gate
  float z = 1.f;
  if (real && a.g_off >= 0)
    z += __expf(-to_f(proj[(size_t)q * a.ld + a.g_off + h]));

  f32x4 o[NV];
  float m = -1e30f, l = 0.f;
#pragma unroll
  for (int v = 0; v < NV; ++v) o[v] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto tile = [&](int t, int set, auto next) {
#pragma unroll
    for (int i = 0; i < St::VL; ++i)  // hidden here, not where asked for
      asm volatile("" : "+v"(pv[set][i]));
    st.hide(lo + t * 64, pv[set], t < t_hi);
    St::store(lk, lv, pk[set], pv[set]);
    __syncthreads();
    next(t, set);
    const int j = lo + t * 64 + wave * 16 + g * 4;
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < KD; ++k)
      s = mfma(*reinterpret_cast<const u32x4*>(
                   &lk[(wave * 16 + n) * St::KP + k * 32 + g * 8]),
               qf[k], s);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      s[i] = t < t_hi && (unsigned)(pos - j - i) <= (unsigned)span ? s[i] : -INFINITY;
    float mx = fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]));
    mx = fmaxf(mx, __shfl_xor(mx, 16, WAVE));
    mx = fmaxf(mx, __shfl_xor(mx, 32, WAVE));
    if (g == 0) lmax[n][wave] = mx;
    __syncthreads();
    mx = m;
#pragma unroll
    for (int i = 0; i < 4; ++i) mx = fmaxf(mx, lmax[n][i]);
    const float keep = __builtin_amdgcn_exp2f(m - mx);
    m = mx;
    l *= keep;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      s[i] = __builtin_amdgcn_exp2f(s[i] - m);
      l += s[i];
    }
    *reinterpret_cast<uint2*>(&lp[n * PP + wave * 16 + g * 4]) =
        make_uint2(to_bf16x2(s[0], s[1]), to_bf16x2(s[2], s[3]));
    __syncthreads();
#pragma unroll
    for (int v = 0; v < NV; ++v) o[v] *= keep;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const u32x4 pf = *reinterpret_cast<const u32x4*>(
          &lp[n * PP + ks * 32 + g * 8]);
#pragma unroll
      for (int v = 0; v < NV; ++v)
        o[v] = mfma(load_columns(&lv[(ks * 32 + g * 8 + (n >> 2)) * St::VP +
                                     (wave * NV + v) * 16 + (n & 3) * 4],
                                 4 * St::VP),
                    pf, o[v]);
    }
    __syncthreads();
  };
  if (two) {
    auto next = [&](int t, int set) {
      ask(t + 2, set);
      st.fetch_pages(lo + t * 64 + 256, pg[set]);
    };
    for (int t = t_lo; t < t_hi; t += 2) {
      tile(t, 0, next);
      if (t + 1 >= t_hi) break;
      tile(t + 1, 1, next);
    }
  } else {
    for (int t = t_lo; t < t_hi; ++t)
      tile(t, 0, [&](int t, int) {
        if (t + 1 >= t_hi) return;
        ask(t + 1, 0);
        st.fetch_pages(lo + t * 64 + 128, pg[0]);
      });
  }
  l += __shfl_xor(l, 16, WAVE);
  l += __shfl_xor(l, 32, WAVE);
  if (g == 0) lsum[n][wave] = l;
  __syncthreads();
  if (!real) return;
  l = lsum[n][0] + lsum[n][1] + lsum[n][2] + lsum[n][3];
  if (parts == 1) {
    const float f = 1.f / (l * z);
    bf16_t* dst = a.out + (size_t)q * a.ld_out + (size_t)h * V;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const int d = (wave * NV + v) * 16 + g * 4;
      if (d < V)
        *reinterpret_cast<uint2*>(dst + d) =
            make_uint2(to_bf16x2(o[v][0] * f, o[v][1] * f),
                       to_bf16x2(o[v][2] * f, o[v][3] * f));
    }
    return;
  }
  const size_t at = ((size_t)q * H + h) * parts + part;
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    const int d = (wave * NV + v) * 16 + g * 4;
    if (d < V)
      *reinterpret_cast<float4*>(a.acc + at * V + d) =
          make_float4(o[v][0], o[v][1], o[v][2], o[v][3]);
  }
  if (wave == 0 && g == 0) {
    a.ml[at * 2] = m;
    a.ml[at * 2 + 1] = l;
  }
}
