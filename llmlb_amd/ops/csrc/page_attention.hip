// Attention of single tokens over a paged cache (Llama family): bf16 pages
// of 64 or 128 numbers a head, or e4m3 pages of 128 with a scale per row.
//
//   out[s] = softmax(q[s] K^T scale) V,  K and V in pages of 16 rows
//
// What bounds it is reading the pages once.  One workgroup per sequence,
// key/value head, up to 16 of its query heads and part of the pages: the
// heads are the columns of the matrix cores' tiles, so a page is read from
// LDS once for all of them.  Its four or eight waves work on pages of their
// own, two at a time, without a barrier: pages are whole runs of memory,
// copied to LDS and waited for by the wave that asked.  What hides the wait is
// other waves, eight or more to a compute unit (a second stage of LDS in their
// place was no faster), and the wave's own other half: the next keys are on their
// way while values are worked on, the next values while keys are (us, both waited
// for at once -> this: 64 sequences of 675 to 900 tokens 40.1 -> 38.6, 32 of 1500 to
// 2000 e4m3 25.5 -> 24.2, 8 of 1000 12.7 -> 11.2, 10 of 100 6.6 -> 6.4).  Weights and
// sums stay floats: a weight enters its product as the sum of three bf16 numbers,
// which are all of its 24 bits.
//
// Sequences use as many parts as their length fills (16 pages each), which
// the host does not know: the rest of the grid ends at once, and where one
// part is all, it writes the result itself.
//
// Against a lane per part of a row, us (sequences, heads, tokens):
//   bf16, 32 on 8 heads of 128: 64 x 675 to 900 76 -> 39 (5.5 TB/s),
//     64 x 3600 255 -> 156 (6.2 TB/s), 1 x 4000 47 -> 16
//   e4m3, the same heads: 64 x 900 70 -> 21; 32 x 2048 in two parts 28, in
//     one of eight waves 25 (5.6 TB/s), 128 x 1500 56.  Values leave LDS as
//     columns of bytes and are widened in registers; widened on a way back
//     through LDS 24, 29 (two parts) and 71, by two conversions to float and
//     a permutation 22, 28.5 and 58
//   bf16, 16 on 4 heads of 64: 64 x 900 61 -> 15, 1 x 100 12.3 -> 5.5
#include "hybrid/lds_copy.h"
#include "hybrid/mfma.h"

#define PARTS_PAGES 16  // pages that are worth a part

// 64 lanes copy 4 bytes each to 256 bytes of LDS
__device__ __forceinline__ void copy4_to_lds(const void* src, unsigned to) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off"
               ::"s"(__builtin_amdgcn_readfirstlane(to)), "v"(src)
               : "memory");
}

__device__ __forceinline__ int parts_used(int len, int parts) {
  const int n = ((len + PAGE - 1) / PAGE + PARTS_PAGES - 1) / PARTS_PAGES;
  return n < 1 ? 1 : (n < parts ? n : parts);
}

// e4m3 to bf16, exactly
__device__ __forceinline__ u32x4 widen8(uint2 v) {
  u32x4 r;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const unsigned x = i ? v.y : v.x;
    r[2 * i] = __builtin_bit_cast(
        unsigned, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(x, 1.f, false));
    r[2 * i + 1] = __builtin_bit_cast(
        unsigned, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(x, 1.f, true));
  }
  return r;
}

// A wave's place in LDS: two pages of keys, two of values
template <int D, bool FP8, int W>
struct PageAttn {
  static constexpr int ROW = D * (FP8 ? 1 : 2), BYTES = PAGE * ROW;
  static constexpr int PR = ROW / 16, CP = BYTES / 1024;  // pieces, copies
  static constexpr int STAGE = 4 * BYTES + (FP8 ? 256 : 0);  // and scales
  static constexpr int OP = D + 4;  // row of the waves' results
  static constexpr int RESULTS = W * 16 * OP * 4;
  static constexpr int LDS = W * STAGE > RESULTS ? W * STAGE : RESULTS;
};

// Piece c of row r lies at c ^ turn(r): lanes reading one piece of 16 rows
// meet every bank once.
template <int ROW>
__device__ __forceinline__ int turn(int r) {
  return ROW == 256 ? r & 15 : (r >> 1) & 7;
}

// acc [n][heads][parts][D], ml [n][heads][parts] (maximum, sum)
template <int D, bool FP8, int W>
__global__ __launch_bounds__(W * 64, 3) void page_attn_kernel(
    bf16_t* __restrict__ out, float* __restrict__ ws_acc,
    float* __restrict__ ws_ml, const bf16_t* __restrict__ q, int ldq,
    const char* __restrict__ kc, const char* __restrict__ vc,
    const float* __restrict__ k_scale, const float* __restrict__ v_scale,
    const int* __restrict__ bt, const int* __restrict__ lens, int max_blocks,
    int H, int G, int parts, float scale) {
  using A = PageAttn<D, FP8, W>;
  constexpr int KD = D / 32, VT = D / 16;
  extern __shared__ __align__(1024) char lds[];
  __shared__ float lm[W][16], ll[W][16];
  const int R = H / G, ht = (R + 15) / 16;
  const int seq = blockIdx.x, part = blockIdx.z;
  const int kv = blockIdx.y / ht, h0 = blockIdx.y % ht * 16;
  const int len = lens[seq];
  const int used = parts_used(len, parts);
  if (part >= used) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int n = lane & 15, g = lane >> 4;
  const int heads = R - h0 < 16 ? R - h0 : 16;

  // pairs of pages of this part, every W-th of this wave
  const int pages = (len + PAGE - 1) / PAGE, pairs = (pages + 1) / 2;
  const int per = (pairs + used - 1) / used;
  const int first = part * per + wave;
  const int stop = part * per + per < pairs ? part * per + per : pairs;
  const int count = first < stop ? (stop - first + W - 1) / W : 0;
  char* const st = lds + wave * A::STAGE;
  const unsigned to = lds_byte(st);
  const int* const row = bt + (size_t)seq * max_blocks;

  // pages of 32 pairs, in lanes
  int ids = 0;
  auto look_up = [&](int i) {
    const int p = 2 * (first + (i + lane / 2) * W) + (lane & 1);
    ids = row[p < pages ? p : pages - 1];
    asm volatile("" : "+v"(ids));  // waited for here, and not by every pass
  };
  // source of lane's piece in copy j of a page
  int off[A::CP];
#pragma unroll
  for (int j = 0; j < A::CP; ++j) {
    const int r = j * (1024 / A::ROW) + lane / A::PR;
    off[j] = r * A::ROW + (((lane % A::PR) ^ turn<A::ROW>(r)) * 16);
  }
  // keys of pair i, with the scales of both, and values
  auto copy = [&](int i, bool values) {
    const char* const from = values ? vc : kc;
    const unsigned there = to + (values ? 2 : 0) * A::BYTES;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int page = __builtin_amdgcn_readlane(ids, 2 * (i % 32) + t);
      const size_t at = ((size_t)page * G + kv) * A::BYTES;
#pragma unroll
      for (int j = 0; j < A::CP; ++j)
        stream_to_lds(
            reinterpret_cast<const bf16_t*>(
                from + at + (FP8 && t && values ? off[j] ^ 64 : off[j])),
            there + t * A::BYTES + j * 1024);
    }
    if (FP8 && !values) {  // 16 of each page's keys, then of the values
      const int page =
          g & 1 ? __builtin_amdgcn_readlane(ids, 2 * (i % 32) + 1)
                : __builtin_amdgcn_readlane(ids, 2 * (i % 32));
      const float* s = g < 2 ? k_scale : v_scale;
      copy4_to_lds(s + ((size_t)page * G + kv) * PAGE + n,
                   to + 4 * A::BYTES);
    }
  };

  // Queries come with the page numbers: waited for later, they would make every
  // pass of the loop wait for all copies.  (Columns past the heads are the first
  // once more.)
  u32x4 qf[KD];
#pragma unroll
  for (int k = 0; k < KD; ++k)
    qf[k] = *reinterpret_cast<const u32x4*>(
        q + (size_t)seq * ldq +
        (size_t)(kv * R + h0 + (n < heads ? n : 0)) * D + k * 32 + g * 8);
  f32x4 o[VT];
  float m = -1e30f, l = 0.f;
#pragma unroll
  for (int v = 0; v < VT; ++v) o[v] = f32x4{0.f, 0.f, 0.f, 0.f};
  // copies of a pair's values, and of its keys
  constexpr int VALUES = 2 * A::CP, KEYS = VALUES + (FP8 ? 1 : 0);
  if (count) look_up(0);
#pragma unroll
  for (int k = 0; k < KD; ++k) asm volatile("" : "+v"(qf[k]));
  if (count) {
    copy(0, false);
    copy(0, true);
  }
  for (int i = 0; i < count; ++i) {
    wait_copies<VALUES>();  // the keys are there
    const int j0 = (first + i * W) * 32;  // the pair's first key
    const bool more = i + 1 < count;
    f32x4 s[2], v_by[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      s[t] = f32x4{0.f, 0.f, 0.f, 0.f};
      const char* k_row = st + t * A::BYTES + n * A::ROW;
#pragma unroll
      for (int k = 0; k < KD; ++k) {
        u32x4 kf;
        if (FP8) {
          const int c = 2 * k + (g >> 1);
          kf = widen8(*reinterpret_cast<const uint2*>(
              k_row + (c ^ turn<A::ROW>(n)) * 16 + (g & 1) * 8));
        } else {
          kf = *reinterpret_cast<const u32x4*>(
              k_row + ((k * 4 + g) ^ turn<A::ROW>(n)) * 16);
        }
        s[t] = mfma(kf, qf[k], s[t]);
      }
      f32x4 by = {scale, scale, scale, scale};
      if (FP8) {
        const char* const scales = st + 4 * A::BYTES + t * 64 + g * 16;
        by *= *reinterpret_cast<const f32x4*>(scales);
        v_by[t] = *reinterpret_cast<const f32x4*>(scales + 128);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r)
        s[t][r] = j0 + t * 16 + g * 4 + r < len ? s[t][r] * by[r] : -INFINITY;
    }
    // all keys have been read before the next ones' copies start
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (more) {
      if ((i + 1) % 32 == 0) look_up(i + 1);
      copy(i + 1, false);
    }
    float mx = m;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) mx = fmaxf(mx, s[t][r]);
    mx = fmaxf(mx, __shfl_xor(mx, 16, WAVE));
    mx = fmaxf(mx, __shfl_xor(mx, 32, WAVE));
    if (__any(mx > m)) {  // seldom after the first pages
      const float keep = __builtin_amdgcn_exp2f(m - mx);
      m = mx;
      l *= keep;
#pragma unroll
      for (int v = 0; v < VT; ++v) o[v] *= keep;
    }
    if (more)
      wait_copies<KEYS>();
    else
      wait_copies<0>();
    if (j0 + 32 > len) {
      // rows past the end: an earlier sequence may have left anything there
      const int r = lane / 2;
      if (j0 + r >= len)
#pragma unroll
        for (int c = 0; c < A::ROW / 32; ++c)
          *reinterpret_cast<uint4*>(st + 2 * A::BYTES + r * A::ROW +
                                    (lane & 1) * (A::ROW / 2) + c * 16) =
              make_uint4(0, 0, 0, 0);
    }
    u32x4 hi, mid, lo;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      f32x4 p;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        p[r] = __builtin_amdgcn_exp2f(s[t][r] - m);
        l += p[r];
      }
      if (FP8) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          p[r] = j0 + t * 16 + g * 4 + r < len ? p[r] * v_by[t][r] : 0.f;
      }
#pragma unroll
      for (int r = 0; r < 4; r += 2) {
        unsigned h, m2, l2;
        split3(p[r], p[r + 1], h, m2, l2);
        hi[2 * t + r / 2] = h;
        mid[2 * t + r / 2] = m2;
        lo[2 * t + r / 2] = l2;
      }
    }
    const char* const values = st + 2 * A::BYTES;
    // columns of four keys of either page: of e4m3 at once, and those of the
    // second page lie turned by four pieces more, in the other banks
    const int t = FP8 ? n >> 3 : 0;
    const int r = g * 4 + (FP8 ? n >> 1 & 3 : n >> 2);
    const char* const v_row = values + t * A::BYTES + r * A::ROW;
#pragma unroll
    for (int v = 0; v < VT; ++v) {
      u32x4 vf;
      if (FP8) {
        vf = widen8(load_byte_columns(
            v_row + (v ^ turn<A::ROW>(r) ^ t * 4) * 16 + (n & 1) * 8));
      } else {
        const int c = 2 * v + ((n >> 1) & 1);
        vf = load_columns(
            reinterpret_cast<const unsigned short*>(
                v_row + (c ^ turn<A::ROW>(r)) * 16 + (n & 1) * 8),
            PAGE * D);
      }
      o[v] = mfma(vf, hi, o[v]);
      o[v] = mfma(vf, mid, o[v]);
      o[v] = mfma(vf, lo, o[v]);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (more) copy(i + 1, true);
  }

  l += __shfl_xor(l, 16, WAVE);
  l += __shfl_xor(l, 32, WAVE);
  if (g == 0) {
    lm[wave][n] = m;
    ll[wave][n] = l;
  }
  __syncthreads();  // the results lie where the stages were
  float* const res = reinterpret_cast<float*>(lds);
  if (n < heads) {
#pragma unroll
    for (int v = 0; v < VT; ++v)
      *reinterpret_cast<f32x4*>(
          &res[(wave * 16 + n) * A::OP + v * 16 + g * 4]) = o[v];
  }
  __syncthreads();
  for (int i = tid; i < heads * (D / 4); i += W * 64) {
    const int h = i / (D / 4), c = i % (D / 4) * 4;
    float top = lm[0][h], sum = 0.f;
#pragma unroll
    for (int w = 1; w < W; ++w) top = fmaxf(top, lm[w][h]);
    f32x4 x = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < W; ++w) {
      const float f = __builtin_amdgcn_exp2f(lm[w][h] - top);
      sum += f * ll[w][h];
      x += *reinterpret_cast<const f32x4*>(&res[(w * 16 + h) * A::OP + c]) * f;
    }
    const size_t at = (size_t)seq * H + kv * R + h0 + h;
    if (used == 1) {
      const float f = sum > 0.f ? 1.f / sum : 0.f;
      *reinterpret_cast<uint2*>(out + at * D + c) =
          make_uint2(to_bf16x2(x[0] * f, x[1] * f),
                     to_bf16x2(x[2] * f, x[3] * f));
    } else {
      *reinterpret_cast<f32x4*>(ws_acc + (at * parts + part) * D + c) = x;
      if (c == 0) {
        ws_ml[(at * parts + part) * 2] = top;
        ws_ml[(at * parts + part) * 2 + 1] = sum;
      }
    }
  }
}

// Joins the parts of sequences that used several; D / 4 lanes a head, each
// with one part's weight.  Four parts are asked for at a time, the first before
// the weights are there: what bounds this is a chain of loads.  us of attention
// with parts, loads one after the other -> now: 32 heads on 8 of 128, 8
// sequences of 1000 tokens 11.7 -> 10.8, 16 of 2048 25.2 -> 24.4; 16 on 4 of 64,
// 4 of 3000 11.5 -> 8.8.
template <int D>
__global__ __launch_bounds__(256) void page_join_kernel(
    bf16_t* __restrict__ out, const float* __restrict__ ws_acc,
    const float* __restrict__ ws_ml, const int* __restrict__ lens, int n_rows,
    int H, int parts) {
  constexpr int LANES = D / 4;
  const int lane = threadIdx.x % LANES;
  const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 4;
  const size_t at = i / D;
  if (at >= (size_t)n_rows * H) return;
  const int used = parts_used(lens[at / H], parts);
  if (used == 1) return;
  const float2* ml = reinterpret_cast<const float2*>(ws_ml) + at * parts;
  const float* acc = ws_acc + at * parts * D + i % D;
  f32x4 part[4];
  auto ask = [&](int p0) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int p = p0 + j < used ? p0 + j : used - 1;
      part[j] = *reinterpret_cast<const f32x4*>(acc + (size_t)p * D);
    }
  };
  ask(0);
  float top = -1e30f, sum = 0.f;
  for (int p = lane; p < used; p += LANES) top = fmaxf(top, ml[p].x);
#pragma unroll
  for (int k = LANES / 2; k; k >>= 1)
    top = fmaxf(top, __shfl_xor(top, k, LANES));
  f32x4 x = {0.f, 0.f, 0.f, 0.f};
  float w = 0.f, l = 0.f;
  for (int p0 = 0; p0 < used; p0 += 4) {
    if (p0 % LANES == 0) {
      const float2 v = ml[p0 + lane < used ? p0 + lane : used - 1];
      w = __builtin_amdgcn_exp2f(v.x - top);
      l = v.y;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (p0 + j >= used) break;
      const float f = __shfl(w, (p0 + j) % LANES, LANES);
      sum += f * __shfl(l, (p0 + j) % LANES, LANES);
      x += part[j] * f;
    }
    if (p0 + 4 < used) ask(p0 + 4);
  }
  const float f = sum > 0.f ? 1.f / sum : 0.f;
  *reinterpret_cast<uint2*>(out + i) = make_uint2(
      to_bf16x2(x[0] * f, x[1] * f), to_bf16x2(x[2] * f, x[3] * f));
}

template <int D, bool FP8, int W>
static int page_attn_launch(void* out, void* acc, void* ml, const void* q,
                            int ldq, const void* kc, const void* vc,
                            const void* ks, const void* vs, const void* bt,
                            const void* lens, int n, int max_blocks, int H,
                            int G, int parts, float scale, hipStream_t st) {
  constexpr int lds = PageAttn<D, FP8, W>::LDS;
  static_assert(lds + W * 128 <= 160 * 1024, "LDS of a compute unit");
  static const hipError_t sized = hipFuncSetAttribute(
      reinterpret_cast<const void*>(page_attn_kernel<D, FP8, W>),
      hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (sized != hipSuccess) return -1;
  const int tiles = G * ((H / G + 15) / 16);
  hipLaunchKernelGGL((page_attn_kernel<D, FP8, W>), dim3(n, tiles, parts),
                     dim3(W * 64), lds, st, (bf16_t*)out, (float*)acc,
                     (float*)ml, (const bf16_t*)q, ldq, (const char*)kc,
                     (const char*)vc, (const float*)ks, (const float*)vs,
                     (const int*)bt, (const int*)lens, max_blocks, H, G,
                     parts, scale * LOG2E);
  HY_CHECK();
  if (parts == 1) return 0;
  const size_t threads = (size_t)n * H * (D / 4);
  hipLaunchKernelGGL(page_join_kernel<D>,
                     dim3((unsigned)((threads + 255) / 256)), dim3(256), 0,
                     st, (bf16_t*)out, (const float*)acc, (const float*)ml,
                     (const int*)lens, n, H, parts);
  HY_CHECK();
  return 0;
}

// q [n, H, D] with rows ldq apart; caches [pages, G, 16, D], e4m3 where
// scales are given; acc and ml for ``parts`` parts, unused by one.
// -2: not for this kernel.
extern "C" int ll_page_attn(void* out, void* acc, void* ml, const void* q,
                            int ldq, const void* kc, const void* vc,
                            const void* ks, const void* vs, const void* bt,
                            const void* lens, int n, int max_blocks, int H,
                            int G, int D, int block_size, int parts,
                            float scale, void* stream) {
  if (n < 0 || G <= 0 || H <= 0 || H % G || block_size != PAGE || parts < 1 ||
      parts > 65535 || (parts > 1 && (!acc || !ml)) || ldq % 8 ||
      (uintptr_t)q % 16 || G * ((H / G + 15) / 16) > 65535)
    return -2;
  if ((ks != nullptr) != (vs != nullptr) || (ks && D != 128)) return -2;
  if (n == 0) return 0;
  hipStream_t st = (hipStream_t)stream;
  // Two parts of four waves are one of eight, with no results to join, where
  // whole ones leave compute units idle no longer than halves do.  Two parts
  // -> one, us, 32 sequences of 2048 and of up to 300 tokens, 32 heads on 8 of
  // 128: bf16 46.2 -> 43.5, 12.6 -> 9.1; e4m3 27.8 -> 24.9, 9.0 -> 6.6; 64 of
  // 3000, 16 on 4 of 64: 29.9 -> 27.8.  Eight waves of bf16 heads of 128 fill a
  // compute unit's LDS, and past one round a long sequence among short ones
  // waits for what its halves would share (50 sequences of 100 tokens, one of
  // 8000: 54.5 -> 74.6; all of 1000 39.2 -> 36.7): two parts there.
  const long long count = (long long)n * G * ((H / G + 15) / 16);
  const bool whole =
      parts == 2 && (count + 255) / 256 * 2 <= (2 * count + 255) / 256 &&
      (count <= 256 || D < 128 || ks);
#define PAGE_ATTN(D, FP8)                                                    \
  do {                                                                       \
    if (whole)                                                               \
      return page_attn_launch<D, FP8, 8>(out, acc, ml, q, ldq, kc, vc, ks,   \
                                         vs, bt, lens, n, max_blocks, H, G,  \
                                         1, scale, st);                      \
    return page_attn_launch<D, FP8, 4>(out, acc, ml, q, ldq, kc, vc, ks, vs, \
                                       bt, lens, n, max_blocks, H, G, parts, \
                                       scale, st);                           \
  } while (0)
  if (ks) PAGE_ATTN(128, true);
  if (D == 128) PAGE_ATTN(128, false);
  if (D == 64) PAGE_ATTN(64, false);
#undef PAGE_ATTN
  return -2;
}
