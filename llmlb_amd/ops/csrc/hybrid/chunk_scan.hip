// Prompt portions of the recurrences with a decay per key channel (gated
// linear attention, see linear_scan.hip; gated delta rule, see
// channel_delta.hip) on the matrix cores, 16 tokens at a time.
//
// With F(s, t) the product of the decays after token s up to token t, of a
// chunk's tokens 0 .. 15, and S the state before it, both are
//   o_t = S^T (q_t F(-1, t)) + sum over s <= t of Q_ts u_s,
//   S  <- F(-1, 15) S + sum over s of (k_s F(s, 15)) u_s^T,
//   Q_ts = sum over channels of q_t k_s F(s, t),
// with u = v for gated linear attention, and for the delta rule
//   u = (I + L)^-1 beta (v - S^T (k F(-1, .))),   L_ts = beta_t K_ts (s < t),
// K being Q with k_t for q_t.  The inverse is made by substitution.
//
// Q and K are products of factors if F(s, t) is taken apart at a token
// between the two: of every 2 B tokens, B = 8, 4, 2, 1, the second half asks
// the first, with the decays of the one from its start on and of the other up
// to its end.  Those are products of decays as they come, by halves that
// double: nothing is divided by a decay, and one may be as small as it likes.
// B = 8 and 4 go to the matrix cores; 2 and 1 are a few pairs within lanes
// next to each other, and are summed where the factors are made.
//
// All is float, as token by token: the products are those of the matrix cores
// for floats (16x16x4).  (As sums of two bf16 numbers their results were off
// by 5e-6 and 7e-6 of their size; now 2e-7, token by token 3e-7.)
//
// Bound by the chain from chunk to chunk.  Waves carry the state, 16 value
// columns each, and work on one chunk while others make what it takes of the
// next ones: the factors, Q and K of them, the inverse.  They meet once a
// chunk, and a chunk takes about as long as what the waves of one SIMD issue
// for it.  8 x 2048 tokens, heads of 128 x 128, us, token by token -> now:
// delta rule, 16 heads, 973 -> 497; gated linear attention, 32 heads, 889
// -> 490.
#include "common.h"
#include "mfma.h"
#include <type_traits>

#define CHUNK 16

template <int A, int B, int C, int D>
__device__ __forceinline__ float quad_lanes(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(
      0, __float_as_int(x), A | B << 2 | C << 4 | D << 6, 0xf, 0xf, true));
}
// x *= by of lane LANE of every 16, in the fours of lanes that BANKS names
template <int LANE, int BANKS>
__device__ __forceinline__ void times_lane(f32x4& x, f32x4 by) {
  float a = x[0], b = x[1], c = x[2], d = x[3];
  // (a number is read from another lane two instructions after it is made)
  asm("s_nop 1\n\t"
      "v_mul_f32_dpp %0, %4, %0 row_newbcast:%8 row_mask:0xf bank_mask:%9\n\t"
      "v_mul_f32_dpp %1, %5, %1 row_newbcast:%8 row_mask:0xf bank_mask:%9\n\t"
      "v_mul_f32_dpp %2, %6, %2 row_newbcast:%8 row_mask:0xf bank_mask:%9\n\t"
      "v_mul_f32_dpp %3, %7, %3 row_newbcast:%8 row_mask:0xf bank_mask:%9"
      : "+v"(a), "+v"(b), "+v"(c), "+v"(d)
      : "v"(by[0]), "v"(by[1]), "v"(by[2]), "v"(by[3]), "n"(LANE),
        "n"(BANKS));
  x = f32x4{a, b, c, d};
}
// four sums over the 16-lane rows, row i with the i-th
__device__ __forceinline__ float by_rows(const float (&x)[4]) {
  auto halves = [](float a, float b) {  // rows a0 + a1, b0 + b1, a2 + a3, ..
    const auto r = __builtin_amdgcn_permlane16_swap(
        __float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
  };
  const auto r = __builtin_amdgcn_permlane32_swap(
      __float_as_uint(halves(x[0], x[1])),
      __float_as_uint(halves(x[2], x[3])), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// c += a^T b for 16 x 16 results and four numbers a lane of the contraction
__device__ __forceinline__ f32x4 mfma4(f32x4 a, f32x4 b, f32x4 c) {
#pragma unroll
  for (int i = 0; i < 4; ++i)
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[i], c, 0, 0, 0);
  return c;
}

// c[0 .. 3] += parts of the sum of four products
__device__ __forceinline__ void products(const f32x4 (&a)[4], const f32x4* b,
                                         f32x4 (&c)[4]) {
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
      c[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j][i], b[j][i], c[j], 0,
                                                  0, 0);
}

template <int BYTES, typename To>
__device__ __forceinline__ void load_bytes(const void* from, To& to) {
  static_assert(sizeof(To) == BYTES);
  if constexpr (BYTES == 8) {
    *reinterpret_cast<uint2*>(to) = *static_cast<const uint2*>(from);
  } else {
#pragma unroll
    for (int i = 0; i < BYTES / 16; ++i)
      reinterpret_cast<u32x4*>(to)[i] = static_cast<const u32x4*>(from)[i];
  }
}

struct ChunkScan {
  float* o;      // [n_tok][H][V]
  float* state;  // [slots][H][V][D]
  // elements from one token to the next: of in, of g, of beta
  const void* in;  // q, k and v of a token
  const float *g, *beta;
  int ld, ld_g, q_off, k_off, v_off;
  const int *e_start, *e_len, *e_pos, *e_row;
  int G, H, D, V;  // G groups of heads share q and k
  float scale;     // of the output
};

// T: bf16 (gated linear attention) or float (delta rule)
// CH: channels of a lane that prepares
template <typename T, int DB, int CH>
struct Chunks {
  static constexpr bool DELTA = sizeof(T) == 4;
  static constexpr int ROW = 4 * DB, PART = CHUNK * ROW;
  // waves that prepare, that make Q, K and the inverse; chunks from the
  // first of these to the state
  static constexpr int PREPARE = DB / (4 * CH), SOLVE = DELTA ? 3 : 1;
  static constexpr int LAG = DELTA ? 3 : 2;
  // for the waves with the state, of LAG + 1 chunks: q F(-1, t), k F(s, 15)
  // transposed, k F(-1, t)
  static constexpr int QT = 0, KH = PART, KT = 2 * PART;
  static constexpr int OWN = DELTA ? 3 * PART : 2 * PART;
  // and of two chunks the factors of B = 8 and 4, 8 rows each: q of tokens
  // that ask, k of those asked, k of those that ask
  static constexpr int LQ = 0, RK = PART, LK = 2 * PART;
  static constexpr int PAIR = DELTA ? 3 * PART : 2 * PART;
  static constexpr int PAIRS = (LAG + 1) * OWN;          // [2][PAIR]
  static constexpr int Q = PAIRS + 2 * PAIR;             // [LAG][1024]
  static constexpr int INV = Q + LAG * 1024;             // [2][1024]
  static constexpr int SUB = INV + (DELTA ? 2048 : 0);   // [2][16][16] floats
  static constexpr int END = SUB + (DELTA ? 2048 : 0);   // [LAG + 1][DB]
  static constexpr int SUMS = END + (LAG + 1) * DB * 4;  // [2][PREPARE][64]
  static constexpr int BETA = SUMS + 2 * PREPARE * 256;  // [4][16]
  static constexpr int LDS = BETA + 256;
  static_assert(LDS <= 160 * 1024, "LDS of a compute unit");

  // 16-byte piece p of row r lies at p ^ r: lanes reading one piece of 16
  // rows meet every bank once
  static __device__ __forceinline__ f32x4 piece(const char* a, int r, int p) {
    return *reinterpret_cast<const f32x4*>(a + r * ROW + (p ^ r) * 16);
  }
  // where channel ch of the transposed rows is, a row of 16 tokens, and
  // tokens 4 p .. 4 p + 3 in it: writing lanes differ in ch / 4, reading
  // ones in ch
  static __device__ __forceinline__ int column(int ch, int p) {
    return ((ch & ~15) + (ch & 3) * 4 + (ch >> 2 & 3)) * 64 +
           (p ^ (ch & 3)) * 16;
  }
  // element (t, s) of a 16 x 16 matrix in bytes
  static __device__ __forceinline__ int element(int t, int s) {
    return t * 64 + ((s >> 2) ^ (t >> 2)) * 16 + (s & 3) * 4;
  }

  // Where token t's sum g is among a wave's 64 (which: 0 Q, 1 K): with
  // itself (Q), with the token before it (t odd), with the first two of its
  // four (t % 4 = 2 or 3); and whether there is one.
  static __device__ __forceinline__ int sum_at(int which, int g, int t) {
    const int j = g == 1 ? t >> 1 : (t >> 2) * 2 + (t & 1);
    return g == 0 ? t : which * 24 + 8 + g * 8 + j;
  }
  static __device__ __forceinline__ bool sum_is(int which, int g, int t) {
    return g == 0 ? which == 0 : g == 1 ? t & 1 : t & 2;
  }

  // -- waves that prepare: lane t = lane % 16 is a token, with CH of the
  // wave's 4 CH channels
  struct Loads {
    float g[CH], beta;
    typename std::conditional<DELTA, float[CH], unsigned[CH / 2]>::type q, k;
  };
  // Products of decays, by token: since the first of its B tokens, and
  // after it to the last of them.
  struct Decays {
    f32x4 pre, suf;
    // B is doubled
    __device__ __forceinline__ void pairs(bool second) {
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const float next = quad_lanes<1, 1, 3, 3>(pre[x]);
        const float both = pre[x] * quad_lanes<0, 0, 2, 2>(pre[x]);
        suf[x] = second ? 1.f : next;
        pre[x] = second ? both : pre[x];
      }
    }
    __device__ __forceinline__ void fours(bool second) {
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const float behind = suf[x] * quad_lanes<3, 3, 3, 3>(pre[x]);
        const float both = pre[x] * quad_lanes<1, 1, 1, 1>(pre[x]);
        suf[x] = second ? suf[x] : behind;
        pre[x] = second ? both : pre[x];
      }
    }
    __device__ __forceinline__ void eights() {
      times_lane<7, 1>(suf, pre);
      times_lane<15, 4>(suf, pre);
      times_lane<3, 2>(pre, pre);
      times_lane<11, 8>(pre, pre);
    }
    __device__ __forceinline__ void sixteen() {
      times_lane<15, 3>(suf, pre);
      times_lane<7, 12>(pre, pre);
    }
  };

  // factors of channels c .. c + 3 for the matrix cores
  template <int B>
  static __device__ __forceinline__ void factors(char* pair, int c, int t,
                                                 f32x4 q, f32x4 k,
                                                 const Decays& f) {
    const bool asks = t & B;
    // of B = 8 the rows are 0 to 7 where tokens ask and 8 to 15 where they
    // are asked, of 4 the other way round: a write's lanes meet every bank
    // once
    const int row = t / (2 * B) * B + t % B + (asks == (B == 8) ? 0 : 8);
    char* to = pair + row * ROW + ((c >> 2) ^ row) * 16;
    const f32x4 by = asks ? f.pre : f.suf;
    *reinterpret_cast<f32x4*>(to + (asks ? LQ : RK)) = (asks ? q : k) * by;
    if (DELTA && asks) *reinterpret_cast<f32x4*>(to + LK) = k * by;
  }

  // chunk i, channels c .. of token t = lane % 16; real: whether there are
  // such
  static __device__ __forceinline__ void prepare(char* lds, int i, int c,
                                                 int t, const Loads& in,
                                                 bool real, bool all_real) {
    char* own = lds + (LAG == 3 ? i & 3 : i % 3) * OWN;
    char* pair = lds + PAIRS + (i & 1) * PAIR;
    float sum[2][4] = {};
#pragma unroll
    for (int h = 0; h < CH / 4; ++h) {
      const int ch = c + h * 4;
      f32x4 q, k;
      Decays f;
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const int j = h * 4 + x;
        f.pre[x] = in.g[j];
        if constexpr (DELTA) {
          q[x] = in.q[j];
          k[x] = in.k[j];
        } else {
          const unsigned a = in.q[j / 2], b = in.k[j / 2];
          q[x] = __uint_as_float(j & 1 ? a & 0xffff0000u : a << 16);
          k[x] = __uint_as_float(j & 1 ? b & 0xffff0000u : b << 16);
        }
      }
      if (!all_real && !real) {
        q = k = f32x4{0.f, 0.f, 0.f, 0.f};
        f.pre = f32x4{1.f, 1.f, 1.f, 1.f};
      }
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const float before = quad_lanes<0, 0, 2, 2>(k[x]);
        sum[0][0] += q[x] * k[x];
        sum[0][1] += q[x] * f.pre[x] * before;
        if (DELTA) sum[1][1] += k[x] * f.pre[x] * before;
      }
      f.pairs(t & 1);
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const float asked = k[x] * f.suf[x];
        const float s0 = quad_lanes<0, 0, 0, 0>(asked);
        const float s1 = quad_lanes<1, 1, 1, 1>(asked);
        const float qf = q[x] * f.pre[x], kf = k[x] * f.pre[x];
        sum[0][2] += qf * s0;
        sum[0][3] += qf * s1;
        if (DELTA) {
          sum[1][2] += kf * s0;
          sum[1][3] += kf * s1;
        }
      }
      f.fours(t & 2);
      factors<4>(pair, ch, t, q, k, f);
      f.eights();
      factors<8>(pair, ch, t, q, k, f);
      f.sixteen();
      const int at = t * ROW + ((ch >> 2) ^ t) * 16;
      *reinterpret_cast<f32x4*>(own + QT + at) = q * f.pre;
      if constexpr (DELTA) *reinterpret_cast<f32x4*>(own + KT + at) = k * f.pre;
      const f32x4 kh = k * f.suf;
#pragma unroll
      for (int x = 0; x < 4; ++x)
        *reinterpret_cast<float*>(own + KH + column(ch + x, t >> 2) +
                                  (t & 3) * 4) = kh[x];
      if (t == 15)
        *reinterpret_cast<f32x4*>(
            lds + END + ((LAG == 3 ? i & 3 : i % 3) * DB + ch) * 4) = f.pre;
    }
    float* sums = reinterpret_cast<float*>(lds + SUMS) +
                  ((i & 1) * PREPARE + c / (4 * CH)) * 64;
    const int g = threadIdx.x >> 4 & 3;
#pragma unroll
    for (int which = 0; which <= DELTA; ++which) {
      const float x = by_rows(sum[which]);
      if (sum_is(which, g, t)) sums[sum_at(which, g, t)] = x;
    }
    if (DELTA && c == 0)
      reinterpret_cast<float*>(lds + BETA)[(i & 3) * 16 + t] =
          real ? in.beta : 0.f;
  }

  // put(t, s, x) with the products of tokens t and s: those of B = 8 and 4
  // of the factors at ``left`` with those asked, and of the sums made above
  // (which: 0 Q, 1 K)
  template <class F>
  static __device__ __forceinline__ void products(const char* lds, int buf,
                                                  int left, int which,
                                                  int lane, F put) {
    const int n = lane & 15, g = lane >> 4;
    const char* pair = lds + PAIRS + buf * PAIR;
    f32x4 a = {0.f, 0.f, 0.f, 0.f}, b = a;
#pragma unroll
    for (int j = 0; j < DB / 16; j += 2) {
      a = mfma4(piece(pair + left, n, 4 * j + g),
                piece(pair + RK, n, 4 * j + g), a);
      b = mfma4(piece(pair + left, n, 4 * j + 4 + g),
                piece(pair + RK, n, 4 * j + 4 + g), b);
    }
    a += b;
    const float* sums = reinterpret_cast<const float*>(lds + SUMS) +
                        buf * PREPARE * 64 + sum_at(which, g, n);
    float x = sums[0];
#pragma unroll
    for (int p = 1; p < PREPARE; ++p) x += sums[p * 64];
    // rows 0 to 7 of a with columns 8 to 15 are of B = 8, rows 8 to 15 with
    // columns 0 to 7 of B = 4, where both are of the same eight tokens
    if ((g < 2) == (n >= 8)) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int t = (4 * g + i) & 7, s = n & 7;
        if (g < 2)
          put(8 + t, s, a[i]);
        else if (t >> 2 == s >> 2)
          put(8 * (t >> 2) + 4 + (t & 3), 8 * (s >> 2) + (s & 3), a[i]);
      }
    }
    if (sum_is(which, g, n))
      put(n, g == 0 ? n : g == 1 ? n - 1 : (n & ~3) + g - 2, x);
  }

  // (I + L)^-1 beta by substitution, four rows at a time: of these lane g
  // makes row g of column n as far as the rows before go, then every lane
  // has all four
  static __device__ __forceinline__ void inverse(const float* L,
                                                 const float* beta, char* m,
                                                 int lane) {
    const int n = lane & 15, g = lane >> 4;
    float x[16];
#pragma unroll
    for (int r = 0; r < 16; r += 4) {
      float y = n == r + g ? 1.f : 0.f;
#pragma unroll
      for (int s = 0; s < r; s += 4) {
        const float4 a =
            *reinterpret_cast<const float4*>(L + (r + g) * 16 + s);
        y -= a.x * x[s] + a.y * x[s + 1] + (a.z * x[s + 2] + a.w * x[s + 3]);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        x[r + i] = __shfl(y, n + 16 * i, WAVE);
#pragma unroll
        for (int s = 0; s < i; ++s)
          x[r + i] -= L[(r + i) * 16 + r + s] * x[r + s];
      }
    }
    const float bn = beta[n];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float y =
          g < 2 ? (g == 0 ? x[i] : x[4 + i]) : (g == 2 ? x[8 + i] : x[12 + i]);
      *reinterpret_cast<float*>(m + element(4 * g + i, n)) = y * bn;
    }
  }
};

// One workgroup: 16 NC value columns of one head of one entry.  In step i
// waves prepare chunk i, make Q and K of chunk i - 1, the inverse of chunk
// i - 2, and those with the state are at chunk i - LAG.
template <typename T, int DB, int CH, int NC>
__global__ __launch_bounds__(64 * (NC + Chunks<T, DB, CH>::PREPARE +
                                   Chunks<T, DB, CH>::SOLVE))
void chunk_scan_kernel(ChunkScan p) {
  using C = Chunks<T, DB, CH>;
  constexpr bool DELTA = C::DELTA;
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  // long portions come last in a batch and take longest: they go first
  const int e = gridDim.y - 1 - blockIdx.y, len = p.e_len[e];
  if (len <= 0) return;
  const int head = blockIdx.x % p.H, D = p.D;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
  const size_t first = (size_t)p.e_start[e];
  const T* in = static_cast<const T*>(p.in) + first * p.ld;
  const int chunks = (len + CHUNK - 1) / CHUNK;

  if (wave >= NC + C::PREPARE) {
    const int part = wave - NC - C::PREPARE;
    if (part == 0)  // what Q has above its diagonal stays zero
      for (int i = lane; i < C::LAG * 64; i += 64)
        *reinterpret_cast<uint4*>(lds + C::Q + i * 16) =
            make_uint4(0, 0, 0, 0);
    float* const beta = reinterpret_cast<float*>(lds + C::BETA);
    float* const sub = reinterpret_cast<float*>(lds + C::SUB);
    __syncthreads();
    for (int i = 0; i < chunks + C::LAG - 2; ++i) {
      if (part == 0) {
        char* m = lds + C::Q + i % C::LAG * 1024;
        if (i < chunks)
          C::products(lds, i & 1, C::LQ, 0, lane,
                      [&](int t, int s, float x) {
                        *reinterpret_cast<float*>(m + C::element(t, s)) = x;
                      });
      } else if (DELTA && part == 1) {
        float* L = sub + (i & 1) * 256;
        const float* b = beta + (i & 3) * 16;
        if (i < chunks)
          C::products(lds, i & 1, C::LK, 1, lane, [&](int t, int s, float x) {
            L[t * 16 + s] = x * b[t];
          });
      } else if (DELTA && i > 0 && i <= chunks) {
        C::inverse(sub + (~i & 1) * 256, beta + ((i - 1) & 3) * 16,
                   lds + C::INV + (~i & 1) * 1024, lane);
      }
      __syncthreads();
    }
    return;
  }
  if (wave >= NC) {
    const int c = ((wave - NC) * 4 + g) * CH;
    const bool real = c < D;
    const int ch = real ? c : 0;
    const int kv = head / (p.H / p.G) * D + ch;
    typename C::Loads x;
    auto fetch = [&](int t) {
      t = t < len ? t : len - 1;
      const T* row = in + (size_t)t * p.ld + kv;
      const float* gr = p.g + (first + t) * p.ld_g + (size_t)head * D + ch;
      constexpr int B = CH * sizeof(T);
      load_bytes<B>(row + p.q_off, x.q);
      load_bytes<B>(row + p.k_off, x.k);
      load_bytes<CH * 4>(gr, x.g);
      if (DELTA) x.beta = p.beta[(first + t) * p.ld + head];
    };
    fetch(n);
    for (int i = 0; i < chunks + C::LAG - 1; ++i) {
      if (i < chunks) {
        C::prepare(lds, i, c, n, x, real && i * CHUNK + n < len,
                   D == DB && (i + 1) * CHUNK <= len);
        fetch((i + 1) * CHUNK + n);
      }
      __syncthreads();
    }
    return;
  }

  // S[a] holds key channels 16 a + 4 g .. + 3 of the lane's column
  const int col = blockIdx.x / p.H * (16 * NC) + wave * 16 + n;
  const bool real = col < p.V;
  const int cv = real ? col : p.V - 1;
  f32x4 S[DB / 16];
  float* sp =
      p.state + (((size_t)p.e_row[e] * p.H + head) * p.V + cv) * (size_t)D;
  const bool resume = p.e_pos[e] > 0;
#pragma unroll
  for (int a = 0; a < DB / 16; ++a) {
    const int d = a * 16 + g * 4;
    S[a] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (resume && d < D) S[a] = *reinterpret_cast<const f32x4*>(sp + d);
  }
  T vn[4];
  auto fetch = [&](int t0) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int t = t0 + 4 * g + i;
      vn[i] = in[(size_t)(t < len ? t : len - 1) * p.ld + p.v_off +
                 (size_t)head * p.V + cv];
    }
  };
  fetch(0);
  float* out = p.o + (first * p.H + head) * p.V + cv;
  const size_t step = (size_t)p.H * p.V;
#pragma unroll
  for (int i = 0; i < C::LAG; ++i) __syncthreads();
  for (int i = 0; i < chunks; ++i) {
    const int place = C::LAG == 3 ? i & 3 : i % 3;
    const char* own = lds + place * C::OWN;
    const char* q = lds + C::Q + i % C::LAG * 1024 + C::element(n, 4 * g);
    f32x4 u;  // of tokens 4 g .. + 3
#pragma unroll
    for (int x = 0; x < 4; ++x) u[x] = to_f(vn[x]);
    fetch((i + 1) * CHUNK);

    // Sums in four parts, so that no product waits for the one before;
    // operands of four products at a time, as more of them do not fit the
    // registers (and what is spilled waits for all loads on their way).
    constexpr int N = DB / 16;
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    f32x4 x[4], o[4];
    auto with_state = [&](const char* rows) {
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] = zero;
#pragma unroll
      for (int a = 0; a < N; a += 4) {
#pragma unroll
        for (int j = 0; j < 4; ++j) x[j] = C::piece(rows, n, 4 * (a + j) + g);
        products(x, S + a, o);
      }
    };
    if constexpr (DELTA) {
      with_state(own + C::KT);
      u = mfma4(*reinterpret_cast<const f32x4*>(
                    lds + C::INV + (i & 1) * 1024 + C::element(n, 4 * g)),
                u - ((o[0] + o[1]) + (o[2] + o[3])), zero);
    }
    with_state(own + C::QT);
    const f32x4 m = *reinterpret_cast<const f32x4*>(q);
    const float* end =
        reinterpret_cast<const float*>(lds + C::END) + place * DB;
#pragma unroll
    for (int r = 0; r < 4; ++r)
      o[r] = __builtin_amdgcn_mfma_f32_16x16x4f32(m[r], u[r], o[r], 0, 0, 0);
#pragma unroll
    for (int a = 0; a < N; a += 4) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        x[j] = *reinterpret_cast<const f32x4*>(
            own + C::KH + C::column(16 * (a + j) + n, g));
        S[a + j] *=
            *reinterpret_cast<const f32x4*>(end + (a + j) * 16 + g * 4);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          S[a + j] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[j][r], u[r],
                                                          S[a + j], 0, 0, 0);
    }
    const f32x4 sum = (o[0] + o[1]) + (o[2] + o[3]);
    // Lanes without a column of their own repeat the last one and store the
    // same.  Only the last chunk asks which tokens there are: what may or
    // may not be stored would be waited for with the next chunk's values.
    if (i + 1 < chunks) {
#pragma unroll
      for (int x = 0; x < 4; ++x)
        out[(i * CHUNK + 4 * g + x) * step] = sum[x] * p.scale;
      __syncthreads();
      continue;
    }
#pragma unroll
    for (int x = 0; x < 4; ++x)
      if (i * CHUNK + 4 * g + x < len)
        out[(i * CHUNK + 4 * g + x) * step] = sum[x] * p.scale;
  }
  if (!real) return;
#pragma unroll
  for (int a = 0; a < DB / 16; ++a) {
    const int d = a * 16 + g * 4;
    if (d < D) *reinterpret_cast<f32x4*>(sp + d) = S[a];
  }
}

// dtype 0: in bf16 (gated linear attention, G = H), 1: in float (delta rule,
// beta [n_tok][ld]); g: the decays
extern "C" int hy_chunk_scan(void* o, void* state, const void* in, int ld,
                             int q_off, int k_off, int v_off, const void* g,
                             int ld_g, const void* beta, const void* e_start,
                             const void* e_len, const void* e_pos,
                             const void* e_row, int n_entries, int G, int H,
                             int D, int V, float scale, int dtype,
                             void* stream) {
  const int each = dtype == 0 ? 8 : 4;  // numbers of 16 bytes
  if (G <= 0 || H <= 0 || H % G || D <= 0 || D % 8 || D > 128 || V <= 0 ||
      V > 4096 || ld % each || q_off % each || k_off % each || ld_g % 4 ||
      n_entries > 65535 || (dtype != 0 && dtype != 1) ||
      (dtype == 1 && !beta) || ((uintptr_t)in | (uintptr_t)g) % 16)
    return -2;
  if (n_entries <= 0) return 0;
  const ChunkScan p{(float*)o, (float*)state, in, (const float*)g,
                    (const float*)beta, ld, ld_g, q_off, k_off, v_off,
                    (const int*)e_start, (const int*)e_len,
                    (const int*)e_pos, (const int*)e_row, G, H, D, V, scale};
#define GO(T, DB, CH, NC)                                                   \
  do {                                                                      \
    using C = Chunks<T, DB, CH>;                                            \
    constexpr int lds = C::LDS, waves = NC + C::PREPARE + C::SOLVE;         \
    static const hipError_t ready = hipFuncSetAttribute(                    \
        reinterpret_cast<const void*>(chunk_scan_kernel<T, DB, CH, NC>),    \
        hipFuncAttributeMaxDynamicSharedMemorySize, lds);                   \
    if (ready != hipSuccess) return -3;                                     \
    const dim3 grid(H * ((V + 16 * NC - 1) / (16 * NC)), n_entries);        \
    hipLaunchKernelGGL((chunk_scan_kernel<T, DB, CH, NC>), grid,            \
                       dim3(64 * waves), lds, (hipStream_t)stream, p);      \
  } while (0)
#define PICK(T, DB)            \
  do {                         \
    if (wide) GO(T, DB, 8, 8); \
    else GO(T, DB, 4, 4);      \
  } while (0)
  // what is prepared serves 128 columns where that still fills the chip
  const bool wide =
      V > 64 && (long long)n_entries * H * ((V + 127) / 128) >= 256;
  if (dtype == 0 && D <= 64) PICK(bf16_t, 64);
  else if (dtype == 0) PICK(bf16_t, 128);
  else if (D <= 64) PICK(float, 64);
  else PICK(float, 128);
#undef PICK
#undef GO
  HY_CHECK();
  return 0;
}
