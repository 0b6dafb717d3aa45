// Prompt portions of the recurrences with a decay per key channel (gated
// linear attention, see linear_scan.hip; gated delta rule, see
// channel_delta.hip) on the matrix cores, 16 tokens at a time.
//
// With F_t the sum of the chunk's log decays up to token t and S the state
// before it, both are
//   o_t = S^T (q_t e^F_t) + sum over s <= t of Q_ts u_s,
//   S  <- e^F_15 S + sum over s of (k_s e^(F_15 - F_s)) u_s^T,
//   Q_ts = sum over channels of q_t k_s e^(F_t - F_s),
// with u = v for gated linear attention, and for the delta rule
//   u = (I + L)^-1 beta (v - S^T (k e^F)),   L_ts = beta_t K_ts (s < t),
// K being Q with k_t for q_t.  The inverse is made by substitution.
//
// Q and K are products of the matrix cores if e^(F_t - F_s) is taken apart:
// within eight tokens as e^(F_t - R) e^(R - F_s), R being F after the first
// four of them, from the second eight to the first as e^(F_t - R) and
// e^(R - F_s), R of the second.  A step's log decay is taken as no less than
// 2^-24, which beside what comes in is what a float keeps, so no factor is
// above 2^96.
//
// Everything enters a product as the sum of two bf16 numbers (relative error
// 2^-17); sums, the state, decays and the substitution are float.
//
// Bound by the chain from chunk to chunk.  Waves carry the state, 16 value
// columns each, and work on one chunk while one or two others make Q and the
// inverse of the next one and the rest the factors of the one after it; they
// meet once a chunk, and a chunk takes about as long as what the waves of
// one SIMD issue for it.  8 x 2048 tokens, heads of 128 x 128, us, token by
// token -> now: delta rule, 16 heads, 1179 -> 340; gated linear attention,
// 32 heads, 1030 -> 395.
#include "common.h"
#include "mfma.h"
#include <type_traits>

#define CHUNK 16

// lane x of every 16 for all of them; the lane n before, or zero
template <int LANE>
__device__ __forceinline__ float row_lane(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(
      0, __float_as_int(x), 0x150 + LANE, 0xf, 0xf, true));
}
template <int N>
__device__ __forceinline__ float row_before(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(
      0, __float_as_int(x), 0x110 + N, 0xf, 0xf, true));
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

// T: bf16 (gated linear attention) or float (delta rule); g: logs of two
// CH: channels of a lane that prepares
template <typename T, int DB, int CH>
struct Chunks {
  static constexpr bool DELTA = sizeof(T) == 4;
  static constexpr int KJ = DB / 32, ROW = 2 * DB, PART = CHUNK * ROW;
  // waves that prepare, and that make Q and the inverse
  static constexpr int PREPARE = DB / (4 * CH), SOLVE = DELTA ? 2 : 1;
  // arrays of hi and lo rows: for the waves with the state, of three chunks
  static constexpr int QT = 0, KH = 2 * PART, KT = 4 * PART;
  static constexpr int OWN = DELTA ? 6 * PART : 4 * PART;
  // and of two chunks left factors, right ones, right ones of the first
  // eight tokens for the second
  static constexpr int LQ = 0, RK = 2 * PART, RB = 4 * PART, LK = 5 * PART;
  static constexpr int PAIR = DELTA ? 7 * PART : 5 * PART;
  static constexpr int PAIRS = 3 * OWN;                  // [2][PAIR]
  static constexpr int MT = PAIRS + 2 * PAIR;            // [2][Q, T][1024]
  static constexpr int END = MT + 4 * 1024;              // [3][DB] floats
  static constexpr int BETA = END + 3 * DB * 4;               // [2][16]
  static constexpr int SUB = BETA + 2 * 64;  // [16][16] floats
  static constexpr int LDS = SUB + (DELTA ? 1024 : 0);

  // 16-byte piece p of row r lies at p ^ turn(r)
  static __device__ __forceinline__ int turn(int r) {
    return DB == 128 ? r & 15 : (r >> 1) & 7;
  }
  static __device__ __forceinline__ u32x4 piece(const char* a, int r, int j,
                                                int g) {
    return *reinterpret_cast<const u32x4*>(
        a + r * ROW + ((j * 4 + g) ^ turn(r)) * 16);
  }
  // sum of the products of hi + lo numbers, but for lo * lo
  static __device__ __forceinline__ f32x4 both(u32x4 ah, u32x4 al, u32x4 bh,
                                               u32x4 bl, f32x4 c) {
    c = mfma(ah, bh, c);
    c = mfma(ah, bl, c);
    return mfma(al, bh, c);
  }

  // -- waves that prepare: lane t = lane % 16 is a token, with CH of the
  // wave's 4 CH channels
  struct Loads {
    float g[CH], beta;
    typename std::conditional<DELTA, float[CH], unsigned[CH / 2]>::type q, k;
  };

  // x e into row t of an array, from channel c on; part: its bytes
  static __device__ __forceinline__ void write(char* a, int c, int t,
                                               const float (&x)[CH],
                                               const float (&e)[CH],
                                               int part = PART) {
    // quads of channels 0 to 3 of every 32 are the first halves of the
    // pieces, 4 to 7 the second: as the state's lanes hold them
#pragma unroll
    for (int h = 0; h < CH; h += 4) {
      uint2 hi, lo;
      split2(x[h] * e[h], x[h + 1] * e[h + 1], hi.x, lo.x);
      split2(x[h + 2] * e[h + 2], x[h + 3] * e[h + 3], hi.y, lo.y);
      const int quad = (c + h) / 4;
      char* to = a + t * ROW +
                 ((quad / 8 * 4 + (quad & 3)) ^ turn(t)) * 16 +
                 (quad >> 2 & 1) * 8;
      *reinterpret_cast<uint2*>(to) = hi;
      *reinterpret_cast<uint2*>(to + part) = lo;
    }
  }

  // chunk i, the j-th of three, channels c .. of token t = lane % 16;
  // real: whether there are such
  static __device__ __forceinline__ void prepare(char* lds, int i, int j,
                                                 int c, int t,
                                                 const Loads& in, bool real,
                                                 bool all_real) {
    float F[CH], q[CH], k[CH], e[CH], first[CH], mid[CH], mid2[CH];
#pragma unroll
    for (int x = 0; x < CH; ++x) {
      const float f = in.g[x];
      F[x] = f < -24.f ? -24.f : f;
      if constexpr (DELTA) {
        q[x] = in.q[x];
        k[x] = in.k[x];
      } else {
        const unsigned a = in.q[x / 2], b = in.k[x / 2];
        q[x] = __uint_as_float(x & 1 ? a & 0xffff0000u : a << 16);
        k[x] = __uint_as_float(x & 1 ? b & 0xffff0000u : b << 16);
      }
    }
    if (!all_real && !real) {
#pragma unroll
      for (int x = 0; x < CH; ++x) F[x] = q[x] = k[x] = 0.f;
    }
    // sums over the tokens, of the second eight without the first
    const bool second = t >= 8;
#pragma unroll
    for (int x = 0; x < CH; ++x) {
      F[x] += row_before<1>(F[x]);
      F[x] += row_before<2>(F[x]);
      F[x] += row_before<4>(F[x]);
      F[x] += row_before<8>(F[x]);
      first[x] = row_lane<7>(F[x]);
      if (second) F[x] -= first[x];
      mid2[x] = row_lane<11>(F[x]);
      mid[x] = second ? mid2[x] : row_lane<3>(F[x]);
    }
    char* own = lds + j * OWN;
    char* pair = lds + PAIRS + (i & 1) * PAIR;
    auto exps = [&](auto&& of) {
#pragma unroll
      for (int x = 0; x < CH; ++x) e[x] = __builtin_amdgcn_exp2f(of(x));
    };
    exps([&](int x) { return F[x] - mid[x]; });
    write(pair + LQ, c, t, q, e);
    if constexpr (DELTA) write(pair + LK, c, t, k, e);
    exps([&](int x) { return mid[x] - F[x]; });
    write(pair + RK, c, t, k, e);
    exps([&](int x) { return first[x] - F[x] + mid2[x]; });
    if (!second) write(pair + RB, c, t, k, e, PART / 2);
    exps([&](int x) {
      const float last = row_lane<15>(F[x]);
      return second ? last - F[x] : first[x] - F[x] + last;
    });
    write(own + KH, c, t, k, e);
    exps([&](int x) { return second ? first[x] + F[x] : F[x]; });
    write(own + QT, c, t, q, e);
    if constexpr (DELTA) write(own + KT, c, t, k, e);
    if (t == 15) {
      float* end = reinterpret_cast<float*>(lds + END) + j * DB + c;
#pragma unroll
      for (int x = 0; x < CH; x += 4)
        *reinterpret_cast<float4*>(end + x) =
            make_float4(e[x], e[x + 1], e[x + 2], e[x + 3]);
    }
    if (DELTA && c == 0)
      reinterpret_cast<float*>(lds + BETA)[(i & 1) * 16 + t] =
          real ? in.beta : 0.f;
  }

  // row t = 4 g + i, column s = n of the left factors' product with the
  // right ones; what is above the diagonal is anything
  static __device__ __forceinline__ f32x4 pairs(const char* pair, int left,
                                                int n, int g) {
    f32x4 a = {0.f, 0.f, 0.f, 0.f}, b = a;
#pragma unroll
    for (int j = 0; j < KJ; ++j) {
      const u32x4 lh = piece(pair + left, n, j, g);
      const u32x4 ll = piece(pair + left + PART, n, j, g);
      a = both(lh, ll, piece(pair + RK, n, j, g),
               piece(pair + RK + PART, n, j, g), a);
      b = both(lh, ll, piece(pair + RB, n & 7, j, g),
               piece(pair + RB + PART / 2, n & 7, j, g), b);
    }
    return g >= 2 && n < 8 ? b : a;
  }

  // a 16 x 16 matrix as the left operand of a product with u: a row's
  // columns 4 g .. + 3, hi and then lo
  static __device__ __forceinline__ void put(char* m, int t, int s, float x) {
    unsigned hi, lo;
    split2(x, 0.f, hi, lo);
    unsigned short* to =
        reinterpret_cast<unsigned short*>(m + t * 64 + (s >> 2) * 16) +
        (s & 3);
    to[0] = hi;
    to[4] = lo;
  }

  static __device__ __forceinline__ void outputs_of_values(char* lds, int buf,
                                                           int lane) {
    const int n = lane & 15, g = lane >> 4;
    const f32x4 m = pairs(lds + PAIRS + buf * PAIR, LQ, n, g);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      put(lds + MT + buf * 2048, 4 * g + i, n, n <= 4 * g + i ? m[i] : 0.f);
  }

  // (I + L)^-1 beta by substitution, four rows at a time: of these lane g
  // makes row g of column n as far as the rows before go, then every lane
  // has all four
  static __device__ __forceinline__ void inverse(char* lds, int buf,
                                                 int lane) {
    const int n = lane & 15, g = lane >> 4;
    const float* beta =
        reinterpret_cast<const float*>(lds + BETA) + buf * 16;
    const float bn = beta[n];
    const float4 bt = *reinterpret_cast<const float4*>(beta + 4 * g);
    const f32x4 m = pairs(lds + PAIRS + buf * PAIR, LK, n, g);
    const f32x4 l = m * f32x4{bt.x, bt.y, bt.z, bt.w};
    float* L = reinterpret_cast<float*>(lds + SUB);
#pragma unroll
    for (int i = 0; i < 4; ++i) L[(4 * g + i) * 16 + n] = l[i];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
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
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float y =
          g < 2 ? (g == 0 ? x[i] : x[4 + i]) : (g == 2 ? x[8 + i] : x[12 + i]);
      put(lds + MT + buf * 2048 + 1024, 4 * g + i, n, y * bn);
    }
  }
};

// One workgroup: 16 NC value columns of one head of one entry.  In step i
// the waves with the state are at chunk i - 2.
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
    __syncthreads();
    for (int i = 0; i < chunks; ++i) {
      if (wave == NC + C::PREPARE)
        C::outputs_of_values(lds, i & 1, lane);
      else if constexpr (DELTA)
        C::inverse(lds, i & 1, lane);
      __syncthreads();
    }
    __syncthreads();
    return;
  }
  if (wave >= NC) {
    const int c = ((wave - NC) * 4 + g) * CH;
    const bool real = c < D;
    const int ch = real ? c : 0;
    const int kv = head / (p.H / p.G) * D + ch;
    typename C::Loads next;
    auto fetch = [&](int t) {
      t = t < len ? t : len - 1;
      const T* row = in + (size_t)t * p.ld + kv;
      const float* gr = p.g + (first + t) * p.ld_g + (size_t)head * D + ch;
      constexpr int B = CH * sizeof(T);
      load_bytes<B>(row + p.q_off, next.q);
      load_bytes<B>(row + p.k_off, next.k);
      load_bytes<CH * 4>(gr, next.g);
      if (DELTA) next.beta = p.beta[(first + t) * p.ld + head];
    };
    fetch(n);
    for (int i = 0, j = 0; i < chunks; ++i, j = j == 2 ? 0 : j + 1) {
      const typename C::Loads now = next;
      if (i + 1 < chunks) fetch((i + 1) * CHUNK + n);
      C::prepare(lds, i, j, c, n, now, real && i * CHUNK + n < len,
                 D == DB && (i + 1) * CHUNK <= len);
      __syncthreads();
    }
    __syncthreads();
    __syncthreads();
    return;
  }

  // S[tile] holds key channels 16 tile + 4 g .. + 3 of the lane's column
  const int col = blockIdx.x / p.H * (16 * NC) + wave * 16 + n;
  const bool real = col < p.V;
  const int cv = real ? col : p.V - 1;
  f32x4 S[2 * C::KJ];
  float* sp =
      p.state + (((size_t)p.e_row[e] * p.H + head) * p.V + cv) * (size_t)D;
  const bool resume = p.e_pos[e] > 0;
#pragma unroll
  for (int a = 0; a < 2 * C::KJ; ++a) {
    const int d = a * 16 + g * 4;
    S[a] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (resume && d < D) {
      const float4 x = *reinterpret_cast<const float4*>(sp + d);
      S[a] = f32x4{x.x, x.y, x.z, x.w};
    }
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
  __syncthreads();
  __syncthreads();
  for (int i = 0, third = 0; i < chunks;
       ++i, third = third == 2 ? 0 : third + 1) {
    const char* own = lds + third * C::OWN;
    const char* mats = lds + C::MT + (i & 1) * 2048 + n * 64 + g * 16;
    T v[4];
#pragma unroll
    for (int x = 0; x < 4; ++x) v[x] = vn[x];
    if (i + 1 < chunks) fetch((i + 1) * CHUNK);

    f32x4 w = {0.f, 0.f, 0.f, 0.f}, o = w;
#pragma unroll
    for (int j = 0; j < C::KJ; ++j) {
      u32x4 sh, sl;
#pragma unroll
      for (int h = 0; h < 4; ++h) {
        unsigned a, b;
        split2(S[2 * j + h / 2][h % 2 * 2], S[2 * j + h / 2][h % 2 * 2 + 1],
               a, b);
        sh[h] = a;
        sl[h] = b;
      }
      if constexpr (DELTA)
        w = C::both(C::piece(own + C::KT, n, j, g),
                    C::piece(own + C::KT + C::PART, n, j, g), sh, sl, w);
      o = C::both(C::piece(own + C::QT, n, j, g),
                  C::piece(own + C::QT + C::PART, n, j, g), sh, sl, o);
    }
    // hi and lo of u, tokens 4 g .. + 3 twice
    u32x4 uh, ul;
    auto parts = [&](f32x4 x) {
      unsigned h0, h1, l0, l1;
      split2(x[0], x[1], h0, l0);
      split2(x[2], x[3], h1, l1);
      uh = u32x4{h0, h1, h0, h1};
      ul = u32x4{l0, l1, l0, l1};
    };
    if constexpr (DELTA) {
      parts(f32x4{v[0] - w[0], v[1] - w[1], v[2] - w[2], v[3] - w[3]});
      const u32x4 m = *reinterpret_cast<const u32x4*>(mats + 1024);
      f32x4 u = {0.f, 0.f, 0.f, 0.f};
      u = mfma(m, uh, u);
      parts(mfma(m, ul, u));
    } else {
      parts(f32x4{to_f(v[0]), to_f(v[1]), to_f(v[2]), to_f(v[3])});
    }
    const u32x4 m = *reinterpret_cast<const u32x4*>(mats);
    o = mfma(m, uh, o);
    if constexpr (DELTA) o = mfma(m, ul, o);
    const float* end =
        reinterpret_cast<const float*>(lds + C::END) + third * DB;
    const int r = 4 * g + (n >> 2);
#pragma unroll
    for (int a = 0; a < 2 * C::KJ; ++a) {
      const float4 f = *reinterpret_cast<const float4*>(end + a * 16 + g * 4);
      const char* at = own + C::KH + r * C::ROW +
                       ((a / 2 * 4 + (n & 3)) ^ C::turn(r)) * 16 + a % 2 * 8;
      const u32x4 k = load_columns(
          reinterpret_cast<const unsigned short*>(at), C::PART / 2);
      S[a] *= f32x4{f.x, f.y, f.z, f.w};
      S[a] = mfma(k, uh, S[a]);
      if constexpr (DELTA) S[a] = mfma(k, ul, S[a]);
    }
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const int t = i * CHUNK + 4 * g + x;
      if (real && t < len) out[t * step] = o[x] * p.scale;
    }
    __syncthreads();
  }
  if (!real) return;
#pragma unroll
  for (int a = 0; a < 2 * C::KJ; ++a) {
    const int d = a * 16 + g * 4;
    if (d < D)
      *reinterpret_cast<float4*>(sp + d) =
          make_float4(S[a][0], S[a][1], S[a][2], S[a][3]);
  }
}

// dtype 0: in bf16 (gated linear attention, G = H), 1: in float (delta rule,
// beta [n_tok][ld]); g: logarithms (of two) of the decays
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
