// The two halves of a parallel layer of windowed attention and routed experts
// side by side, for single tokens: neither half needs the other's results, and
// each is bound by reading memory once, with empty compute units at its ends.
//  * window_up_kernel  attention (window_decode.h) beside the experts' first
//                      product (few_experts.h)
//  * down_out_kernel   their second product beside the output projection
//                      (row_tile.h)
// What takes longer comes first, the other fills the places that it leaves:
// attention of 61 sequences beside products of 16 experts of 4096 x 1280, spread
// evenly among them, made the layer 118.6 us, in front of them 112.7.
//
// us in four launches -> two, from 777 tokens unless noted, 16 experts, 4
// a token:
//   61 tokens  4096 wide, 8 heads of 128, 1280 an expert   121.0 -> 114.8
//   16 tokens  the same                                     86.9 ->  76.7
//   61 tokens  2048 wide, 4 heads of 128, 512 an expert     51.1 ->  43.8
//   128 tokens the same, from 900                           82.8 ->  76.0
//   64 tokens  64 experts, 8 a token                        92.5 ->  83.1
//   64 tokens  1024 wide, 4 heads of 64, 256, from 500      27.5 ->  22.0
//   1 token    the same, 32 experts of 512, from 100        18.5 ->  11.3
// Tiles are those that both can have, so where a half's own kernel has much
// better ones the halves stay apart: see apart_is_faster, and hybrid.few_layer.
// Heads of 33 to 64 and of 97 to 128 (both sides, within their tiles) are those of
// the models that are served; each further pair of sizes is four more kernels.
#include "few_experts.h"
#include "window_decode.h"

template <int DQ, int DV, bool ONCE, int MT>
__global__ __launch_bounds__(256, 2) void window_up_kernel(
    WindowDecode a, FewExperts f, int n_rows, int heads, int attend,
    int up_tiles) {
  extern __shared__ __align__(1024) char lds[];
  __shared__ FewList list;
  static_assert(sizeof(WindowLds<DQ, DV>) <= FEW_LDS<MT>, "one size of LDS");
  int b = blockIdx.x;
  if (b < attend) {
    const int q = b % n_rows, rest = b / n_rows;
    window_decode_block<DQ, DV, ONCE>(
        a, q, rest % heads, rest / heads, attend,
        *reinterpret_cast<WindowLds<DQ, DV>*>(lds));
    return;
  }
  b -= attend;
  few_block<MT>(f, b % up_tiles, b / up_tiles, lds, list);
}

struct FewRows {
  bf16_t* out;       // [N][M]
  const bf16_t* x;   // [N][K]
  const bf16_t* w;   // [M][K]
  int N, M, K;
};
#define OUT_MT 2
template <int NT>
__global__ __launch_bounds__(256, 2) void down_out_kernel(FewRows a,
                                                          FewExperts f,
                                                          int first,
                                                          int down_tiles) {
  using Tile = RowTile<NT, OUT_MT, FEW_KW, NT == 1 ? 3 : 2>;
  static_assert(Tile::LDS <= FEW_LDS<OUT_MT>, "one size of LDS");
  extern __shared__ __align__(1024) char lds[];
  __shared__ FewList list;
  int b = blockIdx.x;
  if (b < first) {
    // row tiles of the same weights on one XCD
    const int row_tiles = (a.N + 16 * NT - 1) / (16 * NT);
    const int m0 = (b / 8 / row_tiles * 8 + b % 8) * 16 * OUT_MT;
    const int r0 = b / 8 % row_tiles * 16 * NT;
    if (m0 >= a.M) return;
    Tile::run(
        lds, a.K, b,
        [&](int r) {
          return a.x + (size_t)(r0 + r < a.N ? r0 + r : a.N - 1) * a.K;
        },
        [&](int r) {
          return a.w + (size_t)(m0 + r < a.M ? m0 + r : a.M - 1) * a.K;
        });
    Tile::each(4 * OUT_MT, [&](int r, int c) {
      if (r0 + r >= a.N || m0 + c >= a.M) return;
      const f32x4 v = Tile::sum(lds, r, c);
      *reinterpret_cast<uint2*>(a.out + (size_t)(r0 + r) * a.M + m0 + c) =
          make_uint2(to_bf16x2(v[0], v[1]), to_bf16x2(v[2], v[3]));
    });
    return;
  }
  b -= first;
  few_block<OUT_MT>(f, b % down_tiles, b / down_tiles, lds, list);
}

// Whether the experts' second product and the output product, N x M and K deep,
// take less in launches of their own.  A tile of 32 x 32 is as many rows of x as
// of W, and by four waves: many tiles of more than 32 rows, which read W again,
// lose to larger ones, the deepest to shares of the depth, and few deep ones
// beside experts that are done long before to 16 x 16 by eight waves.  Both
// launches' time over the one's (experts x their width, outputs, depth, rows):
//   16 x 1280: 4096, 4096 deep 16 rows 1.09, 64 1.01, 96 0.95; 5376 1.11, 1.03,
//       0.93; 8192 1.12, 0.95, 0.86; 6144, 2048 1.08, 1.01, 0.97; 4096 1.08, 0.96,
//       0.92; 64 x 1280: 4096, 5376 1.08, 1.04, 1.01; 8192 1.08, 1.00, 0.98
//   8 x 1536: 8192, 1024 1.05, 1.02, 0.97; 2048 1.04, 1.00, 0.95; 4096 1.05, 0.89
//   16 x 512: 2048, 4096 1.27, 1.18, 1.15; 5376 1.21, 1.09, 1.10; 8192 1.11, 0.99
//   16 x 256: 1024, 2048 1.32, 1.17, 1.32; 4096 1.08, 0.92; 64 x 256: 1.43, 1.24
static bool apart_is_faster(int N, int M, int K, int E, int F) {
  if (K > 3ll * M && (long long)E * F < 3ll * K) return true;
  if (N <= 32) return false;
  const long long tiles = (M + 31ll) / 32 * ((N + 31) / 32);
  return K >= 8192 || tiles >= 768 || tiles * K > 1400000;
}

extern "C" {

int hy_expert_few_tile(int E, int N, int K, int n_pairs);

// 1: done; 0: sizes that take the separate kernels; < 0: an error
int hy_window_up(void* out, int ld_out, void* acc, void* ml, const void* proj,
                 int ld, int g_off, const void* cache, const void* pos,
                 const void* row, const void* bt, int max_blocks, int H, int G,
                 int D, int V, int window, int chunk, int n_rows, int parts,
                 void* u, const void* h, const void* w_up, const void* index,
                 int E, int F, int W, int top, void* stream) {
  const WindowDecode a{(bf16_t*)out, ld_out, (float*)acc, (float*)ml,
                       (const bf16_t*)proj, ld, g_off, (const bf16_t*)cache,
                       (const int*)pos, (const int*)row, (const int*)bt,
                       max_blocks, H, G, D, V, Mask{window, chunk != 0},
                       parts};
  const FewExperts f{(bf16_t*)u, (const bf16_t*)h, (const bf16_t*)w_up,
                     (const int*)index, E, F, W, top, 1, n_rows * top};
  if (!window_decode_ok(a) || !few_ok(f)) return -2;
  if (n_rows <= 0) return 1;
  const bool small = D > 32 && D <= 64 && V <= 64;
  if (!small && (D <= 96 || D > 128 || V <= 64 || V > 128)) return 0;
  const int ht = (H / G + 15) / 16;
  const long long attend = (long long)n_rows * G * ht * parts;
  const int few = hy_expert_few_tile(E, F, W, n_rows * top);
#define RUN(DQ, DV, ONCE, MT)                                                \
  do {                                                                       \
    const int tiles = (F + 16 * MT - 1) / (16 * MT);                         \
    const long long total = attend + (long long)tiles * E;                   \
    if (total > 1 << 30) return 0;                                           \
    static const hipError_t sized = hipFuncSetAttribute(                     \
        reinterpret_cast<const void*>(window_up_kernel<DQ, DV, ONCE, MT>),   \
        hipFuncAttributeMaxDynamicSharedMemorySize, FEW_LDS<MT>);            \
    if (sized != hipSuccess) return -1;                                      \
    hipLaunchKernelGGL((window_up_kernel<DQ, DV, ONCE, MT>),                 \
                       dim3((unsigned)total), dim3(256), FEW_LDS<MT>,        \
                       (hipStream_t)stream, a, f, n_rows, G * ht,            \
                       (int)attend, tiles);                                  \
  } while (0)
#define GO(DQ, DV)                                  \
  do {                                              \
    if (ht == 1 && few == 1) RUN(DQ, DV, true, 1);  \
    else if (ht == 1) RUN(DQ, DV, true, 2);         \
    else if (few == 1) RUN(DQ, DV, false, 1);       \
    else RUN(DQ, DV, false, 2);                     \
  } while (0)
  if (small) GO(64, 64);
  else GO(128, 128);
#undef GO
#undef RUN
  HY_CHECK();
  const int rc = window_merge(a, n_rows, (hipStream_t)stream);
  return rc ? rc : 1;
}

// 1: done; 0: sizes that take the separate kernels; < 0: an error
int hy_down_out(void* out, const void* x, const void* w, int N, int M, int K,
                void* z, const void* u, const void* w_down, const void* index,
                int E, int W, int F, int n_pairs, void* stream) {
  const FewRows a{(bf16_t*)out, (const bf16_t*)x, (const bf16_t*)w, N, M, K};
  const FewExperts f{(bf16_t*)z, (const bf16_t*)u, (const bf16_t*)w_down,
                     (const int*)index, E, W, F, 1, 0, n_pairs};
  if (!few_ok(f) || N <= 0 || M <= 0 || K <= 0 || M % 4 || K % 8 ||
      ((uintptr_t)x | (uintptr_t)w) % 16 || (uintptr_t)out % 8)
    return -2;
  if (apart_is_faster(N, M, K, E, F)) return 0;
  const int tiles = (W + 16 * OUT_MT - 1) / (16 * OUT_MT);
  const int m_tiles = (M + 16 * OUT_MT - 1) / (16 * OUT_MT);
#define GO(NT)                                                               \
  do {                                                                       \
    const long long first =                                                  \
        (m_tiles + 7ll) / 8 * 8 * ((N + 16 * NT - 1) / (16 * NT));           \
    const long long total = first + (long long)tiles * E;                    \
    if (total > 1 << 30) return -2;                                          \
    static const hipError_t sized = hipFuncSetAttribute(                     \
        reinterpret_cast<const void*>(down_out_kernel<NT>),                  \
        hipFuncAttributeMaxDynamicSharedMemorySize, FEW_LDS<OUT_MT>);        \
    if (sized != hipSuccess) return -1;                                      \
    hipLaunchKernelGGL(down_out_kernel<NT>, dim3((unsigned)total),           \
                       dim3(256), FEW_LDS<OUT_MT>, (hipStream_t)stream, a,   \
                       f, (int)first, tiles);                                \
  } while (0)
  if (N <= 16) GO(1);
  else GO(2);
#undef GO
  HY_CHECK();
  return 1;
}

}  // extern "C"
