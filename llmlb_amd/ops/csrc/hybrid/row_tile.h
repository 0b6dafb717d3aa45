// One tile of a product of few rows with a weight matrix, out = x W^T:
// 16 NT rows of x against 16 MT rows of W, bf16, summed in float.
//
//  * W and x come by copies to LDS in rows of 128 bytes.  Loading MFMA
//    operands straight into registers asks for 16 bytes of 16 different
//    rows at a time, which the vector memory path serves one lane a cycle:
//    64 rows against 4096 x 14336 took 77 us that way, 36 this way.
//  * The KW waves of a workgroup share the tile and split the DEPTH, in
//    pieces of 64.  Each copies, waits for and multiplies its own pieces, S
//    of them on their way, without a barrier until the sums meet in LDS.
//  * Workgroups start at different depths: rows lie a multiple of 4 KB
//    apart, and in step they would all ask the same memory channel (3% to
//    10%).
#pragma once
#include "lds_copy.h"
#include "mfma.h"

struct Nothing {
  __device__ __forceinline__ void operator()() const {}
};

template <int NT, int MT, int KW, int S>
struct RowTile {
  static constexpr int ROWS = 16 * (NT + MT), C = ROWS / 8;
  static constexpr int STAGE = ROWS * 128;  // one piece of all rows
  static constexpr int RP = 16 * MT + 4;    // row of the sums
  static constexpr int STAGES = KW * S * STAGE, SUMS = KW * 16 * NT * RP * 4;
  static constexpr int LDS = STAGES > SUMS ? STAGES : SUMS;

  // x_row(r), w_row(r): where the tile's row r of x, of W begins; ``step``:
  // any number, workgroups' differ.  The waves' sums are in LDS after it.
  // DOWN: W's depth goes down, w_row(r) is where r's column begins, r a
  // multiple of 8, and its next number lies ld numbers further.  ``last``:
  // called where a wave's last piece has come, to ask for what follows.
  template <bool DOWN = false, class X, class W, class L = Nothing>
  static __device__ __forceinline__ void run(char* lds, int K, int step,
                                             X x_row, W w_row, int ld = 0,
                                             L last = L{}) {
    static_assert(!DOWN || MT % 2 == 0, "pieces that turn in twos");
    const int tid = threadIdx.x, lane = tid & 63;
    const int lo = lane & 15, hi = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    char* const own = lds + wave * (S * STAGE);
    const unsigned own_byte = lds_byte(own);
    // Copy j of a stage fills rows 8 j .. 8 j + 7, 8 lanes a row.  Piece c
    // of 16 bytes of row r lies at c ^ (r / 2 % 8): lanes reading one piece
    // of 16 rows meet every bank once.  DOWN: of W, 2 MT lanes a number of
    // the depth; pieces turn by two, so that two of the four blocks of eight
    // that are read at once meet other banks.
    const bf16_t* src[C];
    int piece[C];
#pragma unroll
    for (int j = 0; j < C; ++j) {
      if (DOWN && j >= 2 * NT) {
        const int at = (j - 2 * NT) * 64 + lane, k = at / (2 * MT);
        piece[j] = k;
        src[j] = w_row((at % (2 * MT) ^ (k >> 2 & 2)) * 8) + (size_t)k * ld;
        continue;
      }
      const int r = 8 * j + lane / 8;
      piece[j] = ((lane & 7) ^ ((r >> 1) & 7)) * 8;
      src[j] = (j < 2 * NT ? x_row(r) : w_row(r - 16 * NT)) + piece[j];
    }
    const int pieces = (K + 63) / 64;
    const int count = pieces > wave ? (pieces - wave + KW - 1) / KW : 0;
    const int turn = count ? step % count : 0;
    auto copy = [&](int i) {
      const int at = i + turn;
      const int k0 = (wave + (at < count ? at : at - count) * KW) * 64;
      const unsigned to = own_byte + i % S * STAGE;
#pragma unroll
      for (int j = 0; j < C; ++j) {
        // past the depth both sides are zero
        const size_t along = DOWN && j >= 2 * NT ? (size_t)k0 * ld : k0;
        const bf16_t* p = k0 + piece[j] < K
                              ? src[j] + along
                              : reinterpret_cast<const bf16_t*>(zero_piece);
        // (several tiles read columns' lines)
        if (j < 2 * NT || DOWN)
          copy_to_lds(p, to + j * 1024);
        else
          stream_to_lds(p, to + j * 1024);
      }
    };

    f32x4 acc[MT][NT];
#pragma unroll
    for (int a = 0; a < MT; ++a)
#pragma unroll
      for (int b = 0; b < NT; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < S; ++i)
      if (i < count) copy(i);
    for (int i = 0; i < count; ++i) {
      const int newer = count - 1 - i;  // pieces, S - 1 of them on the way
      if (newer >= S - 1)
        wait_copies<(S - 1) * C>();
      else if (S > 2 && newer == 1)
        wait_copies<(S > 2 ? C : 0)>();
      else
        wait_copies<0>();
      if (newer == 0) last();
      const char* st = own + i % S * STAGE;
      u32x4 wf[2][MT], xf[2][NT];
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const int at = lo * 128 + ((s * 4 + hi) ^ (lo >> 1)) * 16;
#pragma unroll
        for (int b = 0; b < NT; ++b)
          xf[s][b] = *reinterpret_cast<const u32x4*>(st + b * 2048 + at);
        const char* const down = st + NT * 2048 +
                                 (s * 32 + hi * 8 + lo / 4) * (32 * MT) +
                                 (lo & 1) * 8;
#pragma unroll
        for (int a = 0; a < MT; ++a)
          wf[s][a] =
              DOWN ? load_columns(
                         reinterpret_cast<const unsigned short*>(
                             down + ((2 * a + (lo >> 1 & 1)) ^ (hi & 1) * 2) *
                                        16),
                         4 * 16 * MT)
                   : *reinterpret_cast<const u32x4*>(st + (NT + a) * 2048 + at);
      }
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int b = 0; b < NT; ++b)
#pragma unroll
          for (int a = 0; a < MT; ++a)
            acc[a][b] = mfma(wf[s][a], xf[s][b], acc[a][b]);
      // the stage has been read before its next copy starts
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      if (i + S < count) copy(i + S);
    }

    if (count == 0) last();
    __syncthreads();  // the sums lie where the stages were
    float* const sums = reinterpret_cast<float*>(lds);
#pragma unroll
    for (int b = 0; b < NT; ++b)
#pragma unroll
      for (int a = 0; a < MT; ++a)
        *reinterpret_cast<f32x4*>(
            &sums[(wave * 16 * NT + b * 16 + lo) * RP + a * 16 + hi * 4]) =
            acc[a][b];
    __syncthreads();
  }

  // outputs c .. c + 3 of the tile's row r of x
  static __device__ __forceinline__ f32x4 sum(const char* lds, int r, int c) {
    const float* const sums = reinterpret_cast<const float*>(lds);
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < KW; ++w)
      v += *reinterpret_cast<const f32x4*>(
          &sums[(w * 16 * NT + r) * RP + c]);
    return v;
  }
  // put(r, c) for every four of the first 4 * quads outputs of all rows
  template <class F>
  static __device__ __forceinline__ void each(int quads, F put) {
    for (int i = threadIdx.x; i < 16 * NT * quads; i += KW * 64)
      put(i / quads, i % quads * 4);
  }
};
