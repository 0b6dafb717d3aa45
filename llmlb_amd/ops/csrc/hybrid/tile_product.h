// Products of many rows with a matrix on the matrix cores, bf16: the tiles of
// tile_gemm.hip (prompts) and of experts_mfma.hip (experts' lists).
#pragma once
#include <type_traits>

#include "lds_copy.h"
#include "row_act.h"

template <int N, int I = 0, class F>
__device__ __forceinline__ void times(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    times<N, I + 1>(static_cast<F&&>(f));
  }
}

// f of the number i, FROM <= i < TO, as a constant
template <int FROM, int TO, class F>
__device__ __forceinline__ void pick(int i, F&& f) {
  if constexpr (TO - FROM == 1) {
    f(std::integral_constant<int, FROM>{});
  } else {
    constexpr int MID = (FROM + TO) / 2;
    if (i < MID) pick<FROM, MID>(i, f);
    else pick<MID, TO>(i, f);
  }
}

constexpr int DEPTH = 64;  // of a step: a row's part is a line of memory

// The tiles of a workgroup, one after the other: BM rows of x against BN rows
// of W, by WM x WN waves.  ``source`` says which: how many tiles there are, and
// of the one ``at(i)`` the rows of x (offsets from x(at)) and W, where
// results go (row(at, r); none: -1) and whether all of it is there.
//
// LDS holds D steps of W's rows and D + 1 of x's.  A step is computed in two
// halves of 32 of its depth; while one is multiplied, the operands of the
// next are read, each into the registers of one that is no longer needed
// (W's, which all of a wave's rows need, have two sets).  The step's only
// barrier stands BP groups of products into its second half: past it every
// wave has read all of the step, whose places the next copies take, and the
// step after is there.  Rows of x are on their way for D - 1/2 steps then,
// those of W for D - 1: small tiles, whose steps are short, need more (48
// tiles of 128 x 128: 0.74 us a step with D = 2, 0.43 with 4).  A tile's first
// steps are fetched while the last of the one before are computed, and its
// results are stored while the next one is.
//
// LDS rows are 8 pieces of 16 bytes; piece c of row r lies at c ^ swizzle(r),
// so that lanes reading one piece of the rows of an operand meet different
// banks.  W's rows enter the matrix cores in an order in which a lane gets 8
// consecutive outputs of each of its rows.
// ROUND: sums are rounded to bf16 before the activation.
// HELD: a tile's results wait in registers, and their stores follow two a step.
// A store counts as done before a copy behind it does, so that a burst of them
// holds the copies up.  It is worth the code in products of experts, whose rows
// lie apart and whose depth is a few steps.
template <int BM, int BN, int WM, int WN, int D, int KIND, bool ROUND,
          bool HELD, class Source>
__device__ __forceinline__ void tile_product(const Source& source,
                                             bf16_t* __restrict__ out,
                                             int ld_out, int M, int K,
                                             RowAct act) {
  constexpr int NW = WM * WN;
  constexpr int TX = BM / WM / 16, TW = BN / WN / 16;  // 16-row tiles a wave
  constexpr int CX = BM / 8 / NW, CW = BN / 8 / NW;    // copies a wave
  constexpr bool GATED = KIND == SWIGLU || KIND == CLAMPED;
  constexpr int OUT = GATED ? BN / 2 : BN;             // outputs a tile
  constexpr int GROUPS = GATED ? TW / 4 : TW / 2;      // of 32 outputs
  constexpr int STORES = GROUPS * TX;
  constexpr int UX = BM * DEPTH, UW = BN * DEPTH;      // a step's rows
  constexpr int BP = TX < 8 ? 1 : 2;
  static_assert(BM % (8 * NW) == 0 && BN % (8 * NW) == 0, "whole copies");
  static_assert(GROUPS >= 1 && D >= 2, "a wave's outputs, steps ahead");
  extern __shared__ __align__(1024) unsigned short tile_lds[];
  unsigned short* const lds = tile_lds;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  // an XCD (every eighth workgroup) has a run of neighbouring tiles
  const int xcd = blockIdx.x & 7, slots = gridDim.x >> 3;
  const long long all = source.tiles();
  const int end = (int)(all * (xcd + 1) / 8);
  int tile = (int)(all * xcd / 8) + (blockIdx.x >> 3);
  if (tile >= end) return;

  auto swizzle_x = [](int r) { return r & 7; };
  auto swizzle_w = [](int r) { return (r & 3) | ((r >> 1) & 4); };

  // -- copies: tile and depth they are at, the lane's offsets in bytes
  unsigned xo[CX], wo[CW];
  const bf16_t *xt, *wt;
  int xk = 0, wk = 0, x_tile = tile, w_tile = tile, to_x = 0, to_w = 0;
  auto aim_x = [&] {
    const auto at = source.at(x_tile);
    xt = source.x(at);
#pragma unroll
    for (int i = 0; i < CX; ++i) {
      const int r = (wave * CX + i) * 8 + (lane >> 3);
      const int c = ((lane & 7) ^ swizzle_x(r)) * 8;
      xo[i] = (source.x_offset(at, r) + c) * 2;
    }
  };
  auto aim_w = [&] {
    const auto at = source.at(w_tile);
    wt = source.w(at);
#pragma unroll
    for (int i = 0; i < CW; ++i) {
      const int r = (wave * CW + i) * 8 + (lane >> 3);
      const int c = ((lane & 7) ^ swizzle_w(r)) * 8;
      // with gate and up, 32 rows of the one and 32 of the other in turn
      const int m = at.m0 + (GATED ? (r >> 6) * 32 + (r & 31) : r);
      const int row =
          (m < M ? m : M - 1) + (GATED && (r & 32) ? act.up : 0);
      wo[i] = ((unsigned)row * (unsigned)K + c) * 2;
    }
  };
  auto next_x = [](int u) { return u == D ? 0 : u + 1; };
  auto next_w = [](int u) { return u == D - 1 ? 0 : u + 1; };
  const unsigned base = lds_byte(lds);
  auto copy_x = [&](int i) {
    copy_to_lds(xt + xk, xo[i], base + to_x * UX * 2 + (wave * CX + i) * 1024);
  };
  auto copy_w = [&](int i) {
    copy_to_lds(wt + wk, wo[i],
                base + ((D + 1) * UX + to_w * UW) * 2 +
                    (wave * CW + i) * 1024);
  };
  // past the last tile its beginning is copied again: every step has as
  // many copies
  auto step_x = [&] {
    to_x = next_x(to_x);
    if ((xk += DEPTH) < K) return;
    xk = 0;
    if (x_tile + slots < end) {
      x_tile += slots;
      if (x_tile + slots < end) source.fetch(x_tile + slots);
      aim_x();
    }
  };
  auto step_w = [&] {
    to_w = next_w(to_w);
    if ((wk += DEPTH) < K) return;
    wk = 0;
    if (w_tile + slots < end) {
      w_tile += slots;
      aim_w();
    }
  };
  source.fetch(tile);
  if (tile + slots < end) source.fetch(tile + slots);
  source.fetched();
  aim_x();
  aim_w();
#pragma unroll
  for (int s = 0; s < D; ++s) {
#pragma unroll
    for (int i = 0; i < CX; ++i) copy_x(i);
    step_x();
#pragma unroll
    for (int i = 0; i < CW; ++i) copy_w(i);
    step_w();
  }

  // -- operands and sums
  const int wm = wave / WN * (BM / WM), wn = wave % WN * (BN / WN);
  const int l = lane & 15, g = lane >> 4;
  const int rx = wm + l, rw = wn + 8 * (l >> 2) + (l & 3);
  const int sx = swizzle_x(rx), sw = swizzle_w(rw);
  u32x4 fx[TX], fw[2][TW];
  f32x4 acc[TX][TW];
  int ux = 0, uw = 0;  // where the step lies
  auto at_x = [&](int half) {
    return lds + ux * UX + rx * DEPTH + ((half * 4 + g) ^ sx) * 8;
  };
  auto at_w = [&](int half) {
    return lds + (D + 1) * UX + uw * UW + rw * DEPTH +
           ((half * 4 + g) ^ sw) * 8;
  };
  auto read_x = [&](const unsigned short* p, int i) {
    fx[i] = *reinterpret_cast<const u32x4*>(p + i * 16 * DEPTH);
  };
  auto read_w = [&](int set, const unsigned short* p, int i) {
    fw[set][i] = *reinterpret_cast<const u32x4*>(
        p + ((i >> 1) * 32 + (i & 1) * 4) * DEPTH);
  };
  // The products of half H of the step; the order alternates, so that one
  // operand stays from each to the next.
  auto half = [&](auto H, auto&& barrier) {
    constexpr int h = H, first = h ? BP : 0;  // where the next reads begin
    constexpr int C = h ? CW : CX, PER = (C + TX - first - 1) / (TX - first);
    const unsigned short *px = at_x(h), *nx, *nw;
    if (!h) nx = at_x(1), nw = at_w(1);
    times<TX>([&](auto IA) {
      constexpr int a = IA;
      if constexpr (h && a == BP) {
        barrier();
        nx = at_x(0), nw = at_w(0);
      }
      times<TW>([&](auto IB) {
        constexpr int i = IB, b = a % 2 ? TW - 1 - i : i;
        // W's reads: every second product, or where groups are few all
        constexpr int LEFT = (TW + TX - first - 1) / (TX - first);
        constexpr int RW = LEFT > TW / 2 ? LEFT : TW / 2;
        constexpr int IS = RW > TW / 2 ? i : (i % 2 ? i / 2 : RW);
        acc[a][b] = mfma(fw[h][b], fx[a], acc[a][b]);
        if constexpr (i == 0 && a == 0) read_x(px, TX - 1);
        if constexpr (i == 0 && a > first) read_x(nx, a - 1);
        if constexpr (h && a == BP && i < BP) read_x(nx, i);
        if constexpr (a >= first && IS < RW && (a - first) * RW + IS < TW)
          read_w(h ^ 1, nw, (a - first) * RW + IS);
        if constexpr (a >= first && i == 2 % TW)
          times<PER>([&](auto IC) {
            constexpr int c = (a - first) * PER + IC;
            if constexpr (c < C) {
              if constexpr (h) copy_w(c);
              else copy_x(c);
            }
          });
        __builtin_amdgcn_sched_barrier(0);
      });
    });
  };
  constexpr std::integral_constant<int, 0> H0{};
  constexpr std::integral_constant<int, 1> H1{};

  // -- results
  constexpr int LATER = 2, SENDS = HELD ? (STORES + LATER - 1) / LATER : 0;
  u32x4 held[HELD ? STORES : 1];
  int sent = SENDS;     // of the last tile's
  bool stored = false;  // its stores are of all lanes
  auto held_at = source.at(tile);
  // group i of the tile's row n of results
  auto store = [&](const auto& at, long long n, int i, int lane_, u32x4 v) {
    const int m = at.m0 + (GATED ? wn / 2 : wn) + i % GROUPS * 32 +
                  (lane_ >> 4) * 8;
    if (n >= 0 && m < M)
      *reinterpret_cast<u32x4*>(out + n * ld_out + m) = v;
  };
  auto send = [&] {
    if constexpr (HELD)
      pick<0, SENDS>(sent++, [&](auto IS) {
        times<LATER>([&](auto IP) {
          constexpr int i = IS * LATER + IP;
          if constexpr (i < STORES) {
            int lane_ = lane;
            // (places of what is held are not to be kept through the steps)
            asm volatile("" : "+v"(lane_));
            store(held_at,
                  source.row(held_at, wm + i / GROUPS * 16 + (lane_ & 15)), i,
                  lane_, held[i]);
          }
        });
      });
  };
  // all but the copies of the steps past the next one, and what has been
  // stored behind the next one's
  constexpr int COPIES = (D - 2) * (CX + CW) + CX;
  auto step = [&](auto&& wait) {
    half(H0, [] {});
    step_x();
    half(H1, [&] {
      wait();
      ux = next_x(ux);
      uw = next_w(uw);
    });
    step_w();
  };

  wait_barrier<(D - 1) * (CX + CW)>();
#pragma unroll
  for (int b = 0; b < TW; ++b) read_w(0, at_w(0), b);
#pragma unroll
  for (int a = 0; a < TX - 1; ++a) read_x(at_x(0), a);
  for (;;) {
#pragma unroll
    for (int a = 0; a < TX; ++a)
#pragma unroll
      for (int b = 0; b < TW; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
    int s = 0;
    if constexpr (HELD) {
      bool last = false;  // the step before has sent LATER
      while (s < K && sent < SENDS) {
        step([&] {
          if (last) wait_barrier<COPIES + LATER>();
          else wait_barrier<COPIES>();
        });
        send();
        last = stored && sent * LATER <= STORES;
        s += DEPTH;
      }
      for (; s < K; s += DEPTH) step([] { wait_barrier<COPIES>(); });
      while (sent < SENDS) send();  // what a shallow product has left
    } else {
      do {
        step([&] {
          if (s < (D - 1) * DEPTH && stored) wait_barrier<COPIES + STORES>();
          else wait_barrier<COPIES>();
        });
      } while ((s += DEPTH) < K);
    }

    const auto at = source.at(tile);
    // edges store less, and the wait is for all of it
    stored = source.whole(at) && at.m0 + OUT <= M;
    held_at = at;
    sent = 0;
    RowAct as = act;
    as.kind = KIND;
    long long n = 0;  // a row's place is looked up once
    times<STORES>([&](auto II) {
      constexpr int I = II, a = I / GROUPS;
      if constexpr (!HELD && I % GROUPS == 0)
        n = source.row(at, wm + a * 16 + (lane & 15));
      constexpr int b = I % GROUPS * (GATED ? 4 : 2);
      unsigned p[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int t = b + i / 2, e = i % 2 * 2;
        float v[2] = {acc[a][t][e], acc[a][t][e + 1]};
        // (plain sums are rounded where they are stored)
        if constexpr (ROUND && KIND != PLAIN) round_bf16x2(v[0], v[1]);
        if constexpr (GATED) {
          float u[2] = {acc[a][t + 2][e], acc[a][t + 2][e + 1]};
          round_bf16x2(u[0], u[1]);
          v[0] = row_gate(as, v[0], u[0]);
          v[1] = row_gate(as, v[1], u[1]);
        } else {
          v[0] = row_act(as, v[0]);
          v[1] = row_act(as, v[1]);
        }
        p[i] = to_bf16x2(v[0], v[1]);
      }
      const u32x4 v{p[0], p[1], p[2], p[3]};
      if constexpr (HELD) held[I] = v;
      else store(at, n, I, lane, v);
    });
    tile += slots;
    if (tile >= end) break;
  }
  while (sent < SENDS) send();
  // no copy is under way when the workgroup's LDS is given back
  wait_barrier<0>();
}
