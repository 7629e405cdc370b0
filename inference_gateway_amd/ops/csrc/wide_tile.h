// y = x W^T for hundreds to thousands of rows of x, gfx950, bf16, products and
// sums in fp32 (16x16x32 matrix instructions); with a GATE W = [gate; up] and the
// result is act(gate) * up of the fp32 sums.
//
// Bound by the matrix cores and, with them, by the card's power: the busier they
// are the lower the clock (1.8 GHz at 74 % busy, 1.5 at 86).  So what counts is
// that nothing else takes energy or makes them wait:
//
//   * tiles of 256 x 256, one workgroup of four waves a compute unit, each with
//     128 x 128 of the tile in its accumulators: 32 LDS reads of a wave for 128
//     matrix instructions (eight waves of 128 x 64 read half as much again and
//     were 6 % slower; 32 x 32 x 16 instructions 6 %);
//   * K in steps of 64, whole 128-byte lines: by DMA to LDS, two steps of x and
//     three of W (all of the 160 KB).  Steps of 32 have longer to arrive and
//     were 9 % slower for their half lines, two buffers of W 6 %;
//   * the fragments of half a step are read between the products of the half
//     before, so a step has one barrier and no wait of its own;
//   * a workgroup walks the tiles of all rounds, and the next tile's first steps
//     are under way while the results are stored;
//   * tiles of fewer rows or columns where they fill the rounds better.
//
// Measured alone, library with silu_mul and here (us): 1024 x 28672 x 4096 217 and
// 176, 8192 rows 1524 and 1384 (1.39 PFLOP/s), 16000 rows 2869 and 2649; between the
// other kernels of a step 193, 1443 and 2710.  On a cooler card 197 and 170, 1377 and
// 1319 (1.46 PFLOP/s), 2804 and 2590; there, with no stores 1242, with every step
// from the caches 1256 at 8192 rows.  With GELU, 5790 rows of 28672 x 4096 in a step
// 1154 (library and gated_act) and 1048.
#pragma once

#include <type_traits>

#include "common.h"

namespace igw {

typedef __attribute__((ext_vector_type(8))) __bf16 wg_bf16x8;
typedef __attribute__((ext_vector_type(4))) float wg_f32x4;
typedef __attribute__((ext_vector_type(4))) uint32_t wg_u32x4;
typedef __attribute__((ext_vector_type(2))) uint32_t wg_u32x2;

constexpr int WG_BK = 64;        // entries of a K step
constexpr int WG_BLOCKS = 256;   // one workgroup per compute unit, 32 per XCD

struct WideArgs {
  uint16_t* out;         // [M, N]
  const uint16_t* x;
  const uint16_t* w;
  int M, N, K;
  int64_t x_rs;
  const int32_t* start;  // [E + 1]: first row of every expert (GROUPED)
  int E;
  float* part;           // [S, M, N]: sums of the parts of K (SPLIT)
  int S;
};

DEVINLINE uint32_t wg_pack(float a, float b) {
  typedef __attribute__((ext_vector_type(2))) float f32x2_t;
  typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2_t;
  const f32x2_t v = {a, b};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
}

// Exchange of the 16-byte pieces of row r: the 16 rows of a matrix operand, read
// by a wave at once, lie in different banks.
DEVINLINE int wg_swz(int r) { return (r & 3) | (r >> 1 & 4); }

// Descriptor of `bytes` bytes from p; a load past them reads zeros.
DEVINLINE wg_u32x4 wg_buffer(const uint16_t* p, int64_t bytes) {
  const uint64_t b = (uint64_t)p;
  const int n = bytes > 0x7fffffff ? 0x7fffffff : (int)bytes;
  return wg_u32x4{(uint32_t)__builtin_amdgcn_readfirstlane((int)b),
                  (uint32_t)__builtin_amdgcn_readfirstlane((int)(b >> 32)) &
                      0xffffu,
                  (uint32_t)__builtin_amdgcn_readfirstlane(n), 0x00020000u};
}

// 64 lanes x 16 bytes from memory straight to LDS, 1024 bytes from `at` on.
template <bool ONCE>
DEVINLINE void wg_dma(wg_u32x4 buf, int lane_off, int off, uint32_t at) {
  if (ONCE)
    asm volatile(
        "s_mov_b32 m0, %0\n\ts_nop 0\n\t"
        "buffer_load_dwordx4 %1, %2, %3 offen nt lds" ::"s"(at),
        "v"(lane_off), "s"(buf), "s"(off)
        : "memory", "m0");
  else
    asm volatile(
        "s_mov_b32 m0, %0\n\ts_nop 0\n\t"
        "buffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(at),
        "v"(lane_off), "s"(buf), "s"(off)
        : "memory", "m0");
}

#define WG_INLINE __attribute__((always_inline))

// MT, NT: 16-row tiles of x and of W of one of the 2 x 2 waves.
// GROUPED: rows start[e] .. start[e + 1] - 1 of x with the e-th of E <= 64
// stacked W, known on the device only; an expert's tiles follow each other.
// SPLIT: K in S parts of whole pairs of steps, as even as they go; a part of a tile
// is an item like a tile and its sums go to `part`.
// ONCE: W is read by one patch of tiles and by nontemporal loads, which leave nothing
// in the memory side's cache.
template <int MT, int NT, int GATE, bool GROUPED, bool SPLIT, bool ONCE>
__global__ __launch_bounds__(256, 1) void wide_gemm_kernel(WideArgs a) {
  constexpr bool SWIGLU = GATE != 0;
  constexpr int XB = 32 * MT * WG_BK, WB = 32 * NT * WG_BK;  // of a K step
  constexpr int TM = 32 * MT, TN = SWIGLU ? 16 * NT : 32 * NT;
  __shared__ __attribute__((aligned(1024))) uint16_t lds[2 * XB + 3 * WB];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wr = wave >> 1, wc = wave & 1;
  const int r16 = lane & 15, quad = lane >> 4;
  const int nt = (a.N + TN - 1) / TN;
  int steps = a.K / WG_BK;
  // of this workgroup's tile: the matrix's first row in x and its row count; of
  // expert `lane`: its tiles, those up to it, its first row, its rows
  int base = 0, M = a.M, expert = 0;
  int mine = 0, upto = 0, first = 0, count = 0;
  if (GROUPED) {
    if (lane < a.E) {
      first = a.start[lane];
      count = a.start[lane + 1] - first;
      mine = (count + TM - 1) / TM * nt;
    }
    upto = mine;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int up = __shfl_up(upto, d, 64);
      if (lane >= d) upto += up;
    }
  }
  const int whole = (a.M + TM - 1) / TM * nt;   // tiles of a part of K
  const int tiles = GROUPED ? __builtin_amdgcn_readlane(upto, 63)
                    : SPLIT ? whole * a.S
                            : whole;

  // Tile of round r; -1: none.  A round's tiles are dealt to the XCDs in
  // stretches (ids go round-robin over the XCDs), and a stretch is a patch of
  // 4 row tiles by 8 column tiles, so that an XCD reads 12 operand tiles for 32
  // products (rows first, 2 or 8 of them: up to 4 % slower).
  auto tile_of = [&](int r) WG_INLINE {
    const int left = min(tiles - r * WG_BLOCKS, WG_BLOCKS);
    const int per = (left + 7) >> 3, slot = blockIdx.x >> 3;
    const int at = (blockIdx.x & 7) * per + slot;
    return slot < per && at < left ? r * WG_BLOCKS + at : -1;
  };
  // the part of K of the tile that is loaded, its first entry and its steps
  int part = 0, k0 = 0, own = steps;
  int turn = 0;    // with ONCE: the bytes into its part where a tile starts
  auto origin = [&](int tile, int* m0, int* n0) WG_INLINE {
    if (SPLIT) {
      part = tile / whole;
      tile -= part * whole;
      const int pairs = a.K / (2 * WG_BK);
      const int from = pairs * part / a.S, to = pairs * (part + 1) / a.S;
      k0 = from * 2 * WG_BK;
      own = 2 * (to - from);
    }
    if (GROUPED) {
      expert = __builtin_ctzll(__ballot(upto > tile));
      tile -= __builtin_amdgcn_readlane(upto - mine, expert);
      base = __builtin_amdgcn_readlane(first, expert);
      M = __builtin_amdgcn_readlane(count, expert);
    }
    constexpr int GM = 4;
    const int panel = tile / (GM * nt), in = tile - panel * (GM * nt);
    const int gm = min(GM, (M + TM - 1) / TM - panel * GM);
    *m0 = (panel * GM + in % gm) * TM;
    *n0 = in / gm * TN;
    if (ONCE && (!SPLIT || (MT <= 4 && own >= 24)))
      turn = (max(((int)blockIdx.x >> 3) - in % gm, 0) / gm * 2 +
              ((int)blockIdx.x & 7) * 8) % own * 128;
    else if (ONCE)
      turn = 0;
  };

  // Pieces: 8 rows of 128 bytes, lane / 8 is the row of one; a wave moves every
  // fourth.  LDS rows are in the order of the matrix instructions' rows; which
  // row of W one is, is said here: lanes end up with neighbouring outputs.
  const int prow = wave * 8 + (lane >> 3);
  const int pbyte = ((lane & 7) ^ wg_swz(prow)) * 16;
  wg_u32x4 xbuf, wbuf;
  int xo[MT], wo[NT];
  // With ONCE the workgroups of an XCD start their walks over K (over their part of
  // it) two steps apart and the XCDs eight, and go on from its beginning.  Rows lie a
  // multiple of 4 KB apart, so that a step's lines meet in a sixteenth of the memory
  // channels, and with them those of every workgroup at the same step (us, together
  // and apart: 128256 x 4096, 16 / 61 / 128 / 256 rows, 213 227 239 268 and 165 175 177
  // 241; 28672 x 4096 as SwiGLU, 64 / 65 / 128 rows, 49.6 50.0 56.0 and 44.5 46.6 52.4;
  // Mixtral's experts, 176 tokens, a step 769 and 678; 4096 x 14336 in parts, 65 / 96 /
  // 128 rows, 31.4 33.6 36.6 and 27.3 30.5 34.5, but short parts and 200 rows 1 to 4 %
  // slower; rows of 10 KB the same).  With every XCD's first at the same step 32768 x
  // 4096, whose XCDs lie 16 MB apart, took 75 us at 64 rows, and takes 44.  Rows of
  // tiles that share W start together.  (By the column of tiles, two steps each, 28672
  // x 4096 took 59 us: its address and the start cancel out in the channel.)
  int xturn = 0, wturn = 0, xwrap = 0, wwrap = 0;   // bytes
  auto turned = [&](int k, int by, int wrap) WG_INLINE {
    const int r = k + by;
    return ONCE && r >= wrap ? r - wrap : r;
  };
  auto x_from = [&](int m0) WG_INLINE {
    if (ONCE) {
      xturn = turn;
      xwrap = own * 128;
    }
    xbuf = wg_buffer(a.x + (base + m0) * a.x_rs + k0,
                     ((M - 1 - m0) * a.x_rs + a.K - k0) * 2);
#pragma unroll
    for (int i = 0; i < MT; ++i)
      xo[i] = min(i * 32 + prow, M - 1 - m0) * ((int)a.x_rs * 2) + pbyte;
  };
  auto w_from = [&](int n0) WG_INLINE {
    if (ONCE) {
      wturn = turn;
      wwrap = own * 128;
    }
    const int rows = SWIGLU ? 2 * a.N : a.N;
    wbuf = wg_buffer(a.w + ((int64_t)expert * rows + n0) * a.K + k0,
                     ((int64_t)(rows - n0) * a.K - k0) * 2);
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      const int r = i * 32 + prow, half = r >= 16 * NT, in = r - half * 16 * NT;
      const int t = in >> 4, q = in >> 2 & 3, e = in & 3;
      int n;
      if (SWIGLU)
        n = half * 8 * NT +
            (t < (NT & ~3)   ? (t >> 2) * 32 + q * 8 + (t & 3) * 2 + (e & 1)
             : t < (NT & ~1) ? (NT & ~3) * 8 + q * 4 + (t & 1) * 2 + (e & 1)
                             : (NT - 1) * 8 + q * 2 + (e & 1));
      else
        n = half * 16 * NT + (t < (NT & ~1)
                                  ? (t >> 1) * 32 + q * 8 + (t & 1) * 4 + e
                                  : t * 16 + q * 4 + e);
      n = min(n, a.N - 1 - n0);
      if (SWIGLU) n += (e >> 1) * a.N;
      wo[i] = n * (a.K * 2) + pbyte;
    }
  };
  const uint32_t lds0 =
      (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint16_t*)lds +
      wave * 8 * WG_BK * 2;
  auto load_x = [&](int i, int off, int buf) WG_INLINE {
    wg_dma<false>(xbuf, xo[i], turned(off, xturn, xwrap),
                  lds0 + (buf + i * 32 * WG_BK) * 2);
  };
  auto load_w = [&](int i, int off, int buf) WG_INLINE {
    wg_dma<ONCE>(wbuf, wo[i], turned(off, wturn, wwrap),
                 lds0 + (buf + i * 32 * WG_BK) * 2);
  };
  // a lane's 8 entries of the first half of a K step, and of the second
  const int f0 = r16 * WG_BK + ((quad ^ wg_swz(r16)) << 3), f1 = f0 ^ 32;
  const int fx0 = f0 + wr * 16 * MT * WG_BK, fx1 = f1 + wr * 16 * MT * WG_BK;
  const int fw0 = f0 + wc * 16 * NT * WG_BK, fw1 = f1 + wc * 16 * NT * WG_BK;
  auto frag = [&](int at, int t) WG_INLINE {
    return *reinterpret_cast<const wg_bf16x8*>(lds + at + t * 16 * WG_BK);
  };

  wg_f32x4 acc[MT][NT];
  wg_bf16x8 fx[2][MT], fw[2][NT];
  // The products of half a K step, from fragments c; between them the fragments
  // of the next half are read (xs, ws) and, with LOAD, the pieces of later
  // steps sent for, x first as it is waited for first.
  auto half = [&](auto first, auto load, int c, int xs, int ws, int xd, int xk,
                  int wd, int wk) WG_INLINE {
    constexpr bool FIRST = decltype(first)::value, LOAD = decltype(load)::value;
    constexpr int G = 2 * MT, R = MT + NT;
#pragma unroll
    for (int g = 0; g < G; ++g) {
#pragma unroll
      for (int j = (R * g + G - 1) / G; j * G < R * (g + 1); ++j) {
        if (j < NT) fw[1 - c][j] = frag(ws, j);
        else fx[1 - c][j - NT] = frag(xs, j - NT);
        if (LOAD) {
          if (j < MT) load_x(j, xk, xd);
          else load_w(j - MT, wk, wd);
        }
      }
      const int m = g >> 1;
      constexpr int N0 = (NT + 1) / 2;
#pragma unroll
      for (int n = g & 1 ? N0 : 0; n < (g & 1 ? NT : N0); ++n)
        acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            fw[c][n], fx[c][m],
            FIRST ? wg_f32x4{0.0f, 0.0f, 0.0f, 0.0f} : acc[m][n], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  int round = 0;
  int w0 = 2 * XB, w1 = 2 * XB + WB, w2 = 2 * XB + 2 * WB;
  using Yes = std::true_type;
  using No = std::false_type;
  // K step in (xc, w0), the next one in (xn, w1).  Behind the barrier every
  // wave has read the step's fragments and everything of the next step is
  // there: the x of the step after it goes to xc, the W of the third to w0.  W
  // comes from HBM and has two steps and a half to arrive, x is shared by more
  // workgroups and has one and a half.
  auto step = [&](auto first, bool tile_start, int xc, int xn, int xk,
                  int wk) WG_INLINE {
    half(first, No{}, 0, xc + fx1, w0 + fw1, 0, 0, 0, 0);
    if (!tile_start)
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(NT) : "memory");
    else   // stores are under way; what is needed was waited for before them
      asm volatile(
          "s_waitcnt lgkmcnt(0)\n\ts_cmp_lg_u32 %0, 0\n\t"
          "s_cbranch_scc1 1f\n\ts_waitcnt vmcnt(%1)\n1:" ::"s"(round),
          "n"(NT)
          : "memory", "scc");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    half(No{}, Yes{}, 1, xn + fx0, w1 + fw0, xc, xk, w0, wk);
    const int f = w0;
    w0 = w1;
    w1 = w2;
    w2 = f;
  };

  int tile = tile_of(0), m0, n0;
  if (tile < 0) return;
  origin(tile, &m0, &n0);
  x_from(m0);
  w_from(n0);
#pragma unroll
  for (int j = 0; j < 3; ++j) {
#pragma unroll
    for (int i = 0; i < MT; ++i)
      if (j < 2) load_x(i, j * 128, j * XB);
#pragma unroll
    for (int i = 0; i < NT; ++i) load_w(i, j * 128, 2 * XB + j * WB);
  }
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(MT + 2 * NT) : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
#pragma unroll
  for (int j = 0; j < NT; ++j) fw[0][j] = frag(w0 + fw0, j);
#pragma unroll
  for (int j = 0; j < MT; ++j) fx[0][j] = frag(fx0, j);
  for (;;) {
    step(Yes{}, true, 0, XB, 256, 384);
    step(No{}, false, XB, 0, 384, 512);
    const int next = tile_of(++round);
    const int mc = m0, nc = n0, Mc = M;
    uint16_t* const oc = a.out + (int64_t)base * a.N;
    float* const pc = SPLIT ? a.part + (int64_t)part * M * a.N : nullptr;
    if (SPLIT) steps = own;
    origin(next < 0 ? tile : next, &m0, &n0);
    int k = 512;
    for (int t = 2; t < steps - 4; t += 2, k += 256) {
      step(No{}, false, 0, XB, k, k + 128);
      step(No{}, false, XB, 0, k + 128, k + 256);
    }
    // the next tile's first steps are under way before this one's results are
    // stored (past the last tile, this one's once more)
    step(No{}, false, 0, XB, k, k + 128);
    w_from(n0);
    step(No{}, false, XB, 0, k + 128, 0);
    x_from(m0);
    step(No{}, false, 0, XB, 0, 128);
    step(No{}, false, XB, 0, 128, 256);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NT) : "memory");

#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const int row = mc + (wr * MT + m) * 16 + r16;
      uint16_t* out = oc + (int64_t)row * a.N;
      if (SPLIT) {
        static_assert(!SPLIT || (!SWIGLU && NT % 2 == 0));
        float* sums = pc + (int64_t)row * a.N;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          const int at = nc + wc * 16 * NT + t / 2 * 32 + quad * 8 + t % 2 * 4;
          if (row < Mc && at < a.N)
            *reinterpret_cast<wg_f32x4*>(sums + at) = acc[m][t];
        }
      } else if (SWIGLU) {
        auto act = [&](int t, int e) WG_INLINE {
          return gate_act<GATE>(acc[m][t][e]) * acc[m][t][e + 2];
        };
        auto pair = [&](int t) WG_INLINE {
          return wg_pack(act(t, 0), act(t, 1));
        };
        const int n = nc + wc * 8 * NT;
#pragma unroll
        for (int t = 0; t < (NT & ~3); t += 4) {
          const wg_u32x4 y = {pair(t), pair(t + 1), pair(t + 2), pair(t + 3)};
          const int at = n + t * 8 + quad * 8;
          if (row < Mc && at < a.N)
            *reinterpret_cast<wg_u32x4*>(out + at) = y;
        }
        if (NT & 2) {
          constexpr int t = NT & ~3;
          const wg_u32x2 y = {pair(t), pair(t + 1)};
          const int at = n + t * 8 + quad * 4;
          if (row < Mc && at < a.N)
            *reinterpret_cast<wg_u32x2*>(out + at) = y;
        }
        if (NT & 1) {
          const uint32_t y = pair(NT - 1);
          const int at = n + (NT - 1) * 8 + quad * 2;
          if (row < Mc && at < a.N) *reinterpret_cast<uint32_t*>(out + at) = y;
        }
      } else {
        const int n = nc + wc * 16 * NT;
        auto pair = [&](int t, int e) WG_INLINE {
          return wg_pack(acc[m][t][e], acc[m][t][e + 1]);
        };
#pragma unroll
        for (int t = 0; t < (NT & ~1); t += 2) {
          const wg_u32x4 y = {pair(t, 0), pair(t, 2), pair(t + 1, 0),
                              pair(t + 1, 2)};
          const int at = n + t * 16 + quad * 8;
          if (row < Mc && at < a.N)
            *reinterpret_cast<wg_u32x4*>(out + at) = y;
        }
        if (NT & 1) {
          const wg_u32x2 y = {pair(NT - 1, 0), pair(NT - 1, 2)};
          const int at = n + (NT - 1) * 16 + quad * 4;
          if (row < Mc && at < a.N)
            *reinterpret_cast<wg_u32x2*>(out + at) = y;
        }
      }
    }
    if (next < 0) break;
    tile = next;
  }
  // the last pieces land in LDS that is this workgroup's until it ends
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

}  // namespace igw
