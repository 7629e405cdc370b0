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
#include <ATen/cuda/CUDAContext.h>
#include <c10/cuda/CUDAGuard.h>
#include <torch/extension.h>

#include <cmath>
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
  int part = 0, k0 = 0, own = 0;
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
  };

  // Pieces: 8 rows of 128 bytes, lane / 8 is the row of one; a wave moves every
  // fourth.  LDS rows are in the order of the matrix instructions' rows; which
  // row of W one is, is said here: lanes end up with neighbouring outputs.
  const int prow = wave * 8 + (lane >> 3);
  const int pbyte = ((lane & 7) ^ wg_swz(prow)) * 16;
  wg_u32x4 xbuf, wbuf;
  int xo[MT], wo[NT];
  auto x_from = [&](int m0) WG_INLINE {
    xbuf = wg_buffer(a.x + (base + m0) * a.x_rs + k0,
                     ((M - 1 - m0) * a.x_rs + a.K - k0) * 2);
#pragma unroll
    for (int i = 0; i < MT; ++i)
      xo[i] = min(i * 32 + prow, M - 1 - m0) * ((int)a.x_rs * 2) + pbyte;
  };
  auto w_from = [&](int n0) WG_INLINE {
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
    wg_dma<false>(xbuf, xo[i], off, lds0 + (buf + i * 32 * WG_BK) * 2);
  };
  auto load_w = [&](int i, int off, int buf) WG_INLINE {
    wg_dma<ONCE>(wbuf, wo[i], off, lds0 + (buf + i * 32 * WG_BK) * 2);
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

// Tiles of 32 * MT rows by 32 * NT rows of W, and what a round of 256 of them
// costs in hundredths of one of 256 x 256 (K = 4096, 1024 to 16000 rows: 95 us).
struct WideTile {
  int MT, NT, cost;
};
static constexpr WideTile wide_tiles[] = {
    {8, 8, 100}, {8, 7, 91}, {8, 6, 82}, {6, 8, 82}, {4, 8, 66}};

// The tile that M rows and N outputs take the least time on, by whole rounds of
// the 256 compute units; 0: this kernel is not ahead of the library.
//
// With SWIGLU the library has a second launch that reads the product back, 10 %
// of its time at K = 4096, and is behind wherever half of the compute units
// have a tile (us, library with silu_mul and here: 256 x 28672 x 4096 79.1 and
// 69.6; 1024 rows 197 and 170, 3000 575 and 506, 16000 2804 and 2590; 1024 x
// 35840 x 5120 393 and 283, 128 rows 104 and 93; 1024 x 7168 x 4096 58.0 and
// 49.1), not below (128 x 28672 x 4096, 112 tiles: 62.3 and 68.1; 512 x 7168 x
// 4096 37.7 and 44.2).  Over a long K the second launch weighs less: 2033 x
// 7168 x 8192 167 and 172, 4096 x 57344 x 8192 2548 and 2591, but 1024 rows of
// the latter 773 and 658.  As a plain product the library reaches 1.55 PFLOP/s
// where its own tiles fill the rounds, this kernel 1.45; ahead is a vocabulary's
// width of hundreds of rows, from more of them on the longer K is (65536 to 262144
// outputs x 512 to 8192; of the library's time at 257 to 320 rows 0.63 to 1.15 up to K
// = 4096, 0.94 to 1.35 at 6144; 321 to 640 rows 0.47 to 1.19 up to 6144, 0.83 to 1.1 at
// 8192; 641 to 1024 rows 0.53 to 1.08; 128256 x 4096 at 288, 384 and 1024 rows 0.80,
// 0.75 and 0.87, 892 us and 776).  Of 256 rows and of more than 1024 it is as often
// behind (65536 x 8192, 256 rows, 232 and 264; 98304 x 2048, 1500 rows, 11 %; 131072
// x 4096, 2048 rows, 1 %, where 128256 is 6 % ahead).
int64_t wide_gemm_tile(int64_t M, int64_t N, int64_t K, bool swiglu) {
  if (M < 65 || K < 6 * WG_BK || K % (2 * WG_BK) != 0 || N < 8 || N % 8 != 0)
    return 0;
  int64_t best = 0, least = 0, tiles = 0;
  for (const auto& c : wide_tiles) {
    const int64_t tm = 32 * c.MT, tn = (swiglu ? 16 : 32) * c.NT;
    const int64_t n = ((M + tm - 1) / tm) * ((N + tn - 1) / tn);
    const int64_t cost = (n + WG_BLOCKS - 1) / WG_BLOCKS * c.cost;
    if (best == 0 || cost < least) {
      best = c.MT * 16 + c.NT;
      least = cost;
      tiles = n;
    }
  }
  if (swiglu) return tiles >= WG_BLOCKS / 2 && (K < 8192 || M <= 1536) ? best : 0;
  const int64_t from = K <= 4096 ? 257 : K <= 6144 ? 321 : 641;
  return N >= 65536 && K <= 8192 && M >= from && M <= 1024 ? best : 0;
}

// Whether the kernel's 32-bit offsets reach everything: rows of x in a tile,
// and with SWIGLU all of W.
bool wide_gemm_fits(int64_t x_rs, int64_t N, int64_t K, bool swiglu) {
  return x_rs < (1 << 21) && K < (1 << 21) &&
         (!swiglu || 2 * N * K < (int64_t)1 << 30);
}

// Up to this many rows a gated product reads W once and by nontemporal loads (us, plain
// and so: 28672 x 4096, 200 / 256 / 384 / 512 rows 70.4 73.3 82.9 96.7 and 66.8 69.4 80.2
// 94.1, 35840 x 5120 103 113 153 169 and 98.4 100 160 165; 8192 rows, where W comes
// back from the caches for every patch of tiles, 1 % behind).
constexpr int64_t WIDE_ONCE = 256;

void wide_gemm(torch::Tensor out, torch::Tensor x, torch::Tensor w,
               int64_t gate, int64_t tile) {
  const bool swiglu = gate != 0;
  TORCH_CHECK(gate >= 0 && gate <= 2);
  TORCH_CHECK(x.is_cuda() && x.dim() == 2 && x.stride(1) == 1 &&
              x.dtype() == torch::kBFloat16 && w.dtype() == x.dtype() &&
              w.dim() == 2 && w.is_contiguous() && out.dim() == 2 &&
              out.is_contiguous() && out.dtype() == x.dtype());
  const int64_t M = x.size(0), K = x.size(1), N = out.size(1);
  TORCH_CHECK(M >= 1 && N >= 8 && N % 8 == 0 && K >= 6 * WG_BK &&
              K % (2 * WG_BK) == 0 && M < (1 << 30) && N < (1 << 30) &&
              wide_gemm_fits(x.stride(0), N, K, swiglu));
  TORCH_CHECK(out.size(0) == M && w.size(1) == K &&
              w.size(0) == (swiglu ? 2 * N : N) && x.stride(0) % 8 == 0);
  TORCH_CHECK(w.device() == x.device() && out.device() == x.device(),
              "tensors on different devices");
  for (const auto* t : {&out, &x, &w})
    TORCH_CHECK((reinterpret_cast<uintptr_t>(t->data_ptr()) & 15) == 0);
  const at::cuda::CUDAGuard guard(x.device());
  hipStream_t stream = at::cuda::getCurrentCUDAStream();
  const WideArgs a{(uint16_t*)out.data_ptr(), (const uint16_t*)x.data_ptr(),
                   (const uint16_t*)w.data_ptr(), (int)M, (int)N, (int)K,
                   x.stride(0), nullptr, 0, nullptr, 1};
  const bool once = M <= WIDE_ONCE;
#define LAUNCH_WIDE_AS(...)                                                   \
  hipLaunchKernelGGL((wide_gemm_kernel<__VA_ARGS__>), dim3(WG_BLOCKS),        \
                     dim3(256), 0, stream, a)
#define LAUNCH_WIDE(MT, NT)                                                   \
  case MT * 16 + NT:                                                          \
    if (gate == 2 && once)                                                    \
      LAUNCH_WIDE_AS(MT, NT, 2, false, false, true);                          \
    else if (gate == 2)                                                       \
      LAUNCH_WIDE_AS(MT, NT, 2, false, false, false);                         \
    else if (gate == 1 && once)                                               \
      LAUNCH_WIDE_AS(MT, NT, 1, false, false, true);                          \
    else if (gate == 1)                                                       \
      LAUNCH_WIDE_AS(MT, NT, 1, false, false, false);                         \
    else                                                                      \
      LAUNCH_WIDE_AS(MT, NT, 0, false, false, false);                         \
    break
  switch (tile) {
    LAUNCH_WIDE(8, 8);
    LAUNCH_WIDE(8, 7);
    LAUNCH_WIDE(8, 6);
    LAUNCH_WIDE(6, 8);
    LAUNCH_WIDE(4, 8);
    default: TORCH_CHECK(false, "no such tile: ", tile);
  }
#undef LAUNCH_WIDE
#undef LAUNCH_WIDE_AS
  HIP_CHECK_KERNEL();
}

// Products of rows that leave the chip idle, K in parts.
//
// Tiles of the kernel above with a part of K each, their fp32 sums to memory, and a
// second kernel to add them (with the residual and the norm behind it where there is
// one).  wide_split picks the tile and the parts by what they cost: rounds of 256
// items at `step` us a K step of 64 and `start` to begin, against W from HBM, and
// the sums' way to memory and back.  Of 768 measured pairs of a tile and parts the
// model is off by 4 % on average, and its choice is 2 % behind the best.
struct SplitTile {
  int MT, NT;
  double step;
};
static constexpr SplitTile split_tiles[] = {
    {3, 4, 0.500}, {4, 4, 0.567}, {4, 6, 0.712}, {6, 4, 0.671}, {6, 6, 0.845},
    {6, 8, 1.069}, {8, 4, 0.799}, {8, 6, 1.049}, {8, 8, 1.387}};

// 256 times the tile (16 MT + NT) and the parts of K, at least two; 0: cannot be.
int64_t wide_split(int64_t M, int64_t N, int64_t K) {
  if (M < 65 || M > (1 << 16) || N < 8 || N % 8 != 0 || N > (1 << 20) ||
      K % (2 * WG_BK) != 0 || K > (1 << 20))
    return 0;
  int64_t best = 0;
  double least = 0.0;
  const int64_t pairs = K / (2 * WG_BK);
  for (const auto& c : split_tiles)
    for (int64_t S = 2; S <= 16 && 3 * S <= pairs; ++S) {
      const int64_t items = (M + 32 * c.MT - 1) / (32 * c.MT) *
                            ((N + 32 * c.NT - 1) / (32 * c.NT)) * S;
      const int64_t rounds = (items + WG_BLOCKS - 1) / WG_BLOCKS;
      const double work =
          rounds * (2 * ((pairs + S - 1) / S) * c.step + 0.11);
      const double stream = N * K * 2e-6 / 4.6;
      // about the longer of the two
      const double a = work * work, b = stream * stream;
      const double cost =
          std::sqrt(std::sqrt(a * a + b * b)) + S * M * N * 4e-6 * 0.36;
      if (best == 0 || cost < least) {
        best = (c.MT * 16 + c.NT) * 256 + S;
        least = cost;
      }
    }
  return best;
}

// Whether that is ahead of the library; norm: where the norm that follows adds the
// parts, of the library and fused_add_rmsnorm.  Measured at 19 sizes of W by 16 of
// 65 to 2600 rows (us, library and here; then with the norm).  Over a long K the
// library's tiles are few: 4096 x 14336, 65 / 128 / 256 / 512 / 1024 / 2033 rows 50.6
// 76.5 63.8 90.9 134 204 and 36.1 38.9 49.3 65.7 108 185; 5120 x 17920, 65 / 256 / 1024
// 148 222 249 and 45.8 65.1 158, but 2033 rows 291 and 320; 8192 x 28672, 512 / 640
// rows 312 260 and 195 289.  Of squarer W the parts' way to memory weighs more: 4096 x
// 4096, 128 / 256 / 512 / 1024 / 1600 rows 24.0 22.4 30.9 42.1 55.6 and 18.0 21.8 30.7
// 43.4 66.9 (with the norm 27.2 25.9 36.0 48.9 65.4 and 19.1 23.1 32.6 46.1 70.2), 5120
// x 5120, 256 / 640 / 1024 rows 50.8 51.3 62.7 and 30.7 47.5 60.7, 7680 x 5120, 128 /
// 512 / 640 rows 34.9 52.1 58.0 and 28.0 51.0 63.6, 6144 x 4096, 128 / 160 / 200 rows
// 26.5 29.1 26.5 and 23.8 26.1 30.0, 8192 x 8192, 65 / 128 rows 38.9 51.8 and 43.6
// 46.6.  Small W and a short K pay for the second launch: 1024 x 4096, 128 rows, 10.3
// and 11.9, 4096 x 2048 13.1 and 15.4, as do wide ones: 16384 x 4096 40.3 and 46.9.
bool wide_split_ahead(int64_t M, int64_t N, int64_t K, bool norm) {
  if (wide_split(M, N, K) == 0) return false;
  const int64_t least = N > 7680 && K < 2 * N ? 128 : 65;
  int64_t most;
  if (norm) {
    if (K < 3584 || N * K < (int64_t)12 << 20 || N > 16384) return false;
    most = K >= 3 * N   ? N > 5120 ? 512 : N > 4096 ? 1600 : 2048
           : K >= 2 * N ? N > 5120 ? 512 : 1600
           : K >= N     ? N > 7680 ? 512 : 1024
                        : 512;
  } else {
    if (K < 4096 || N * K < (int64_t)16 << 20 || N < 2048 || N > 10240)
      return false;
    most = K >= 3 * N   ? N > 5120 ? 512 : N > 4096 ? 1600 : 2048
           : K >= 2 * N ? N > 5120 ? 512 : 1300
           : K >= 5120  ? 512
           : K >= N     ? 256
                        : 160;
  }
  return M >= least && M <= most;
}

// The sums [S, M, N] of the parts that wide_split says.
torch::Tensor split_parts(const torch::Tensor& x, const torch::Tensor& w,
                          int64_t tile, int64_t S) {
  TORCH_CHECK(x.is_cuda() && x.dim() == 2 && x.stride(1) == 1 &&
              x.dtype() == torch::kBFloat16 && w.dtype() == x.dtype() &&
              w.dim() == 2 && w.is_contiguous());
  const int64_t M = x.size(0), K = x.size(1), N = w.size(0);
  TORCH_CHECK(M >= 1 && N >= 8 && N % 8 == 0 && S >= 1 && S <= 64 &&
              K / (2 * WG_BK) >= 3 * S && K % (2 * WG_BK) == 0 &&
              M <= (1 << 20) && N <= (1 << 20) && K <= (1 << 20) &&
              wide_gemm_fits(x.stride(0), N, K, false));
  TORCH_CHECK(w.size(1) == K && x.stride(0) % 8 == 0);
  TORCH_CHECK(w.device() == x.device(), "tensors on different devices");
  for (const auto* t : {&x, &w})
    TORCH_CHECK((reinterpret_cast<uintptr_t>(t->data_ptr()) & 15) == 0);
  const at::cuda::CUDAGuard guard(x.device());
  hipStream_t stream = at::cuda::getCurrentCUDAStream();
  auto part = torch::empty({S, M, N}, x.options().dtype(torch::kFloat32));
  const WideArgs a{nullptr, (const uint16_t*)x.data_ptr(),
                   (const uint16_t*)w.data_ptr(), (int)M, (int)N, (int)K,
                   x.stride(0), nullptr, 0, part.data_ptr<float>(), (int)S};
  // nontemporal where one patch of tiles has all rows (8192 x 28672, 65 / 256 / 1024
  // rows 107 154 347 and 91 131 337)
#define LAUNCH_SPLIT_AS(...)                                                  \
  hipLaunchKernelGGL((wide_gemm_kernel<__VA_ARGS__>), dim3(WG_BLOCKS),        \
                     dim3(256), 0, stream, a)
#define LAUNCH_SPLIT(MT, NT)                                                  \
  case MT * 16 + NT:                                                          \
    if (M <= 4 * 32 * MT) LAUNCH_SPLIT_AS(MT, NT, 0, false, true, true);      \
    else LAUNCH_SPLIT_AS(MT, NT, 0, false, true, false);                      \
    break
  switch (tile) {
    LAUNCH_SPLIT(3, 4);
    LAUNCH_SPLIT(4, 4);
    LAUNCH_SPLIT(4, 6);
    LAUNCH_SPLIT(6, 4);
    LAUNCH_SPLIT(6, 6);
    LAUNCH_SPLIT(6, 8);
    LAUNCH_SPLIT(8, 4);
    LAUNCH_SPLIT(8, 6);
    LAUNCH_SPLIT(8, 8);
    default: TORCH_CHECK(false, "no such tile: ", tile);
  }
#undef LAUNCH_SPLIT
#undef LAUNCH_SPLIT_AS
  HIP_CHECK_KERNEL();
  return part;
}

// Tiles of a grouped product and what a round of them costs (hundredths of one
// of 256 x 256 over many rounds: fewer columns or rows come cheaper there than
// above, where the rounds are few).
static constexpr WideTile grouped_tiles[] = {
    {8, 8, 98}, {8, 7, 85}, {6, 8, 77}, {6, 7, 69}, {4, 8, 57}, {4, 6, 45}};

// The tile for `rows` rows that E experts share.  How many each has is known on
// the device only; they spread by about the root of the mean, and four points
// of that spread stand for the tiles that whole rounds are counted for
// (us, by 16-row tiles of x and W; eight experts of 4096 and 14336: 4200 rows,
// up 88 1008, 87 962, 68 837, 67 836, 48 986, down 617 599 527 483 566; 2048
// rows, up 621 590 670 674 551, down 342 340 310 475 387; 128 rows, up 435 386
// 394 365 372 and 46 356, down 263 267 241 203 204 and 175).
int64_t grouped_tile(int64_t rows, int64_t E, int64_t N, bool swiglu) {
  const double r = (double)rows / (double)E, s = std::sqrt(r);
  int64_t best = 0;
  double least = 0.0;
  for (const auto& c : grouped_tiles) {
    const int64_t nt = (N + (swiglu ? 16 : 32) * c.NT - 1) /
                       ((swiglu ? 16 : 32) * c.NT);
    double m = 0.0;
    for (const double at : {r - 1.5 * s, r - 0.5 * s, r + 0.5 * s, r + 1.5 * s})
      m += std::max(1.0, std::ceil(at / (32 * c.MT))) / 4.0;
    const double cost = std::ceil(m * (E * nt) / WG_BLOCKS) * c.cost;
    if (best == 0 || cost < least) {
      best = c.MT * 16 + c.NT;
      least = cost;
    }
  }
  return best;
}

// out[r] = x[r] W_e^T for the rows start[e] .. start[e + 1] - 1 of every expert
// e, w [E, N or 2 N, K]; rows past start[E] are left alone.
void grouped_gemm(torch::Tensor out, torch::Tensor x, torch::Tensor w,
                  torch::Tensor start, bool swiglu, int64_t tile) {
  TORCH_CHECK(x.is_cuda() && x.dim() == 2 && x.is_contiguous() &&
              x.dtype() == torch::kBFloat16 && w.dtype() == x.dtype() &&
              w.dim() == 3 && w.is_contiguous() && out.dim() == 2 &&
              out.is_contiguous() && out.dtype() == x.dtype() &&
              start.dtype() == torch::kInt32 && start.is_contiguous());
  const int64_t R = x.size(0), K = x.size(1), N = out.size(1), E = w.size(0);
  TORCH_CHECK(R >= 1 && E >= 1 && E <= 64 && start.numel() == E + 1 && N >= 8 &&
              N % 8 == 0 && K >= 6 * WG_BK && K % (2 * WG_BK) == 0 &&
              R < (1 << 30) && N < (1 << 30) && wide_gemm_fits(K, N, K, swiglu));
  TORCH_CHECK(out.size(0) == R && w.size(2) == K &&
              w.size(1) == (swiglu ? 2 * N : N));
  TORCH_CHECK(w.device() == x.device() && out.device() == x.device() &&
                  start.device() == x.device(),
              "tensors on different devices");
  for (const auto* t : {&out, &x, &w})
    TORCH_CHECK((reinterpret_cast<uintptr_t>(t->data_ptr()) & 15) == 0);
  const at::cuda::CUDAGuard guard(x.device());
  hipStream_t stream = at::cuda::getCurrentCUDAStream();
  const WideArgs a{(uint16_t*)out.data_ptr(), (const uint16_t*)x.data_ptr(),
                   (const uint16_t*)w.data_ptr(), (int)R, (int)N, (int)K, K,
                   (const int32_t*)start.data_ptr(), (int)E, nullptr, 1};
  // nontemporal W where one patch of tiles has an expert's rows (three prompts of
  // 560 to 700 tokens on eight experts of 14336 x 4096: a step 1442 and 1330 us)
#define LAUNCH_GROUPED_AS(...)                                                \
  hipLaunchKernelGGL((wide_gemm_kernel<__VA_ARGS__>), dim3(WG_BLOCKS),        \
                     dim3(256), 0, stream, a)
#define LAUNCH_GROUPED(MT, NT)                                                \
  case MT * 16 + NT:                                                          \
    if (swiglu && R <= E * 4 * 32 * MT)                                       \
      LAUNCH_GROUPED_AS(MT, NT, 1, true, false, true);                        \
    else if (swiglu)                                                          \
      LAUNCH_GROUPED_AS(MT, NT, 1, true, false, false);                       \
    else if (R <= E * 4 * 32 * MT)                                            \
      LAUNCH_GROUPED_AS(MT, NT, 0, true, false, true);                        \
    else                                                                      \
      LAUNCH_GROUPED_AS(MT, NT, 0, true, false, false);                       \
    break
  switch (tile > 0 ? tile : grouped_tile(R, E, N, swiglu)) {
    LAUNCH_GROUPED(8, 8);
    LAUNCH_GROUPED(8, 7);
    LAUNCH_GROUPED(6, 8);
    LAUNCH_GROUPED(6, 7);
    LAUNCH_GROUPED(4, 8);
    LAUNCH_GROUPED(4, 6);
    default: TORCH_CHECK(false, "no such tile: ", tile);
  }
#undef LAUNCH_GROUPED
#undef LAUNCH_GROUPED_AS
  HIP_CHECK_KERNEL();
}

}  // namespace igw
