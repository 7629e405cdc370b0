// Prompt attention on MFMA tiles (gfx950, bf16): the part that the engine's
// prompt attentions share.  A workgroup of four waves owns 128 query rows of
// one head, 32 per wave, and walks the keys they can see 64 at a time.
//
// What bounds it: per score NK + NV MFMA multiply-adds, and on the vector
// units one max, one multiply-add, one exponential (quarter rate), one add
// (fp32, of the weight before it is rounded) and half a conversion, at NK = NV
// = 128 about as many cycles as the MFMAs take.  The design keeps everything
// else off those two units:
//
//   * S^T = K Q^T with mfma_f32_32x32x16_bf16: a lane then holds 16 keys of
//     ONE query row per tile, so row maxima and sums are in-lane, with one
//     exchange between lane halves per 64 keys (the sums only at the end);
//   * O^T += V^T P^T: the C layout of S^T (keys 8a + 4h + 0..3 of lane half
//     h) is fed to the B operand as it is, the key order inside the
//     contraction being free as long as V^T is read in the same order, so
//     the probabilities never leave their registers;
//   * V stays row-major in LDS, ds_read_b64_tr_b16 transposes 4 keys x 16
//     dims on the way to the A operand (no transposing stores);
//   * K and V tiles go from global memory straight to LDS, the next tile
//     being fetched while this one is used: two buffers, one barrier a tile,
//     four LDS objects so that the reads of one buffer do not wait for the
//     writes to the other;
//   * 16-byte chunks are XOR-swizzled by row (on the global side, a DMA
//     writes LDS linearly): K so that the 16 rows that the LDS serves at a time
//     of a fragment's 32 (0-3, 12-15, 20-27, and the rest) lie in different
//     banks, V by the rows that one transposing read spreads over its lanes;
//   * the accumulators are rescaled only where a row of the wave has a new
//     maximum, which gets rare along the keys (raising it only when it is
//     outgrown by 2^8 leaves the largest weight another value than one and
//     rounds it for the product: up to 10 % more error against 64 bits);
//   * masks are evaluated only in tiles that some row of the wave sees in
//     part, and a wave skips tiles that none of its rows sees.
//
// Two waves per SIMD (256 registers, up to 80 KB of LDS per workgroup) let
// one wave's softmax run beside the other's MFMAs.  A wave waits a fifth of its
// time (for LDS reads and its workgroup), so what it can it has under way: K
// fragments four products ahead, V one step, the weights of the second 32 keys
// between the products of the first.  Next to nothing is left of the addresses
// of tiles that lie whole in one sequence.  One prompt of 16000 tokens, 32
// heads on 8, before and after these, alone and on one card: 2290 and 2148 us, of
// 4000 178 and 157, 16 of 512 77 and 70, 2000 rows behind 6000 277 and 256 (on
// another card 1979, 146, 71 and 236 after them).  Computing the next
// tile's scores beside this one's weights wants more registers than there are.
#pragma once

#include <climits>
#include <type_traits>

#include "common.h"

namespace igw {

typedef __attribute__((ext_vector_type(4))) short ft_short4;
typedef __attribute__((ext_vector_type(2))) __bf16 ft_bf16x2;
typedef __attribute__((ext_vector_type(8))) __bf16 ft_bf16x8;
typedef __attribute__((ext_vector_type(16))) float ft_f32x16;

constexpr int FT_BN = 64;    // keys per tile
constexpr int FT_WAVES = 4;  // waves per workgroup, 32 query rows each
constexpr int FT_BM = 32 * FT_WAVES;
#define FT_INLINE __attribute__((always_inline))
// classes of instructions, as __builtin_amdgcn_sched_group_barrier names them
constexpr int FT_VALU = 0x2, FT_MFMA = 0x8, FT_DS_READ = 0x100;
constexpr float FT_LOG2E = 1.44269504088896340736f;

// two floats -> packed bf16 pair, round to nearest even
DEVINLINE uint32_t ft_pack_bf16(float a, float b) {
  typedef __attribute__((ext_vector_type(2))) float f32x2_t;
  const f32x2_t v = {a, b};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, ft_bf16x2));
}

// x of lane i and of lane i ^ 32, in both lanes: a = lower half's value, b =
// upper half's.  Written out because the compiler folds the builtin's two
// results into one when its operands are equal; the s_nop is the wait that
// the swap needs behind the instruction that wrote its operands.
DEVINLINE void ft_both_halves(float x, float& a, float& b) {
  a = b = x;
  asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 0" : "+v"(a), "+v"(b));
}

// Head and tile of a workgroup in a grid of ntiles * heads.  Ids go
// round-robin over the 8 XCDs: heads are dealt to id % 8, so heads that share
// keys run on one XCD, the tiles of a head follow each other there, the last
// (longest) tiles of each prompt first.
DEVINLINE void ft_head_and_tile(int heads, int ntiles, int* head, int* tile) {
  const int id = blockIdx.x;
  if (heads % 8 == 0) {
    const int hp = heads >> 3, local = id >> 3;
    *head = (id & 7) * hp + local % hp;
    *tile = ntiles - 1 - local / hp;
  } else {
    *head = id % heads;
    *tile = ntiles - 1 - id / heads;
  }
}

// Sequence and row offset of tile t when each of the B sequences of cu takes
// ceil(rows / BM) tiles (found here: a tile map made on the host costs copies
// that wait for the stream).  One step per 64 sequences; false when there is
// no such tile.
template <int BM>
DEVINLINE bool ft_find_tile(const int32_t* cu, int B, int t, int* seq,
                            int* off) {
  const int lane = threadIdx.x & 63;
  int before = 0;
  for (int base = 0; base < B; base += 64) {
    const int i = base + lane;
    const int n = i < B ? (cu[i + 1] - cu[i] + BM - 1) / BM : 0;
    int sum = n;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int up = __shfl_up(sum, d, 64);
      if (lane >= d) sum += up;
    }
    const uint64_t past = __ballot(before + sum > t);
    if (past) {
      const int w = __builtin_ctzll(past);
      *seq = __builtin_amdgcn_readfirstlane(base + w);
      *off = __builtin_amdgcn_readfirstlane(
          (t - before - __shfl(sum - n, w, 64)) * BM);
      return true;
    }
    before += __builtin_amdgcn_readfirstlane(__shfl(sum, 63, 64));
  }
  return false;
}

// The key tiles of a workgroup, in order: [kept_from, kept), then [first, end).
struct FlashSpan {
  int kv_len;            // keys of the sequence
  int kept, first, end;  // kept and first are multiples of FT_BN
  int kept_from = 0;
  DEVINLINE int begin() const { return kept > kept_from ? kept_from : first; }
  DEVINLINE int next(int kb) const {
    kb += FT_BN;
    return kb >= kept && kb < first ? first : kb;
  }
};

// Scores of this lane's query row.
struct FlashScore {
  int pos;         // its position; it sees keys lo .. pos and < keep
  int lo, keep;
  int wave_pos;    // position of the wave's first row
  int wave_lo[2];  // lo of the wave's first and last row
  float c;         // raw score -> log2 of the weight, > 0 when PLAIN
  float cap;       // > 0: c * s goes through cap tanh(. / cap), in log2
  float slope;     // per key of distance, in log2
};

// 16 bytes of zeros: what a key chunk past the row's width is read from.  The
// query is zero there, but 0 * infinity of some other chunk would not be.
static __device__ const uint16_t ft_zeros[8] = {0, 0, 0, 0, 0, 0, 0, 0};

// K and V rows of one sequence.  begin(kbase, wave) is called before the
// addresses of a tile are asked for, with the wave (which moves the tile's
// rows 16 wave .. + 15); rows past the last key repeat it (they are masked).
// prefetch(kbase, wave) is called one tile ahead.  STRAIGHT sources also have
// tiles (straight(kbase)) whose chunks lie at a scalar base per tile and wave
// and at lane offsets, in bytes, that are the same for all of them.

// In pages of any size; with a multiple of 16 a wave's rows lie in one page,
// whose number was asked for one tile ahead, and the address is a scalar base
// and a small lane offset (700 decoded tokens of 200 keys on pages of 32, 16
// heads of 64 on 2: 51.2 us where every row looks its page up, 33.9 so).
// kp<PAD>: the rows are narrower than the tile.
struct PagedRows {
  const uint16_t *k, *v;   // [pages, heads, size, width]
  const int32_t* table;    // the sequence's pages
  int head, heads, size, kw, vw, kv_len;
  int page = 0, last = 0, tile = 0;
  int64_t base = 0;
  // the first of the wave's 16 rows, or of the sequence's last 16
  DEVINLINE int first_row(int kbase, int wave) const {
    return min((kbase >> 4) + wave, (kv_len - 1) >> 4) << 4;
  }
  DEVINLINE void prefetch(int kbase, int wave) {
    if (size % 16 != 0) return;
    const int row = first_row(kbase, wave);
    page = table[size == 16 ? row >> 4 : row / size];
  }
  DEVINLINE void begin(int kbase, int wave) {
    tile = kbase;
    if (size % 16 != 0) return;
    const int row = first_row(kbase, wave);
    last = kv_len - 1 - row;
    base = ((int64_t)__builtin_amdgcn_readfirstlane(page) * heads + head) *
               size + (size == 16 ? 0 : row % size);
  }
  DEVINLINE const uint16_t* at(const uint16_t* p, int w, int r, int c) const {
    // a chunk past the width repeats the first one
    const int d = c * 8 < w ? c * 8 : 0;
    if (size % 16 == 0)
      return p + base * w + (uint32_t)(min(r & 15, last) * w + d);
    const int pos = min(tile + r, kv_len - 1);
    return p + (((int64_t)table[pos / size] * heads + head) * size +
                pos % size) * w + d;
  }
  DEVINLINE int key_width() const { return kw; }
  template <bool PAD>
  DEVINLINE const uint16_t* kp(int r, int c) const {
    return !PAD || c * 8 < kw ? at(k, kw, r, c) : ft_zeros;
  }
  // values past the width are not stored
  DEVINLINE const uint16_t* vp(int r, int c) const { return at(v, vw, r, c); }
  static constexpr bool STRAIGHT = true;
  DEVINLINE bool straight(int kbase) const {
    return size % 16 == 0 && kbase + FT_BN <= kv_len;
  }
  DEVINLINE const uint16_t* k_base() const { return k + base * kw; }
  DEVINLINE const uint16_t* v_base() const { return v + base * vw; }
  DEVINLINE int k_off(int r, int c) const { return (r & 15) * kw * 2 + c * 16; }
  DEVINLINE int v_off(int r, int c) const {
    return (r & 15) * vw * 2 + (c * 8 < vw ? c * 16 : 0);
  }
};

// Dense: k and v point to the sequence's first row, this head.  A tile's rows
// are 32-bit offsets from its first.
struct DenseRows {
  const uint16_t *k, *v;
  int k_rs, v_rs;
  int kv_len;
  const uint16_t *kt = nullptr, *vt = nullptr;
  int last = 0;
  DEVINLINE void prefetch(int, int) {}
  DEVINLINE void begin(int kbase, int) {
    kt = k + (int64_t)kbase * k_rs;
    vt = v + (int64_t)kbase * v_rs;
    last = kv_len - 1 - kbase;
  }
  DEVINLINE int key_width() const { return INT_MAX; }
  template <bool>
  DEVINLINE const uint16_t* kp(int r, int c) const {
    return kt + (uint32_t)(min(r, last) * k_rs + c * 8);
  }
  DEVINLINE const uint16_t* vp(int r, int c) const {
    return vt + (uint32_t)(min(r, last) * v_rs + c * 8);
  }
  static constexpr bool STRAIGHT = true;
  DEVINLINE bool straight(int kbase) const { return kbase + FT_BN <= kv_len; }
  DEVINLINE const uint16_t* k_base() const { return kt; }
  DEVINLINE const uint16_t* v_base() const { return vt; }
  DEVINLINE int k_off(int r, int c) const { return r * k_rs * 2 + c * 16; }
  DEVINLINE int v_off(int r, int c) const { return r * v_rs * 2 + c * 16; }
};

// Swizzle of V's 16-byte chunks in row r.
template <int NV>
DEVINLINE int ft_vswz(int r) {
  return NV >= 128 ? (r & 3) << 2 : ((r >> 1) & 1) << 2;
}

// Swizzle of the 16-byte chunks of K row r, rows of NK entries: 256 bytes apart
// in the banks' 256 (or a multiple), or 128 (latent_decode's transposing reads
// of four neighbouring rows want bit 2 to tell rows 0 and 2 apart).  By r & 7
// two rows met in a bank at every fragment.
template <int NK>
DEVINLINE int ft_kswz(int r) {
  static_assert(NK % 64 == 0);
  return NK % 128 == 0 ? r & 15 : (r & 2) << 1 | (r >> 2 & 3);
}

// Walks the tiles.  qf: the query row as B operand (dims 16 s + 8 half);
// k0 .. v1: LDS of FT_BN rows of NK (NV) bf16.  Out: o[dt][i] is dim 32 dt +
// 8 (i / 4) + 4 half + i % 4 of the lane's row, unnormalised; l the row's sum
// and m its reference, in log2 (both lane halves alike).
// PLAIN: causal only, the maximum is of raw scores.
// VD < NV: the four waves have the SAME 32 query rows and each the VD value
// dims from dim0 on (decoded rows: the heads that share keys).
// ONCE: decoded rows, whose keys nobody reads again soon: loads are nontemporal and
// leave nothing in the memory side's cache.
template <int NK, int NV, bool PLAIN, class Rows, int VD = NV,
          bool ONCE = false>
DEVINLINE void flash_tiles(Rows& rows, const FlashSpan& span,
                           const FlashScore& sc,
                           const ft_bf16x8 (&qf)[NK / 16], uint8_t* k0,
                           uint8_t* k1, uint8_t* v0, uint8_t* v1,
                           ft_f32x16 (&o)[VD / 32], float& m, float& l,
                           int dim0 = 0) {
  constexpr int BN = FT_BN, CK = NK / 8, CV = NV / 8;
  constexpr int VROW = NV * 2;        // bytes of a V row
  constexpr int RW = BN / FT_WAVES;   // rows that a wave moves
  constexpr int AUX = ONCE ? 2 : 0;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int half = lane >> 5, col = lane & 31;

  // rows and chunks of this lane's pieces
  auto k_row = [&](int i) { return wave * RW + (i * 64 + lane) / CK; };
  auto k_chunk = [&](int i) {
    return ((i * 64 + lane) % CK) ^ ft_kswz<NK>(k_row(i));
  };
  auto v_row = [&](int i) { return wave * RW + (i * 64 + lane) / CV; };
  auto v_chunk = [&](int i) {
    return ((i * 64 + lane) % CV) ^ ft_vswz<NV>(v_row(i));
  };
  // Addresses of whole tiles cost the vector units nothing: they are a scalar
  // base and these offsets (64-bit sums per lane were a third of the vector
  // instructions of a tile).
  constexpr bool STRAIGHT = Rows::STRAIGHT;
  int ko[CK / 4], vo[CV / 4];
  if constexpr (STRAIGHT) {
#pragma unroll
    for (int i = 0; i < CK / 4; ++i) ko[i] = rows.k_off(k_row(i), k_chunk(i));
#pragma unroll
    for (int i = 0; i < CV / 4; ++i) vo[i] = rows.v_off(v_row(i), v_chunk(i));
  }
  auto stage = [&](int kbase, uint8_t* kd, uint8_t* vd) FT_INLINE {
    rows.begin(kbase, wave);
    bool straight = false;
    if constexpr (STRAIGHT) {
      straight = rows.straight(kbase) && rows.key_width() >= NK;
      if (straight) {
        typedef __attribute__((address_space(3))) void lds_void;
        const auto kr = __builtin_amdgcn_make_buffer_rsrc(
            (void*)rows.k_base(), 0, -1, 0x00020000);
        const auto vr = __builtin_amdgcn_make_buffer_rsrc(
            (void*)rows.v_base(), 0, -1, 0x00020000);
#pragma unroll
        for (int i = 0; i < CK / 4; ++i)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(
              kr, (lds_void*)(kd + (wave * (CK / 4) + i) * 1024), 16, ko[i], 0,
              0, AUX);
#pragma unroll
        for (int i = 0; i < CV / 4; ++i)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(
              vr, (lds_void*)(vd + (wave * (CV / 4) + i) * 1024), 16, vo[i], 0,
              0, AUX);
      }
    }
    if (!straight) {
      auto keys = [&](auto pad) {
#pragma unroll
        for (int i = 0; i < CK / 4; ++i)
          __builtin_amdgcn_global_load_lds(
              reinterpret_cast<const uint32_t*>(
                  rows.template kp<decltype(pad)::value>(k_row(i), k_chunk(i))),
              reinterpret_cast<uint32_t*>(kd + (wave * (CK / 4) + i) * 1024),
              16, 0, AUX);
      };
      // where nothing is padded the address stays a scalar base and an offset
      if (rows.key_width() < NK) keys(std::true_type{});
      else keys(std::false_type{});
#pragma unroll
      for (int i = 0; i < CV / 4; ++i)
        __builtin_amdgcn_global_load_lds(
            reinterpret_cast<const uint32_t*>(rows.vp(v_row(i), v_chunk(i))),
            reinterpret_cast<uint32_t*>(vd + (wave * (CV / 4) + i) * 1024), 16,
            0, AUX);
    }
    rows.prefetch(span.next(kbase), wave);
  };

  // LDS offsets of this lane's fragments
  int koff[NK / 16];  // K row `col` (+ 32 per sub-tile), dims 16 s + 8 half
#pragma unroll
  for (int s = 0; s < NK / 16; ++s)
    koff[s] = col * (NK * 2) + (((2 * s + half) ^ ft_kswz<NK>(col)) << 4);
  int voff[VD / 32][2];  // V^T: dims 32 dt + 16 (lane bit 4), keys 4 half + 8 e
#pragma unroll
  for (int dt = 0; dt < VD / 32; ++dt)
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int i = lane & 15, r = 4 * half + 8 * e + (i >> 2);
      const int c =
          dim0 / 8 + 4 * dt + 2 * ((lane >> 4) & 1) + ((i & 3) >> 1);
      voff[dt][e] = r * VROW +
                    ((c ^ ft_vswz<NV>(r)) << 4) +
                    8 * (i & 1);
    }

  m = -INFINITY;
  l = 0.0f;  // this lane half's keys, until the end
#pragma unroll
  for (int dt = 0; dt < VD / 32; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[dt][i] = 0.0f;
  // tanh by exp2: cap - 2 cap / (1 + 2^(cap_k s))
  const float cap_k = sc.cap > 0.0f ? 2.0f * FT_LOG2E * sc.c / sc.cap : 0.0f;

  auto step = [&](int kbase, int knext, uint8_t* kb, uint8_t* vb, uint8_t* kn,
                  uint8_t* vn) {
    // this wave's loads of the tile have arrived; behind the barrier all
    // have, and nobody reads the other buffer any more
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (knext < span.end) stage(knext, kn, vn);
    if (kbase > sc.wave_pos + 31) return;
    if (!PLAIN && kbase + BN <= sc.wave_lo[0] && kbase >= sc.keep) return;

    ft_f32x16 s[2];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) s[t][i] = 0.0f;
    // K fragments are read KD products ahead (left to itself the compiler reads
    // a pair, waits for it and uses it)
    constexpr int KD = NK / 16 < 4 ? NK / 16 : 4;
    ft_bf16x8 kf[KD][2];
    auto read_k = [&](int d) FT_INLINE {
#pragma unroll
      for (int t = 0; t < 2; ++t)
        kf[d % KD][t] = *reinterpret_cast<const ft_bf16x8*>(
            kb + koff[d] + t * 32 * NK * 2);
    };
#pragma unroll
    for (int d = 0; d < KD; ++d) read_k(d);
#pragma unroll
    for (int d = 0; d < NK / 16; ++d) {
#pragma unroll
      for (int t = 0; t < 2; ++t)
        s[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[d % KD][t], qf[d],
                                                       s[t], 0, 0, 0);
      if (d + KD < NK / 16) read_k(d + KD);
    }
    __builtin_amdgcn_sched_group_barrier(FT_DS_READ, 2 * KD, 0);
#pragma unroll
    for (int d = 0; d < NK / 16; ++d) {
      __builtin_amdgcn_sched_group_barrier(FT_MFMA, 2, 0);
      if (d + KD < NK / 16) __builtin_amdgcn_sched_group_barrier(FT_DS_READ, 2, 0);
    }
    __builtin_amdgcn_sched_barrier(0);

    if (!PLAIN) {
      if (sc.cap > 0.0f) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int i = 0; i < 16; ++i)
            s[t][i] = fmaf(-2.0f * sc.cap,
                           __builtin_amdgcn_rcpf(
                               1.0f + __builtin_amdgcn_exp2f(s[t][i] * cap_k)),
                           sc.cap);
      } else {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int i = 0; i < 16; ++i) s[t][i] *= sc.c;
      }
      if (sc.slope != 0.0f) {
        const float base = (float)(kbase + 4 * half - sc.pos) * sc.slope;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int i = 0; i < 16; ++i)
            s[t][i] += fmaf(sc.slope, (float)(32 * t + (i & 3) + 8 * (i >> 2)),
                            base);
      }
    }
    bool partly = kbase + BN - 1 > sc.wave_pos;
    if (!PLAIN) partly |= kbase < sc.wave_lo[1] && kbase + BN > sc.keep;
    if (partly) {
      const int seen = min(sc.pos, span.kv_len - 1) - kbase - 4 * half;
      const int lo = sc.lo - kbase - 4 * half;
      const int keep = sc.keep - kbase - 4 * half;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int key = 32 * t + (i & 3) + 8 * (i >> 2);
          bool hide = key > seen;
          if (!PLAIN) hide |= key < lo && key >= keep;
          if (hide) s[t][i] = -INFINITY;
        }
    }

    float mx = s[0][0];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[t][i]);
    {
      float lo, hi;
      ft_both_halves(mx, lo, hi);
      mx = fmaxf(lo, hi);
    }
    const float c = PLAIN ? sc.c : 1.0f;
    if (__any(mx > m)) {
      const float mn = fmaxf(m, mx);
      const float alpha =
          m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f((m - mn) * c);
      m = mn;
      l *= alpha;
#pragma unroll
      for (int dt = 0; dt < VD / 32; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[dt][i] *= alpha;
    }
    const float mc = m == -INFINITY ? 0.0f : m * c;
    // Weights of 32 keys, and their products with V 16 keys at a time: those of
    // the second 32 are computed between the products of the first, and V
    // fragments are read one step of products ahead.
    uint32_t p[2][8];
    auto weigh = [&](int t) FT_INLINE {
      float sum = 0.0f;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        s[t][i] = __builtin_amdgcn_exp2f(PLAIN ? fmaf(s[t][i], c, -mc)
                                               : s[t][i] - mc);
        sum += s[t][i];
      }
#pragma unroll
      for (int i = 0; i < 8; ++i)
        p[t][i] = ft_pack_bf16(s[t][2 * i], s[t][2 * i + 1]);
      return sum;
    };
    union {
      ft_short4 h[2];
      ft_bf16x8 v;
    } vf[2][VD / 32];
    auto read_v = [&](int j) FT_INLINE {
      typedef __attribute__((address_space(3))) ft_short4 lds_short4;
#pragma unroll
      for (int dt = 0; dt < VD / 32; ++dt)
#pragma unroll
        for (int e = 0; e < 2; ++e)
          vf[j & 1][dt].h[e] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (lds_short4*)(vb + voff[dt][e] + 16 * j * VROW));
    };
    __builtin_amdgcn_sched_barrier(0);
    read_v(0);
    const float sum0 = weigh(0);
    __builtin_amdgcn_sched_barrier(0);
    float sum1 = 0.0f;
    __builtin_amdgcn_s_setprio(1);   // before the other wave's softmax
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (j < 3) read_v(j + 1);
      if (j == 0) sum1 = weigh(1);
      union {
        uint32_t u[4];
        ft_bf16x8 v;
      } pf;
#pragma unroll
      for (int e = 0; e < 4; ++e) pf.u[e] = p[j >> 1][(j & 1) * 4 + e];
#pragma unroll
      for (int dt = 0; dt < VD / 32; ++dt)
        o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[j & 1][dt].v, pf.v,
                                                        o[dt], 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < VD / 8; ++i) {
      __builtin_amdgcn_sched_group_barrier(FT_MFMA, 1, 0);
      if (i < 3 * (VD / 32))
        __builtin_amdgcn_sched_group_barrier(FT_DS_READ, 2, 0);
      if (i < 2 * (VD / 32))
        __builtin_amdgcn_sched_group_barrier(FT_VALU, 224 / VD * 4, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(0);
    l += sum0 + sum1;
  };

  int kb = span.begin();
  if (kb < span.end) {
    rows.prefetch(kb, wave);
    stage(kb, k0, v0);
    while (true) {
      int kn = span.next(kb);
      step(kb, kn, k0, v0, k1, v1);
      if (kn >= span.end) break;
      kb = kn;
      kn = span.next(kb);
      step(kb, kn, k1, v1, k0, v0);
      if (kn >= span.end) break;
      kb = kn;
    }
  }
  float lo, hi;
  ft_both_halves(l, lo, hi);
  l = lo + hi;
  if (PLAIN) m *= sc.c;
}

// Decoded rows: a sequence's key tiles are cut for `nsplit` workgroups, the
// part's unnormalised fp32 sums are merged by flash_merge_kernel.  Part `split`
// of the tiles of a span (whose kept tiles come first).
DEVINLINE FlashSpan flash_part(FlashSpan s, int split, int nsplit) {
  if (nsplit == 1) return s;
  const int kept = s.kept / FT_BN;
  const int n = kept + (s.end - s.first + FT_BN - 1) / FT_BN;
  const int per = (n + nsplit - 1) / nsplit;
  const int a = min(split * per, n), b = min(a + per, n);
  FlashSpan p = s;
  // tile t of the walk starts at key 64 t, or behind the kept ones at first
  p.first = a > kept ? s.first + (a - kept) * FT_BN : s.first;
  p.end = b > kept ? min(s.end, s.first + (b - kept) * FT_BN) : s.first;
  p.kept = 0;
  if (a < kept) {          // [64 a, min(kept, 64 b)), then the rest
    p.kept_from = a * FT_BN;
    p.kept = min(b, kept) * FT_BN;
    if (b <= kept) p.end = p.first = p.kept;   // nothing behind them
  } else if (a == b) {
    p.end = p.first;
  }
  return p;
}

// Stores the lane's dims d of an output row times f(d), 4 dims at a time; P
// is the row's real width.
template <int NV, class F>
DEVINLINE void flash_store(uint16_t* row, const ft_f32x16 (&o)[NV / 32], int P,
                           int half, F f) {
#pragma unroll
  for (int dt = 0; dt < NV / 32; ++dt)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int d = 32 * dt + 8 * g + 4 * half;
      if (d < P) {
        uint2 w;
        w.x = ft_pack_bf16(o[dt][4 * g] * f(d), o[dt][4 * g + 1] * f(d + 1));
        w.y = ft_pack_bf16(o[dt][4 * g + 2] * f(d + 2),
                           o[dt][4 * g + 3] * f(d + 3));
        *reinterpret_cast<uint2*>(row + d) = w;
      }
    }
}

// The unnormalised sums of decoded rows, one slot per (row, head, part).
struct FlashParts {
  float* o;    // [rows, heads, nsplit, width]
  float* ml;   // [rows, heads, nsplit, 2]: reference (log2) and sum
  int nsplit;
};

// Dims dim0 .. of the lane's row to a part's slot.
template <int VD>
DEVINLINE void flash_store_part(const FlashParts& p, int64_t pair, int split,
                                int width, const ft_f32x16 (&o)[VD / 32],
                                int dim0, float m, float l, int half) {
  const int64_t slot = pair * p.nsplit + split;
#pragma unroll
  for (int dt = 0; dt < VD / 32; ++dt)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int d = dim0 + 32 * dt + 8 * g + 4 * half;
      if (d < width)
        *reinterpret_cast<float4*>(p.o + slot * width + d) =
            make_float4(o[dt][4 * g], o[dt][4 * g + 1], o[dt][4 * g + 2],
                        o[dt][4 * g + 3]);
    }
  if (dim0 == 0 && half == 0) {
    p.ml[2 * slot] = m;
    p.ml[2 * slot + 1] = l;
  }
}

// What closes a decoded row: sink and gate per head (fp32) or a sigmoid gate
// from bf16 logits, per head or per value.
struct FlashClose {
  uint16_t* out;           // [tokens, heads, width]
  int heads, width;
  const float* sinks;      // [heads]
  const float* gate;       // [tokens, heads]
  const uint16_t* logits;  // [tokens, heads * logit_w], row stride logits_rs
  int64_t logits_rs;
  int logit_w;
  DEVINLINE float sum(int head, float m, float l) const {
    return sinks ? l + __builtin_amdgcn_exp2f(fmaf(sinks[head], FT_LOG2E, -m))
                 : l;
  }
  DEVINLINE float factor(int64_t tok, int head, int d) const {
    float f = gate ? gate[tok * heads + head] : 1.0f;
    if (logits) {
      const float x = bf16_to_f32(logits[tok * logits_rs + head * logit_w +
                                         (logit_w > 1 ? d : 0)]);
      f *= __frcp_rn(1.0f + __expf(-x));
    }
    return f;
  }
};

// One workgroup of width / 4 threads per (row, head); row r is token tokens[r],
// or r without a list.
static __global__ void flash_merge_kernel(FlashClose c, FlashParts p,
                                          const int32_t* tokens) {
  const int64_t pair = blockIdx.x;
  const int head = pair % c.heads;
  const int64_t row = pair / c.heads;
  const int64_t tok = tokens ? tokens[row] : row;
  const int d = threadIdx.x * 4;
  const float2* ml =
      reinterpret_cast<const float2*>(p.ml) + pair * p.nsplit;
  float m = -INFINITY;
  for (int s = 0; s < p.nsplit; ++s) m = fmaxf(m, ml[s].x);
  float l = 0.0f;
  float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll 4
  for (int s = 0; s < p.nsplit; ++s) {
    const float2 v = ml[s];
    const float4 a = *reinterpret_cast<const float4*>(
        p.o + (pair * p.nsplit + s) * c.width + d);
    const float f = v.x == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(v.x - m);
    l = fmaf(f, v.y, l);
    o.x = fmaf(f, a.x, o.x);
    o.y = fmaf(f, a.y, o.y);
    o.z = fmaf(f, a.z, o.z);
    o.w = fmaf(f, a.w, o.w);
  }
  const float inv = 1.0f / c.sum(head, m, l);
  uint2 w;
  w.x = ft_pack_bf16(o.x * inv * c.factor(tok, head, d),
                     o.y * inv * c.factor(tok, head, d + 1));
  w.y = ft_pack_bf16(o.z * inv * c.factor(tok, head, d + 2),
                     o.w * inv * c.factor(tok, head, d + 3));
  *reinterpret_cast<uint2*>(c.out + (tok * c.heads + head) * c.width + d) = w;
}

}  // namespace igw
