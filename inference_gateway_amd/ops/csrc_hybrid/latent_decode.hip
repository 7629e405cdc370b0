// Absorbed latent attention of decoded tokens (gfx950, bf16).
//
// All heads of a token read the same cached rows (latent | rotated key), so 32
// heads are the query columns of one workgroup and a row of the cache is its
// own key AND value: tiles of 64 rows go to LDS once, by DMA and double
// buffered, K fragments and transposed V fragments are read from the same
// image.  Of a tile each of the four waves scores the 16 rows that it moved
// (S^T = K Q^T, mfma 16x16x32; one lane swap leaves a lane with 8 keys of one
// head), the waves exchange their maxima and then their weights through LDS
// (fp32, and bf16 as the next product's operand), and each adds all 64 rows to its
// quarter of the value dims (O^T = V^T P^T, mfma 32x32x16).  So scores and weights
// are computed once, about 1200 cycles of matrix instructions and as many of LDS
// reads a tile of 73 KB; where every wave scored all 64 rows for itself, without
// an exchange, they were 2800, and the loads behind them waited.
//
// Bound by HBM where every compute unit has a long part (256 tokens of 2048 keys
// 5.5 TB/s), else by the latency of a tile's loads, one tile ahead, and by start and
// end of a part: about 8 us, with its sums, 64 KB, written and read again by the
// merge.  Nothing of the start waits that need not: the first tile is sent for
// before the queries, and the code is short (rows of pages that are no multiple of
// 16, or narrower than the tile, are moved by a loop), since a launch fetches it
// anew.  One workgroup per compute unit (152 KB of LDS).
//
// Measured, all waves scoring all rows, contexts in equal numbers of parts, and
// this (us): 32 heads, rank 512 + 64, 48 tokens of 700 to 3500 keys 58.8 and 42.4,
// of 2000 47.0 and 40.8, 256 of 2048 150 and 110 (5.5 TB/s), 512 of 300 65.7 and
// 54.5, one of 3000 29.3 and 22.2, 64 of 10 12.2 and 11.0; 128 heads, 256 of 2048
// 569 and 416; rank 256, 16 heads, 48 of 700 to 3500 34.9 and 26.8, 256 of 2048
// 96.4 and 65.4.
#include "../csrc/flash_tile.h"
#include "act_types.h"

namespace igw {

// Contexts cut for `slots` workgroups; 0: a workgroup takes a token whole.
struct LatentParts {
  float* o;     // [slots, heads, R]: unnormalised sums
  float2* ml;   // [slots, heads]: reference (log2) and sum
  int2* rows;   // [tokens]: first slot and number of parts, if `each` is 0
  int slots, tokens;
  int each;     // parts of every token, 0: by its length
  int shortest; // then: tiles of a part at least, but for a context's last
};

struct LatentDecodeArgs {
  const uint16_t *qa, *qr;   // [T, H, R], [T, H, RD]
  int64_t qa_s0, qa_s1, qr_s0, qr_s1;
  const uint16_t* cache;     // [pages, size, R + RD]
  const int32_t *block_table, *row_seq, *positions;
  int max_blocks, RD, size, window;
  float scale;
  FlashClose close;
  LatentParts parts;
};

// From this many bytes of rows on (as if every context were the longest) they are
// read with nontemporal loads: the memory side's cache, of this size, holds them
// neither for the next step nor beside other layers' (us, eight caches in turn, plain
// and nontemporal: 256 tokens of 2048, rank 512, 32 / 64 / 128 heads 147.4 291 573 and
// 146.2 286 567, rank 256, 16 / 64 heads 89.5 172.6 and 85.8 168.0).  Smaller ones are
// as fast with plain loads or faster, above all where groups of heads read the rows
// again (16 of 2000, rank 512, 32 / 64 / 128 heads 28.7 32.3 45.5 and 30.2 36.0 49.5;
// 48 of 2000 46.2 71.0 121.8 and 47.6 73.3 123.2; of 700 to 3500 59.1 102.8 and 59.0
// 103.6; 512 of 300 64.8 120.1 and 64.3 123.5, but rank 256, 16 heads, 36.6 and 35.2).
constexpr int64_t LD_ONCE = 256 << 20;

constexpr int LD_SETS = 2;     // 64 tokens each, whose lengths are looked at
constexpr int LD_PARTS = 32;   // of a context at most

DEVINLINE int ld_first(int pos, int window) {   // key
  return window > 0 ? max(0, pos - window + 1) : 0;
}

// Running sums and maxima (of numbers >= 0) over the wave's lanes.
template <bool MAX = false>
DEVINLINE int ld_scan(int x) {
  auto add = [&](auto ctrl, auto rows) {
    const int y = __builtin_amdgcn_update_dpp(
        0, x, decltype(ctrl)::value, decltype(rows)::value, 0xf, false);
    x = MAX ? max(x, y) : x + y;
  };
  std::integral_constant<int, 0xf> all;
  add(std::integral_constant<int, 0x111>{}, all);   // from 1, 2, 4, 8 lanes
  add(std::integral_constant<int, 0x112>{}, all);   // below, in its 16
  add(std::integral_constant<int, 0x114>{}, all);
  add(std::integral_constant<int, 0x118>{}, all);
  // the last of the 16 below, of the lower half
  add(std::integral_constant<int, 0x142>{}, std::integral_constant<int, 0xa>{});
  add(std::integral_constant<int, 0x143>{}, std::integral_constant<int, 0xc>{});
  return x;
}
template <bool MAX = false>
DEVINLINE int ld_all(int x) {
  return __builtin_amdgcn_readlane(ld_scan<MAX>(x), 63);
}

// Token, part and number of parts of slot b: all contexts are cut into parts of
// `per` tiles, about the least with which the parts of all of them are no more than
// the slots.  Every wave finds it for itself.  False: no part for this slot.
DEVINLINE bool ld_share(const LatentDecodeArgs& a, int b, int* token, int* part,
                        int* of) {
  const int lane = threadIdx.x & 63, T = a.parts.tokens;
  int pos[LD_SETS];
  float n[LD_SETS];
#pragma unroll
  for (int j = 0; j < LD_SETS; ++j)
    pos[j] = a.positions[min(j * 64 + lane, T - 1)];
  int most = 1, sum = 0;
#pragma unroll
  for (int j = 0; j < LD_SETS; ++j) {
    const int tiles =
        j * 64 + lane < T
            ? pos[j] / FT_BN - ld_first(pos[j], a.window) / FT_BN + 1
            : 0;
    most = max(most, tiles);
    sum += tiles;
    n[j] = (float)tiles;
  }
  // ceil(n / per), in floats, which is exact below 2^20 tiles
  auto parts = [&](int j, int per) {
    return (int)((n[j] + (float)per - 0.5f) * __builtin_amdgcn_rcpf((float)per));
  };
  auto fits = [&](int per) {
    int c = 0;
#pragma unroll
    for (int j = 0; j < LD_SETS; ++j) c += parts(j, per);
    return ld_all(c) <= a.parts.slots;
  };
  int per = max(max((ld_all(sum) + a.parts.slots - 1) / a.parts.slots,
                    a.parts.shortest),
                (ld_all<true>(most) + LD_PARTS - 1) / LD_PARTS);
  // ends: with the longest context's tiles there are no more parts than tokens
  while (!fits(per)) per += 1 + per / 8;
  int before = 0;
#pragma unroll
  for (int j = 0; j < LD_SETS; ++j) {
    const int c = parts(j, per), to = ld_scan(c);
    const uint64_t past = __ballot(before + to > b);
    if (past) {
      const int w = __builtin_ctzll(past);
      *token = j * 64 + w;
      *of = __builtin_amdgcn_readlane(c, w);
      *part = b - before - (__builtin_amdgcn_readlane(to, w) - *of);
      return true;
    }
    before += __builtin_amdgcn_readlane(to, 63);
  }
  return false;
}

// All waves' LDS accesses are done; tiles on their way from memory are not waited for.
DEVINLINE void ld_lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

template <int NK, int R, bool ONCE>
DEVINLINE void latent_decode_body(const LatentDecodeArgs& a) {
  typedef __attribute__((ext_vector_type(4))) float f32x4;
  constexpr int VD = R / FT_WAVES, ROWB = NK * 2, CK = NK / 8;
  constexpr int LOADS = CK / FT_WAVES, KS = NK / 32, AUX = ONCE ? 2 : 0;
  __shared__ __attribute__((aligned(1024))) uint8_t k_s0[FT_BN * ROWB];
  __shared__ __attribute__((aligned(1024))) uint8_t k_s1[FT_BN * ROWB];
  __shared__ __attribute__((aligned(16))) uint16_t p_s[FT_WAVES][64][8];
  __shared__ __attribute__((aligned(16))) float x_s[32][FT_WAVES];
  const int lane = threadIdx.x & 63, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int token = blockIdx.x, part = 0, of = 1;
  if (a.parts.each > 0) {
    of = a.parts.each;
    token = blockIdx.x / of;
    part = blockIdx.x - token * of;
  } else if (a.parts.slots > 0) {
    if (!ld_share(a, blockIdx.x, &token, &part, &of)) return;
    if (part == 0 && blockIdx.y == 0 && threadIdx.x == 0)
      a.parts.rows[token] = make_int2(blockIdx.x, of);
  }
  const int64_t t = token;
  const int H = a.close.heads;
  const int head = blockIdx.y * 32 + (lane & 31);
  const int pos = a.positions[t];

  const int lo = ld_first(pos, a.window);
  const float c = a.scale * FT_LOG2E;
  const FlashSpan span =
      flash_part(FlashSpan{pos + 1, 0, lo / FT_BN * FT_BN, pos + 1},
                 part, of);
  PagedRows rows{a.cache, nullptr,
                 a.block_table + (int64_t)a.row_seq[t] * a.max_blocks, 0, 1,
                 a.size, R + a.RD, 0, pos + 1};

  // a wave moves the 16 rows that it scores
  auto k_row = [&](int i) { return wave * 16 + (i * 64 + lane) / CK; };
  auto k_chunk = [&](int i) {
    return ((i * 64 + lane) % CK) ^ ft_kswz<NK>(k_row(i));
  };
  int ko[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) ko[i] = rows.k_off(k_row(i), k_chunk(i));
  auto stage = [&](int kbase, uint8_t* kd) FT_INLINE {
    rows.begin(kbase, wave);
    if (a.size % 16 == 0 && rows.key_width() >= NK) {
      typedef __attribute__((address_space(3))) void lds_void;
      const auto kr = __builtin_amdgcn_make_buffer_rsrc((void*)rows.k_base(), 0,
                                                        -1, 0x00020000);
      if (rows.last >= 15) {
#pragma unroll
        for (int i = 0; i < LOADS; ++i)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(
              kr, (lds_void*)(kd + (wave * LOADS + i) * 1024), 16, ko[i], 0, 0,
              AUX);
      } else {   // rows past the last repeat it
#pragma unroll
        for (int i = 0; i < LOADS; ++i)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(
              kr, (lds_void*)(kd + (wave * LOADS + i) * 1024), 16,
              ko[i] - max((i * 64 + lane) / CK - rows.last, 0) * ROWB, 0, 0,
              AUX);
      }
    } else {
#pragma unroll 1   // rare, and the code of a launch is fetched anew
      for (int i = 0; i < LOADS; ++i)
        __builtin_amdgcn_global_load_lds(
            reinterpret_cast<const uint32_t*>(
                rows.template kp<true>(k_row(i), k_chunk(i))),
            reinterpret_cast<uint32_t*>(kd + (wave * LOADS + i) * 1024), 16, 0,
            AUX);
    }
    rows.prefetch(span.next(kbase), wave);
  };

  // LDS offsets of fragments.  Scores: row lane % 16 of the wave's, chunk
  // 4 s + lane / 16; the swizzle stays within eight chunks.
  int koff[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int r = lane & 15;
    koff[u] = (wave * 16 + r) * ROWB +
              (((4 * u + (lane >> 4)) ^ ft_kswz<NK>(r)) << 4);
  }
  // Values, transposed: entries 32 dt + 16 (lane bit 4) .. of this wave's, keys
  // 8 half + 4 e .. + 3
  int voff[2][2];
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int i = lane & 15, r = 8 * half + 4 * e + (i >> 2);
      const int ch = 4 * u + 2 * ((lane >> 4) & 1) + ((i & 3) >> 1);
      voff[u][e] = wave * VD * 2 + r * ROWB + ((ch ^ ft_kswz<NK>(r)) << 4) +
                   8 * (i & 1);
    }

  // the first tile is on its way before the queries
  int kb = span.begin();
  if (kb < span.end) {
    rows.prefetch(kb, wave);
    stage(kb, k_s0);
  }
  // Queries as B operand of 16 x 16 x 32: heads 16 u + lane % 16, entries
  // 32 s + 8 (lane / 16) .. + 7.  No branches: what is not there is another
  // head's, which is not stored, or zeros.
  ft_bf16x8 qf[2][KS];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int64_t h = min((int)blockIdx.y * 32 + 16 * u + (lane & 15), H - 1);
    const uint16_t* qa = a.qa + t * a.qa_s0 + h * a.qa_s1 + 8 * (lane >> 4);
    const uint16_t* qr = a.qr + t * a.qr_s0 + h * a.qr_s1;
#pragma unroll
    for (int s = 0; s < R / 32; ++s)
      qf[u][s] = *reinterpret_cast<const ft_bf16x8*>(qa + 32 * s);
#pragma unroll
    for (int s = R / 32; s < KS; ++s) {
      const int d = 32 * s - R + 8 * (lane >> 4);
      qf[u][s] = *reinterpret_cast<const ft_bf16x8*>(
          d < a.RD ? qr + d : ft_zeros);
    }
  }
  ft_f32x16 o[VD / 32];
  float m = -INFINITY, l = 0.0f;   // l: of the wave's and lane half's keys
#pragma unroll
  for (int dt = 0; dt < VD / 32; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[dt][i] = 0.0f;

  auto step = [&](int kbase, int knext, uint8_t* kb, uint8_t* kn) {
    // this wave's loads of the tile have arrived; behind the barrier all
    // have, and nobody reads the other buffer any more
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (knext < span.end) stage(knext, kn);

    f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    constexpr int KD = 4;   // fragments under way
    ft_bf16x8 kf[KD];
    auto read_k = [&](int s) FT_INLINE {
      kf[s % KD] = *reinterpret_cast<const ft_bf16x8*>(kb + koff[s & 1] +
                                                       (s >> 1) * 128);
    };
#pragma unroll
    for (int s = 0; s < KD; ++s) read_k(s);
#pragma unroll
    for (int s = 0; s < KS; ++s) {
#pragma unroll
      for (int u = 0; u < 2; ++u)
        acc[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[s % KD], qf[u][s],
                                                         acc[u], 0, 0, 0);
      if (s + KD < KS) read_k(s + KD);
    }
    __builtin_amdgcn_sched_group_barrier(FT_DS_READ, KD, 0);
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      __builtin_amdgcn_sched_group_barrier(FT_MFMA, 2, 0);
      if (s + KD < KS) __builtin_amdgcn_sched_group_barrier(FT_DS_READ, 1, 0);
    }
    __builtin_amdgcn_sched_barrier(0);

    // lane: head lane % 32, keys 16 wave + 8 half + 0 .. 7
    float s[8];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float x = acc[0][i], y = acc[1][i];
      asm("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 0"
          : "+v"(x), "+v"(y));
      s[i] = x * c;
      s[4 + i] = y * c;
    }
    if (kbase + FT_BN - 1 > pos || kbase < lo) {
      const int first = kbase + wave * 16 + 8 * half;
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (first + i > pos || first + i < lo) s[i] = -INFINITY;
    }
    float mx = s[0];
#pragma unroll
    for (int i = 1; i < 8; ++i) mx = fmaxf(mx, s[i]);
    {
      float x, y;
      ft_both_halves(mx, x, y);
      mx = fmaxf(x, y);
    }
    if (half == 0) x_s[lane][wave] = mx;
    ld_lds_barrier();
    const float4 all = *reinterpret_cast<const float4*>(x_s[lane & 31]);
    mx = fmaxf(fmaxf(all.x, all.y), fmaxf(all.z, all.w));
    if (__any(mx > m)) {
      const float mn = fmaxf(m, mx);
      const float alpha =
          m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m - mn);
      m = mn;
      l *= alpha;
#pragma unroll
      for (int dt = 0; dt < VD / 32; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[dt][i] *= alpha;
    }
    const float mc = m == -INFINITY ? 0.0f : m;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      s[i] = __builtin_amdgcn_exp2f(s[i] - mc);
      l += s[i];
    }
    *reinterpret_cast<uint4*>(p_s[wave][lane]) =
        make_uint4(ft_pack_bf16(s[0], s[1]), ft_pack_bf16(s[2], s[3]),
                   ft_pack_bf16(s[4], s[5]), ft_pack_bf16(s[6], s[7]));
    ld_lds_barrier();
    // weights as B operand of 32 x 32 x 16, 16 keys at a time
    ft_bf16x8 pf[FT_WAVES];
#pragma unroll
    for (int j = 0; j < FT_WAVES; ++j)
      pf[j] = *reinterpret_cast<const ft_bf16x8*>(p_s[j][lane]);
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
              (lds_short4*)(kb + voff[dt & 1][e] + (dt >> 1) * 128 +
                            16 * j * ROWB));
    };
    read_v(0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < FT_WAVES; ++j) {
      if (j + 1 < FT_WAVES) read_v(j + 1);
#pragma unroll
      for (int dt = 0; dt < VD / 32; ++dt)
        o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[j & 1][dt].v, pf[j],
                                                        o[dt], 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < VD / 8; ++i) {
      __builtin_amdgcn_sched_group_barrier(FT_MFMA, 1, 0);
      if (i < 3 * (VD / 32))
        __builtin_amdgcn_sched_group_barrier(FT_DS_READ, 2, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };

  if (kb < span.end) {
    while (true) {
      int kn = span.next(kb);
      step(kb, kn, k_s0, k_s1);
      if (kn >= span.end) break;
      kb = kn;
      kn = span.next(kb);
      step(kb, kn, k_s1, k_s0);
      if (kn >= span.end) break;
      kb = kn;
    }
  }
  // the sum of all waves' keys; nobody reads the last maxima any more
  {
    float x, y;
    ft_both_halves(l, x, y);
    if (half == 0) x_s[lane][wave] = x + y;
    __syncthreads();
    const float4 all = *reinterpret_cast<const float4*>(x_s[lane & 31]);
    l = (all.x + all.y) + (all.z + all.w);
  }
  if (head >= H) return;
  if (of > 1) {
    const int64_t slot = (int64_t)blockIdx.x * H + head;
#pragma unroll
    for (int dt = 0; dt < VD / 32; ++dt)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<float4*>(a.parts.o + slot * R + wave * VD + 32 * dt +
                                   8 * g + 4 * half) =
            make_float4(o[dt][4 * g], o[dt][4 * g + 1], o[dt][4 * g + 2],
                        o[dt][4 * g + 3]);
    if (wave == 0 && half == 0) a.parts.ml[slot] = make_float2(m, l);
    return;
  }
  const float f = a.close.factor(t, head, 0) / a.close.sum(head, m, l);
  flash_store<VD>(a.close.out + (t * H + head) * R + wave * VD, o, VD, half,
                  [&](int) { return f; });
}

template <int NK, int R, bool ONCE>
__global__ __launch_bounds__(64 * FT_WAVES, 1) void latent_decode_kernel(
    LatentDecodeArgs a) {
  latent_decode_body<NK, R, ONCE>(a);
}

// One workgroup of R / 4 threads per (token, head).
static __global__ void latent_merge_kernel(FlashClose c, LatentParts p) {
  const int head = blockIdx.x % c.heads;
  const int64_t t = blockIdx.x / c.heads;
  const int2 row =
      p.each > 0 ? make_int2((int)t * p.each, p.each) : p.rows[t];
  if (row.y < 2) return;
  const int d = threadIdx.x * 4;
  const int64_t slot = (int64_t)row.x * c.heads + head;
  float m = -INFINITY;
  for (int s = 0; s < row.y; ++s)
    m = fmaxf(m, p.ml[slot + (int64_t)s * c.heads].x);
  float l = 0.0f;
  float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll 4
  for (int s = 0; s < row.y; ++s) {
    const int64_t at = slot + (int64_t)s * c.heads;
    const float2 v = p.ml[at];
    const float4 x = *reinterpret_cast<const float4*>(p.o + at * c.width + d);
    const float f = v.x == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(v.x - m);
    l = fmaf(f, v.y, l);
    o.x = fmaf(f, x.x, o.x);
    o.y = fmaf(f, x.y, o.y);
    o.z = fmaf(f, x.z, o.z);
    o.w = fmaf(f, x.w, o.w);
  }
  const float f = c.factor(t, head, 0) / c.sum(head, m, l);
  uint2 w;
  w.x = ft_pack_bf16(o.x * f, o.y * f);
  w.y = ft_pack_bf16(o.z * f, o.w * f);
  *reinterpret_cast<uint2*>(c.out + (t * c.heads + head) * c.width + d) = w;
}

// The decoded-token half of latent_attention_mfma (which has checked the
// tensors); false when the sizes do not fit.
bool latent_decode(torch::Tensor out, torch::Tensor q_abs,
                   torch::Tensor q_rot, torch::Tensor cache,
                   torch::Tensor block_table, torch::Tensor row_seq,
                   torch::Tensor positions, c10::optional<torch::Tensor> sink,
                   double scale, int64_t window, int64_t max_keys,
                   c10::optional<torch::Tensor> gate) {
  const int64_t T = q_abs.size(0), H = q_abs.size(1), R = q_abs.size(2);
  const int64_t RD = q_rot.size(2);
  auto aligned = [](const torch::Tensor& t) {
    return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0 &&
           t.stride(0) % 8 == 0 && t.stride(1) % 8 == 0;
  };
  if ((R != 512 && R != 256) || RD % 8 || RD > 64 || !aligned(q_abs) ||
      !aligned(q_rot) || !aligned(cache))
    return false;
  const int64_t groups = (H + 31) / 32;
  const int64_t cus =
      at::cuda::getCurrentDeviceProperties()->multiProcessorCount;
  const int64_t tiles = (max_keys + FT_BN - 1) / FT_BN;
  // Several groups of heads read a token's rows several times, one workgroup
  // per compute unit: of rank 256 the stacked tiles of latent_attn_mfma.hip
  // read them once for all heads, several workgroups per compute unit, and are
  // ahead from two rounds of these workgroups on (64 heads, 512 tokens of 10 /
  // 200 / 1500: 32, 66 and 297 us here, 21, 50 and 242 there; 256 tokens 18, 35
  // and 140 here, 17, 44 and 209 there).
  if (R == 256 && groups > 1 && T * groups > 2 * cus) return false;
  // Slots for the parts: as many rounds of workgroups, one per compute unit, as
  // are the fewest times the tiles of a part and about two for a workgroup's start
  // and end, if all contexts were the longest.  A part has four tiles or more (its
  // sums are as many bytes as one), of few tokens two (one of 3000 23.1 and
  // 19.3 us; 16 of 2000 27.0 and 29.6).  Up to 128 tokens share the slots by their
  // contexts' lengths, which is found on the device (32 heads, rank 512, in equal
  // numbers of parts and so: 48 of 700 to 3500 49.2 and 42.4, of 2000 each 40.4 and
  // 40.8).  Up to four tokens of rank 256 whose parts, as many as there can be, are
  // one round have them in equal numbers, of which each counts a quarter of a tile in
  // the merge (us, in equal numbers of the tile walk before, shared without that, and
  // so: 32 heads, 2 / 4 tokens of 4000 21.7 22.3, 22.8 24.8 and 19.4 20.3, of 8000 23.8
  // 24.8, 25.7 28.1 and 24.7 25.7, of 600 19.8 19.8, 13.5 13.7 and 12.8 13.1); of rank
  // 512 shared ones are ahead in a window and where lengths differ (4 tokens, 3000 and
  // three of 30, 64 heads 24.6 and 26.2).
  const bool one_round =
      R == 256 && T <= 4 && T * groups * LD_PARTS <= cus;
  const bool shared = T > 1 && T <= 64 * LD_SETS && !one_round;
  const int64_t shortest = T <= 4 ? 2 : 4;
  int64_t slots = 0, each = 0;
  int64_t least = (T * groups + cus - 1) / cus * (tiles + 2) * 4;
  for (int64_t n = 2; n <= std::min<int64_t>(LD_PARTS, tiles / shortest); ++n) {
    const int64_t rounds = (T * groups * n + cus - 1) / cus;
    const int64_t cost = rounds * ((tiles + n - 1) / n + 2) * 4 +
                         (one_round ? n : 0);
    if (cost < least) {
      least = cost;
      each = shared ? 0 : n;
      slots = shared ? std::max(rounds * cus / groups, T * n) : T * n;
    }
  }
  torch::Tensor part;
  LatentDecodeArgs a{
      (const uint16_t*)q_abs.data_ptr(), (const uint16_t*)q_rot.data_ptr(),
      q_abs.stride(0), q_abs.stride(1), q_rot.stride(0), q_rot.stride(1),
      (const uint16_t*)cache.data_ptr(), (const int32_t*)block_table.data_ptr(),
      (const int32_t*)row_seq.data_ptr(), (const int32_t*)positions.data_ptr(),
      (int)block_table.size(1), (int)RD, (int)cache.size(1), (int)window,
      (float)scale,
      FlashClose{(uint16_t*)out.data_ptr(), (int)H, (int)R,
                 sink.has_value() ? (const float*)sink->data_ptr() : nullptr,
                 gate.has_value() ? (const float*)gate->data_ptr() : nullptr,
                 nullptr, 0, 1},
      LatentParts{nullptr, nullptr, nullptr, (int)slots, (int)T, (int)each,
                  (int)shortest}};
  if (slots > 0) {
    part = torch::empty({slots * H * (R + 2) + 2 * T},
                        q_abs.options().dtype(torch::kFloat32));
    a.parts.o = part.data_ptr<float>();
    a.parts.ml = (float2*)(a.parts.o + slots * H * R);
    a.parts.rows = (int2*)(a.parts.ml + slots * H);
  }
  hipStream_t stream = at::cuda::getCurrentCUDAStream();
  const dim3 grid(slots > 0 ? slots : T, groups), block(64 * FT_WAVES);
  const bool once = T * max_keys * (R + RD) * 2 >= LD_ONCE;
  auto* kern = R == 512 ? once ? latent_decode_kernel<576, 512, true>
                               : latent_decode_kernel<576, 512, false>
               : once   ? latent_decode_kernel<320, 256, true>
                        : latent_decode_kernel<320, 256, false>;
  hipLaunchKernelGGL(kern, grid, block, 0, stream, a);
  HIP_CHECK_KERNEL();
  if (slots > 0) {
    hipLaunchKernelGGL(latent_merge_kernel, dim3(T * H), dim3(R / 4), 0, stream,
                       a.close, a.parts);
    HIP_CHECK_KERNEL();
  }
  return true;
}

}  // namespace igw
