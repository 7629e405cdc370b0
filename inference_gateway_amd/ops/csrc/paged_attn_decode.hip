// Paged-attention decode kernel for gfx950 (MI355X).
//
// Net-new engine scope (SURVEY.md §7 stage 3b): single-query attention over a
// paged KV cache, GQA-aware. One workgroup per (sequence, kv_head); the GQA
// group's G query heads ride along so each K/V byte is read exactly once per
// step.  Bound by reading the cache; what a wave needs besides is kept small so
// that its loads are always under way:
//
//   * a wave takes two pages (32 tokens) at a time, K to registers, V by DMA to
//     LDS, both one step ahead: 16 KB a wave, 128 KB a compute unit under way;
//   * eight neighbouring lanes load a 128-byte line of K, and the lines become
//     matrix operands through 2 KB of LDS of the wave's own.  Loaded as the matrix
//     unit wants them, neighbouring lanes in neighbouring tokens, a load is 64
//     requests of 16 bytes and takes the cache 65 cycles instead of 16 (61
//     sequences of 200 to 4000 tokens 112 and 109 us, 16 of 500 10.5 and 8.4, 64 of
//     100 to 2000 with a head each 54 and 52; 1024 of 570 the same);
//   * scores: S^T = K Q^T with mfma 16x16x32, the query heads in the columns,
//     each once for every part of its weights: 8 instructions for what took 256 dot
//     products;
//   * the result's token order follows from the layout of S^T and V is read from
//     LDS in the same order (ds_read_b64_tr_b16), so weights stay in their
//     lanes;
//   * weights keep all 24 bits of their mantissa: three bf16 parts, each the
//     truncated rest of the ones before.  Up to four heads leave columns for all
//     three (one product for them, their sums added at the end), eight for two.
//     No rest is below the smallest normal number, so that an infinite value stays
//     infinite at every weight.  Results that are not the nearest bf16 to 64 bits
//     (128 sequences of 200 to 700 tokens, normal entries): 2.1e-4 of them with fp32
//     multiply-adds, 1.5e-4 here, 3.7e-3 with two parts (as products of their own the
//     three took one sequence of 500 tokens 10.3 us, here 9.7, two parts 8.4; 1024 of
//     570 the same);
//   * addresses are a scalar base per page and fixed lane offsets; rows past a
//     part's end lie past the buffer descriptor's and read as zeros, without a
//     branch, so that the compiler knows which loads are under way;
//   * waves stripe over pairs of pages and merge via LDS once at the end
//     (flash-decoding style rescale);
//   * a sequence's pages are split over up to nsplit workgroups when
//     sequences x key/value heads alone do not fill the chip.  The split is
//     by the sequence's own length (read on the device, so a captured launch
//     stays right as contexts grow); the parts' unnormalised sums (fp32) are
//     merged by a second kernel.
//
// Measured, with dot products and fp32 multiply-adds on the vector units (450
// instructions a page) and here, before the loads were nontemporal (PD_ONCE; 32 heads
// on 8, us): 1024 sequences of 554 to 590 tokens 466 and 410 (5.9 TB/s), 300 of 3000
// 764 and 637, 61 of 200 to 4000 134 and 104, 128 of 100 to 2000 159 and 109, 16 of
// 500 16.5 and 11.2; 64 heads on 8, 64 of 400 to 4000 250 and 119.  One, two or eight
// waves a workgroup: 691, 654, 635 for the 637, 120, 119, 108 for the 109, 114, 109, 114
// for the 104.

#include <ATen/cuda/CUDAContext.h>
#include <torch/extension.h>

#include <type_traits>

#include "common.h"

namespace igw {

typedef __attribute__((ext_vector_type(4))) short pd_short4;
typedef __attribute__((ext_vector_type(8))) __bf16 pd_bf16x8;
typedef __attribute__((ext_vector_type(4))) float pd_f32x4;
typedef __attribute__((ext_vector_type(4))) uint32_t pd_u32x4;

#define PD_INLINE __attribute__((always_inline))
constexpr float PD_LOG2E = 1.44269504088896340736f;

// x of lanes i and i ^ 16 (i ^ 32) in a and b of both.  Written out because the
// compiler folds the builtins' two results into one when their operands are
// equal; the s_nops are the waits that the swaps need.
DEVINLINE void pd_both16(float x, float& a, float& b) {
  a = b = x;
  asm("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 0" : "+v"(a), "+v"(b));
}
DEVINLINE void pd_both32(float x, float& a, float& b) {
  a = b = x;
  asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 0" : "+v"(a), "+v"(b));
}

// From this many tokens x key heads on, a workgroup's own context for every
// sequence of the step (40 MB of keys and values), the cache is read with
// nontemporal loads.  What is read once a step and cannot wait for the next one in
// the 256 MB memory-side cache is then not put there first: 1024 sequences of 570
// tokens 5.8 and 6.5 TB/s.  Below, several layers' caches fit it together, and loads
// that pass it by are the slower ones (us, 32 heads on 8, eight caches in turn,
// plain and nontemporal: 9 of 500 10.5 and 12.1, of 700 12.2 and 14.1, of 1500 23.6
// and 21.8; 16 of 500 11.4 and 12.4, of 700 16.6 and 14.8; 4 of 1500 14.8 and 14.7,
// of 4000 21.7 and 19.5; 64 of 700 40.4 and 34.8, 128 of 700 75 and 63, 1024 of 500
// 376 and 337; 33 of 16000 400 and 351).
constexpr int64_t PD_ONCE = 80000;

// maximum and sum over the four lanes that share lane & 15
DEVINLINE float pd_max(float x) {
  float a, b;
  pd_both16(x, a, b);
  pd_both32(fmaxf(a, b), a, b);
  return fmaxf(a, b);
}
DEVINLINE float pd_sum(float x) {
  float a, b;
  pd_both16(x, a, b);
  pd_both32(a + b, a, b);
  return a + b;
}

// How a sequence of ctx tokens is cut for nsplit workgroups: `count` parts of
// `blocks` pages, a part no shorter than min_blocks pages.  Up to 32 pages are
// not cut: what a merge costs is not won back (1 sequence of 200 tokens 5.7 us
// whole, 7.2 cut; of 500 8.0 and 8.2, of 700 9.8 and 9.1, of 1500 16.4 and 8.9).
struct DecodeSplit {
  int blocks, count;
  DEVINLINE DecodeSplit(int ctx, int nsplit, int min_blocks) {
    const int n = (ctx + 15) / 16;
    blocks = max((n + nsplit - 1) / nsplit, min_blocks);
    if (nsplit == 1 || n <= 32) blocks = max(n, 1);
    count = max((n + blocks - 1) / blocks, 1);
  }
};

// What rope_append would have done before: queries are rotated as they are loaded,
// and a sequence's new key and value go to the cache from the wave that reads their
// page, before it does (a wave's accesses to memory keep their order).  That is the
// last page of the context, or else every wave looks its own pages through and each
// that has the slot's writes it, the same bytes, and the last wave in any case.  What
// other sequences read must not be written: a sequence that reads another's slot sees
// it as it was or as it becomes.  As a launch of its own it takes 2 to 3 us of a small
// step's layer; ops.rope_paged_attn_decode says up to where this is ahead.
struct DecodeRope {
  const int32_t* positions;   // [B]
  const int32_t* slots;       // [B]: page * 16 + offset, < 0: not stored
  const float* cos_sin;       // [positions, HD]
  const uint16_t *k, *v;      // [B, NKV * HD], row strides k_rs and v_rs
  int64_t k_rs, v_rs;
};

template <int G, int NWAVES, bool ROPE>
__global__ __launch_bounds__(NWAVES* WAVE_SIZE, 2) void paged_attn_decode_kernel(
    uint16_t* __restrict__ out,          // [B, NQ, HD]
    const uint16_t* __restrict__ q,      // [B, NQ, HD]
    uint16_t* kcache,                    // [NB, NKV, BS, HD]
    uint16_t* vcache,                    // [NB, NKV, BS, HD]
    const int32_t* __restrict__ block_table, // [B, max_blocks]
    const int32_t* __restrict__ ctx_lens,    // [B]
    int max_blocks, int nkv, float scale, int q_rs,
    float* __restrict__ part_o,   // [B, NQ, nsplit, HD] when nsplit > 1
    float* __restrict__ part_ml,  // [B, NQ, nsplit, 2]: maximum (log2), sum
    int nsplit, int min_blocks, int once_ctx, DecodeRope rope) {
  // q_rs: q row stride in elements (q may be a view into the fused QKV
  // GEMM output — no .contiguous() copy on the decode hot path)
  constexpr int HD = 128, BS = 16, PAGE = BS * HD;  // tokens, entries of a page
  // columns of the matrix products: the heads, once for each part of their
  // weights (with eight heads the second column has the third part too)
  constexpr int PARTS = G <= 4 ? 3 : 2, COLS = PARTS * G;
  static_assert(COLS * HD * 4 <= 2 * PAGE * 2, "a wave's results fit its V tiles");
  // a wave's own V tiles, two pages each, and K lines: nothing here waits for
  // another wave.
  // Two objects, so that reads of one do not wait for loads to the other.
  __shared__ __attribute__((aligned(1024))) uint16_t v_s0[NWAVES][2 * PAGE];
  __shared__ __attribute__((aligned(1024))) uint16_t v_s1[NWAVES][2 * PAGE];
  __shared__ __attribute__((aligned(1024))) pd_u32x4 k_s[NWAVES][128];
  __shared__ float m_lds[NWAVES][G];
  __shared__ float l_lds[NWAVES][G];
  const int kvh = blockIdx.x;
  const int seq = blockIdx.y;
  const int nq = nkv * G;
  const int ctx = __builtin_amdgcn_readfirstlane(ctx_lens[seq]);
  const int split = blockIdx.z;
  const DecodeSplit part(ctx, nsplit, min_blocks);
  if (split >= part.count) return;
  const int block0 = split * part.blocks;
  const int nblocks = min((ctx + BS - 1) / BS, block0 + part.blocks);
  const int limit = min(ctx, nblocks * BS);        // the part's tokens end here
  const int pairs = (nblocks - block0 + 1) >> 1;   // wave, wave + NWAVES, ...

  const int tid = threadIdx.x;
  const int lane = tid & (WAVE_SIZE - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, quad = lane >> 4;
  const int32_t* bt_row = block_table + (int64_t)seq * max_blocks;

  // page numbers of this wave's next 32 pairs, one per lane: an address does
  // not wait for a table entry, and its base is in scalar registers
  int ids = 0;
  auto load_ids = [&](int u) PD_INLINE {
    const int b = block0 + 2 * (u + (lane >> 1) * NWAVES) + (lane & 1);
    ids = bt_row[min(b, nblocks - 1)];
    __builtin_amdgcn_s_waitcnt(0x0f70);   // here, not at every use
  };
  if (wave < pairs) load_ids(wave);

  // the query heads as columns: head r16 % G, dims 32 kk + 8 quad ..
  pd_bf16x8 qf[4];
#pragma unroll
  for (int kk = 0; kk < 4; ++kk) {
    pd_bf16x8 f{};
    if (r16 < COLS)
      f = *reinterpret_cast<const pd_bf16x8*>(q + (int64_t)seq * q_rs +
                                              (kvh * G + r16 % G) * HD +
                                              kk * 32 + quad * 8);
    qf[kk] = f;
  }
  if (ROPE) {
    const float* cs = rope.cos_sin + (int64_t)rope.positions[seq] * HD;
    auto turned = [&](ushort8& a, ushort8& b, int d) PD_INLINE {
      const float4* c = reinterpret_cast<const float4*>(cs + d);
      const float4* s = reinterpret_cast<const float4*>(cs + HD / 2 + d);
      const float4 c0 = c[0], c1 = c[1], s0 = s[0], s1 = s[1];
      const float cv[8] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w};
      const float sv[8] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};
#pragma unroll
      for (int j = 0; j < 8; ++j) rope_pair(a.v[j], b.v[j], cv[j], sv[j]);
    };
    const int slot = rope.slots[seq];
    bool write = split == part.count - 1 && slot >= 0 &&
                 wave == (pairs > 0 ? (pairs - 1) % NWAVES : 0);
    if (slot >= 0 && ctx > 0 && slot / BS != bt_row[(ctx - 1) / BS]) {
      bool here = false;
      for (int u = wave; u < pairs; u += 32 * NWAVES) {
        const int b = block0 + 2 * (u + (lane >> 1) * NWAVES) + (lane & 1);
        here |= b < nblocks && bt_row[min(b, nblocks - 1)] == slot / BS;
      }
      write |= __ballot(here) != 0;
    }
    if (write) {
      const int64_t cell =
          ((int64_t)(slot / BS * nkv + kvh) * BS + slot % BS) * HD;
      if (lane < 8) {
        const uint16_t* k = rope.k + seq * rope.k_rs + kvh * HD + lane * 8;
        ushort8 a = *reinterpret_cast<const ushort8*>(k);
        ushort8 b = *reinterpret_cast<const ushort8*>(k + HD / 2);
        turned(a, b, lane * 8);
        *reinterpret_cast<ushort8*>(kcache + cell + lane * 8) = a;
        *reinterpret_cast<ushort8*>(kcache + cell + HD / 2 + lane * 8) = b;
      } else if (lane >= 16 && lane < 32) {
        *reinterpret_cast<ushort8*>(vcache + cell + (lane - 16) * 8) =
            *reinterpret_cast<const ushort8*>(rope.v + seq * rope.v_rs +
                                              kvh * HD + (lane - 16) * 8);
      }
      asm volatile("" ::: "memory");
    }
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      ushort8 a = __builtin_bit_cast(ushort8, qf[kk]);
      ushort8 b = __builtin_bit_cast(ushort8, qf[kk + 2]);
      turned(a, b, kk * 32 + quad * 8);
      qf[kk] = __builtin_bit_cast(pd_bf16x8, a);
      qf[kk + 2] = __builtin_bit_cast(pd_bf16x8, b);
    }
  }

  // lane offsets into a page, bytes: K half a row of eight rows a load, turned
  // with its 16-byte pieces permuted by the row (no bank conflicts); V four rows
  // a load, 16-byte chunks exchanged so that the eight rows which 32 lanes
  // of a transposing read take 32 bytes of each lie in different banks
  const int kx = (lane >> 3) * HD * 2 + (lane & 7) * 16;
  const LineTurn turn(lane);
  int vx[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = i * 4 + quad;
    vx[i] = r * HD * 2 + ((r16 ^ ((r & 7) << 1)) << 4);
  }
  struct Keys {
    pd_u32x4 k[2][4];
  };
  typedef __attribute__((address_space(3))) void lds_void;
  // pair u; past the part's end nothing is read and the values are zeros
  auto fetch = [&](auto once, int u, Keys& K, uint16_t* vs) PD_INLINE {
    constexpr int NT = decltype(once)::value ? 2 : 0;   // bit 1: nontemporal
    const int at = (u - wave) / NWAVES;
    const int left = limit - (block0 + 2 * u) * BS;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int64_t page = __builtin_amdgcn_readlane(ids, (at & 31) * 2 + h);
      const int64_t base = (page * nkv + kvh) * PAGE;
      const int rows =
          __builtin_amdgcn_readfirstlane(max(0, min(BS, left - h * BS)));
      const auto kr = __builtin_amdgcn_make_buffer_rsrc(
          (void*)(kcache + base), 0, rows * HD * 2, 0x00020000);
      const auto vr = __builtin_amdgcn_make_buffer_rsrc(
          (void*)(vcache + base), 0, rows * HD * 2, 0x00020000);
#pragma unroll
      for (int kk = 0; kk < 4; ++kk)
        K.k[h][kk] =
            __builtin_amdgcn_raw_buffer_load_b128(
                kr, kx + (kk >> 1) * 128 + (kk & 1) * 8 * HD * 2, 0, NT);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            vr, (lds_void*)(vs + h * PAGE + i * 512), 16, vx[i], 0, 0, NT);
    }
  };

  // O^T: column r16, dims 16 d + 4 quad ..; m in log2, l of this lane's tokens
  pd_f32x4 acc[8];
#pragma unroll
  for (int d = 0; d < 8; ++d) acc[d] = pd_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  // what this column's part leaves out of a weight
  const int part_of = r16 / G;
  constexpr uint32_t TOP = 0xffff0000u;
  const uint32_t first = part_of > 0 ? TOP : 0, second = part_of > 1 ? TOP : 0;
  const uint32_t third = part_of == 1 ? ~0u : 0;
  const float least = part_of > 0 ? 0x1p-126f : 0.0f;
  float m = -INFINITY, l = 0.0f;
  const float c = scale * PD_LOG2E;
  const int vrow = 4 * quad + (r16 >> 2);
  auto use = [&](int u, const Keys& K, uint16_t* vs) PD_INLINE {
    pd_f32x4 s[2], s1[2];   // of the dims' halves: half the roundings
#pragma unroll
    for (int h = 0; h < 2; ++h) s[h] = s1[h] = pd_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    pd_u32x4* ks = k_s[wave];
    pd_u32x4 kf[2][4];
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        turn(ks, K.k[h][2 * c], K.k[h][2 * c + 1], kf[h][2 * c],
             kf[h][2 * c + 1]);
#pragma unroll
    for (int kk = 0; kk < 4; ++kk)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        pd_f32x4& sum = kk < 2 ? s[h] : s1[h];
        sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            __builtin_bit_cast(pd_bf16x8, kf[h][kk]), qf[kk], sum, 0, 0, 0);
      }
#pragma unroll
    for (int h = 0; h < 2; ++h) s[h] += s1[h];
    // token 16 (j / 4) + 4 quad + j % 4 of the pair
    float t[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) t[j] = s[j >> 2][j & 3] * c;
    const int left = limit - (block0 + 2 * u) * BS;
    if (left < 2 * BS) {
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if ((j >> 2) * 16 + 4 * quad + (j & 3) >= left) t[j] = -INFINITY;
    }
    float mx = t[0];
#pragma unroll
    for (int j = 1; j < 8; ++j) mx = fmaxf(mx, t[j]);
    mx = pd_max(mx);
    if (__any(mx > m)) {
      const float mn = fmaxf(m, mx);
      const float alpha =
          m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m - mn);
      m = mn;
      l *= alpha;
#pragma unroll
      for (int d = 0; d < 8; ++d) acc[d] *= alpha;
    }
    const float mc = m == -INFINITY ? 0.0f : m;
    float p[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      // one rounding, of the difference
      const float x = fmaf(s[j >> 2][j & 3], c, -mc);
      p[j] = t[j] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(x);
    }
    l += ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
    union {
      uint32_t u[4];
      pd_bf16x8 v;
    } w, w3;
    auto minus = [](float x, uint32_t mask) PD_INLINE {
      return x - __uint_as_float(__float_as_uint(x) & mask);
    };
    auto pack = [](float a, float b) PD_INLINE {   // truncated
      return (__float_as_uint(a) >> 16) | (__float_as_uint(b) & TOP);
    };
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float x[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) x[i] = minus(p[2 * e + i], first);
      if (PARTS == 3) {
#pragma unroll
        for (int i = 0; i < 2; ++i) x[i] = minus(x[i], second);
      } else {
        float y[2];
#pragma unroll
        for (int i = 0; i < 2; ++i)
          y[i] = fmaxf(__uint_as_float(__float_as_uint(minus(x[i], TOP)) & third),
                       0x1p-126f);
        w3.u[e] = pack(y[0], y[1]);
      }
      w.u[e] = pack(fmaxf(x[0], least), fmaxf(x[1], least));
    }
    typedef __attribute__((address_space(3))) pd_short4 lds_short4;
#pragma unroll
    for (int d = 0; d < 8; ++d) {
      union {
        pd_short4 h[2];
        pd_bf16x8 v;
      } vf;
      const int chunk = (2 * d + ((r16 & 3) >> 1)) ^ ((vrow & 7) << 1);
#pragma unroll
      for (int h = 0; h < 2; ++h)
        vf.h[h] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (lds_short4*)(vs + h * PAGE + vrow * HD + chunk * 8 +
                          (r16 & 1) * 4));
      if (PARTS == 2)
        acc[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf.v, w3.v, acc[d], 0,
                                                         0, 0);
      acc[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf.v, w.v, acc[d], 0, 0,
                                                       0);
    }
  };

  Keys k0, k1;
  auto walk = [&](auto once) PD_INLINE {
    auto ahead = [&](int u, Keys& K, uint16_t* vs) PD_INLINE {
      if ((((u - wave) / NWAVES) & 31) == 0 && u < pairs) load_ids(u);
      fetch(once, u, K, vs);
    };
    fetch(once, wave, k0, v_s0[wave]);
    for (int u = wave;; u += 2 * NWAVES) {
      ahead(u + NWAVES, k1, v_s1[wave]);
      use(u, k0, v_s0[wave]);
      if (u + NWAVES >= pairs) break;
      ahead(u + 2 * NWAVES, k0, v_s0[wave]);
      use(u + NWAVES, k1, v_s1[wave]);
      if (u + 2 * NWAVES >= pairs) break;
    }
  };
  if (wave < pairs) {
    if (ctx >= once_ctx) walk(std::true_type{});   // PD_ONCE
    else walk(std::false_type{});
  }
  l = pd_sum(l);

  // ---- cross-wave merge, in the memory of the V tiles (the loads that are
  //      still under way there read nothing, and are waited for first)
  // (up to four pages are the first or the first two waves')
  const int waves = pairs <= 2 ? max(pairs, 1) : NWAVES;
  float* acc_lds = reinterpret_cast<float*>(&v_s0[0][0]);  // [NWAVES][COLS][HD]
  __builtin_amdgcn_s_waitcnt(0x0f70);
  __syncthreads();
  if (wave < waves && r16 < COLS) {
    if (r16 < G && quad == 0) {
      m_lds[wave][r16] = m;
      l_lds[wave][r16] = l;
    }
#pragma unroll
    for (int d = 0; d < 8; ++d)
      *reinterpret_cast<pd_f32x4*>(acc_lds + (wave * COLS + r16) * HD + d * 16 +
                                   quad * 4) = acc[d];
  }
  __syncthreads();

  auto merge = [&](auto waves_) PD_INLINE {
    constexpr int WAVES = decltype(waves_)::value;
    for (int i = tid; i < G * HD; i += NWAVES * WAVE_SIZE) {
      const int j = i / HD;
      const int d = i % HD;
      float M = -INFINITY;
#pragma unroll
      for (int w = 0; w < WAVES; ++w) M = fmaxf(M, m_lds[w][j]);
      float L = 0.0f, o = 0.0f;
#pragma unroll
      for (int w = 0; w < WAVES; ++w) {
        const float f = m_lds[w][j] == -INFINITY
                            ? 0.0f
                            : __builtin_amdgcn_exp2f(m_lds[w][j] - M);
        L = fmaf(f, l_lds[w][j], L);
        float sum = 0.0f;   // of the parts, the smallest first
#pragma unroll
        for (int t = PARTS - 1; t >= 0; --t)
          sum += acc_lds[(w * COLS + t * G + j) * HD + d];
        o = fmaf(f, sum, o);
      }
      const int64_t head = (int64_t)seq * nq + kvh * G + j;
      if (part.count == 1) {
        out[head * HD + d] = f32_to_bf16(o / L);
      } else {
        part_o[(head * nsplit + split) * HD + d] = o;
        if (d == 0) {
          part_ml[(head * nsplit + split) * 2] = M;
          part_ml[(head * nsplit + split) * 2 + 1] = L;
        }
      }
    }
  };
  if (waves == 1) merge(std::integral_constant<int, 1>{});
  else if (waves == 2) merge(std::integral_constant<int, 2>{});
  else merge(std::integral_constant<int, NWAVES>{});
}

// Merges the parts of every (sequence, head) that has more than one: one
// workgroup of HD threads each.  The threads first weigh the parts side by
// side (a loop over them would wait for memory at every step), then each sums
// one dim over the parts, 8 loads in flight.
template <int HD>
__global__ __launch_bounds__(HD) void paged_attn_merge_kernel(
    uint16_t* __restrict__ out, const float* __restrict__ part_o,
    const float* __restrict__ part_ml, const int32_t* __restrict__ ctx_lens,
    int nq, int nsplit, int min_blocks) {
  constexpr int NW = HD / WAVE_SIZE;
  __shared__ float red[NW];
  __shared__ float weight[HD];
  const int seq = blockIdx.y, tid = threadIdx.x;
  const DecodeSplit part(ctx_lens[seq], nsplit, min_blocks);
  if (part.count == 1) return;
  const int64_t head = (int64_t)seq * nq + blockIdx.x;
  const float2* ml = reinterpret_cast<const float2*>(part_ml) + head * nsplit;
  const float* po = part_o + head * nsplit * HD + tid;
  float M = -INFINITY;
  for (int s = tid; s < part.count; s += HD) M = fmaxf(M, ml[s].x);
  M = wave_reduce_max(M);
  if ((tid & 63) == 0) red[tid >> 6] = M;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < NW; ++w) M = fmaxf(M, red[w]);
  float L = 0.0f, o = 0.0f;
  for (int s0 = 0; s0 < part.count; s0 += HD) {
    const int n = min(HD, part.count - s0);
    __syncthreads();   // weight (and red) were read by everybody
    float l = 0.0f;
    if (tid < n) {
      const float2 v = ml[s0 + tid];
      const float f =
          v.x == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(v.x - M);
      weight[tid] = f;
      l = f * v.y;
    }
    l = wave_reduce_sum(l);
    if ((tid & 63) == 0) red[tid >> 6] = l;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < NW; ++w) L += red[w];
#pragma unroll 8
    for (int s = 0; s < n; ++s)
      o = fmaf(weight[s], po[(int64_t)(s0 + s) * HD], o);
  }
  out[head * HD + tid] = f32_to_bf16(o / L);
}

template <int G>
static void launch_decode(torch::Tensor& out, const torch::Tensor& q,
                          const torch::Tensor& kcache,
                          const torch::Tensor& vcache,
                          const torch::Tensor& block_table,
                          const torch::Tensor& ctx_lens, float scale,
                          const DecodeRope* rope, hipStream_t stream) {
  const int B = q.size(0);
  const int nkv = kcache.size(1);
  constexpr int HD = 128;
  const int nq = q.size(1);
  const int max_blocks = block_table.size(1);
  // The chip holds 512 of these workgroups (two per compute unit, by their
  // registers).  Where sequences x heads are an eighth of that, they wait for
  // memory, pair of pages after pair, and gain from parts of a pair per wave
  // until they fill the chip once or a merge has 32 parts.  From there on the
  // chip as a whole is at the memory's rate and equal contexts gain nothing
  // (they lose what the merge costs); cut in long parts, the long ones among
  // ragged contexts do not end alone.  Measured, whole and cut by these lines
  // (us): 8 heads, 1 sequence of 3000 tokens 29.1 and 8.5, of 8000 71.4 and
  // 10.6, 5 of 750 to 1500 16.6 and 11.4, 8 of 1000 13.0 and 10.7; 33 of 300 to
  // 3000 47.5 and 40.5, 40 of 200 to 4000 93.5 and 72.2, 61 of them 117 and 104,
  // 90 of 100 to 3000 119 and 115; but 24 of 3000 46.4 and 53.6, 64 of 4000 183
  // and 188.  With 1024 workgroups a split only adds the merge (128 of 100 to
  // 2000 tokens: 107 and 110).  Whether anything is cut is known on the device
  // only: where the block table is wide and the contexts are short the merge is
  // launched for nothing (1.6 to 2 us).
  const int whole = std::max(1, B * nkv);
  const bool few = whole <= 64;
  const int min_blocks = few ? 8 : 64;
  const int nsplit =
      whole >= 1024 || max_blocks <= 32
          ? 1
          : std::max(1, std::min(few ? std::min(512 / whole, 32) : 2048 / whole,
                                 (max_blocks + min_blocks - 1) / min_blocks));
  torch::Tensor part;
  float *part_o = nullptr, *part_ml = nullptr;
  if (nsplit > 1) {
    const int64_t n = (int64_t)B * nq * nsplit;
    part = torch::empty({n * (HD + 2)}, q.options().dtype(torch::kFloat32));
    part_o = part.data_ptr<float>();
    part_ml = part_o + n * HD;
  }
  const int once_ctx = (int)((PD_ONCE + whole - 1) / whole);
  auto launch = [&](auto waves_) {
    constexpr int NWAVES = decltype(waves_)::value;
    auto kern = rope ? paged_attn_decode_kernel<G, NWAVES, true>
                     : paged_attn_decode_kernel<G, NWAVES, false>;
    hipLaunchKernelGGL(kern, dim3(nkv, B, nsplit), dim3(NWAVES * WAVE_SIZE), 0,
                       stream, (uint16_t*)out.data_ptr(),
                       (const uint16_t*)q.data_ptr(),
                       (uint16_t*)kcache.data_ptr(),
                       (uint16_t*)vcache.data_ptr(),
                       (const int32_t*)block_table.data_ptr(),
                       (const int32_t*)ctx_lens.data_ptr(), max_blocks, nkv,
                       scale, (int)q.stride(0), part_o, part_ml, nsplit,
                       min_blocks, once_ctx, rope ? *rope : DecodeRope{});
  };
  // Four waves a workgroup, but two where one or two query heads share a key head and
  // the chip is filled many times over: the bytes of a short context are few for its
  // workgroup's start and end, and twice as many are there at a time (us, four and
  // two: a head each, 256 sequences of 60 tokens 20.7 and 18.4, 1024 70.6 and 55, of
  // 500 and more the same; 64 of 4000 189 and 200).  With more heads two are 3 %
  // behind over long contexts.
  if (G <= 2 && whole >= 1024)
    launch(std::integral_constant<int, G <= 2 ? 2 : 4>{});
  else
    launch(std::integral_constant<int, 4>{});
  HIP_CHECK_KERNEL();
  if (nsplit > 1) {
    hipLaunchKernelGGL((paged_attn_merge_kernel<HD>), dim3(nq, B), dim3(HD), 0,
                       stream, (uint16_t*)out.data_ptr(), part_o, part_ml,
                       (const int32_t*)ctx_lens.data_ptr(), nq, nsplit,
                       min_blocks);
    HIP_CHECK_KERNEL();
  }
}

static void decode(torch::Tensor& out, const torch::Tensor& q,
                   const torch::Tensor& kcache, const torch::Tensor& vcache,
                   const torch::Tensor& block_table,
                   const torch::Tensor& ctx_lens, double scale,
                   const DecodeRope* rope) {
  TORCH_CHECK(q.is_cuda() && q.dtype() == torch::kBFloat16);
  TORCH_CHECK(q.stride(-1) == 1 && q.stride(1) == q.size(2));
  TORCH_CHECK(out.is_contiguous());
  TORCH_CHECK(kcache.size(3) == 128, "only head_dim=128 is supported");
  TORCH_CHECK(kcache.size(2) == 16, "only block_size=16 is supported");
  TORCH_CHECK(block_table.dtype() == torch::kInt32 &&
              ctx_lens.dtype() == torch::kInt32);
  const int nkv = kcache.size(1);
  const int nq = q.size(1);
  const int G = nq / nkv;
  TORCH_CHECK(nq % nkv == 0, "n_q_heads must be a multiple of n_kv_heads");
  hipStream_t stream = at::cuda::getCurrentCUDAStream();
  switch (G) {
    case 1:
      launch_decode<1>(out, q, kcache, vcache, block_table, ctx_lens,
                       (float)scale, rope, stream);
      break;
    case 2:
      launch_decode<2>(out, q, kcache, vcache, block_table, ctx_lens,
                       (float)scale, rope, stream);
      break;
    case 4:
      launch_decode<4>(out, q, kcache, vcache, block_table, ctx_lens,
                       (float)scale, rope, stream);
      break;
    case 8:
      launch_decode<8>(out, q, kcache, vcache, block_table, ctx_lens,
                       (float)scale, rope, stream);
      break;
    default:
      TORCH_CHECK(false, "unsupported GQA group size: ", G);
  }
}

void paged_attn_decode(torch::Tensor out, torch::Tensor q,
                       torch::Tensor kcache, torch::Tensor vcache,
                       torch::Tensor block_table, torch::Tensor ctx_lens,
                       double scale) {
  decode(out, q, kcache, vcache, block_table, ctx_lens, scale, nullptr);
}

// rope_append of q, k and v (q and k are left as they are), then
// paged_attn_decode of the rotated q [B, NQ * HD].
void rope_paged_attn_decode(torch::Tensor out, torch::Tensor positions,
                            torch::Tensor q, torch::Tensor k, torch::Tensor v,
                            torch::Tensor cos_sin_cache, torch::Tensor kcache,
                            torch::Tensor vcache, torch::Tensor slot_mapping,
                            torch::Tensor block_table, torch::Tensor ctx_lens,
                            double scale) {
  TORCH_CHECK(q.is_cuda() && q.dim() == 2 && k.dim() == 2 && v.dim() == 2 &&
              q.dtype() == torch::kBFloat16 && k.dtype() == q.dtype() &&
              v.dtype() == q.dtype() && kcache.dtype() == q.dtype() &&
              vcache.dtype() == q.dtype());
  TORCH_CHECK(positions.dtype() == torch::kInt32 &&
              slot_mapping.dtype() == torch::kInt32 &&
              positions.is_contiguous() && slot_mapping.is_contiguous());
  TORCH_CHECK(cos_sin_cache.dtype() == torch::kFloat32 &&
              cos_sin_cache.is_contiguous() && cos_sin_cache.size(-1) == 128);
  TORCH_CHECK(kcache.dim() == 4 && kcache.is_contiguous() &&
              vcache.is_contiguous() && vcache.sizes() == kcache.sizes() &&
              kcache.size(3) == 128);
  const int64_t B = q.size(0), nkv = kcache.size(1);
  TORCH_CHECK(positions.numel() == B && slot_mapping.numel() == B &&
              k.size(0) == B && v.size(0) == B && k.size(1) == nkv * 128 &&
              v.size(1) == nkv * 128 && q.size(1) % (nkv * 128) == 0);
  for (const auto* t : {&q, &k, &v})
    TORCH_CHECK(t->stride(1) == 1 && t->stride(0) % 8 == 0 &&
                (reinterpret_cast<uintptr_t>(t->data_ptr()) & 15) == 0);
  for (const auto* t : {&out, &positions, &k, &v, &cos_sin_cache, &kcache,
                        &vcache, &slot_mapping, &block_table, &ctx_lens})
    TORCH_CHECK(t->device() == q.device(), "tensors on different devices");
  const DecodeRope rope{(const int32_t*)positions.data_ptr(),
                        (const int32_t*)slot_mapping.data_ptr(),
                        (const float*)cos_sin_cache.data_ptr(),
                        (const uint16_t*)k.data_ptr(),
                        (const uint16_t*)v.data_ptr(), k.stride(0),
                        v.stride(0)};
  decode(out, q.unflatten(1, {-1, 128}), kcache, vcache, block_table, ctx_lens,
         scale, &rope);
}

}  // namespace igw
