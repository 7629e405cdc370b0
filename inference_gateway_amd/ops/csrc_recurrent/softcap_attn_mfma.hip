// Causal softmax attention with a score cap on MFMA tiles (gfx950, bf16):
// the serving path of softcap_attention, generalised over the engine's prompt
// attention by
//
//   * key width N and value width P of their own, each padded with zeros
//     to the template's NP / PP (N, P multiples of 8);
//   * any page size;
//   * score = q.k * scale * temp(position), then cap * tanh(. / cap);
//   * an optional sliding window (with, optionally, the first tokens of the
//     sequence kept in sight: the tiles between them and the window are
//     never fetched), an optional restriction to the row's own chunk of
//     positions, an optional linear distance bias per head
//     (slope * (row position - key position) is taken off the score), an
//     optional sink term per head in the softmax denominator and an
//     optional sigmoid output gate (per value entry or per head).
//
// Values of at most 128 entries run the tile walk of flash_tile.h
// (softcap_prompt_kernel: 128 rows of one head; softcap_decode_kernel: the
// heads that share a key/value head), decoded rows of 128 entries in pages of 16
// softcap_pages_kernel.  Wider ones, whose accumulators do not
// fit two waves per SIMD there, run softcap_attention_mfma_kernel: 64 rows x
// 64 keys, 4 waves of 16 rows, mfma_f32_16x16x32_bf16, K staged row-major and
// V transposed in swizzled LDS, probabilities through a per-wave LDS tile.  Its
// row maps: prompt tiles (64 consecutive tokens of one head), and decoded rows
// (HEADS_ROWS), where the rows of a tile are the query heads that share one
// key/value head, so every K/V page is staged once per group instead of once
// per head (grid = decoded rows x key/value heads).
//
// Measured (32 heads on 8, N = P = 128), 64-row tiles for all and the tile
// walk: prompts of 3000 and 2790 tokens, window 1024 with 16 kept tokens,
// distance bias and head gate 563 and 156 us; 4 prompts of 2048, causal, with
// a sink 1293 and 197 us, with a score cap 1412 and 227 us; decoded, on pages of a
// size that softcap_pages_kernel does not take, 256 tokens of 2048 keys 863 and 388 us
// (5.5 TB/s), 48 of 700 to 3500 with that window 103 and 51, one of 3000 181 and 17
// (split over workgroups).
//
// Everything is read from the paged cache; a row's own key is already
// appended.  Sequence s has rows [seq_cu[s], seq_cu[s+1]) whose first sits
// at position seq_start[s]; the first sequences are the prompt portions.
#include "../csrc/flash_tile.h"
#include "../csrc_hybrid/act_types.h"

namespace igw {

typedef __attribute__((ext_vector_type(8))) short short8v;
typedef __attribute__((ext_vector_type(4))) float float4v;

// XOR byte swizzle inside a row of ROWB bytes: 16-lane 16-byte fragment
// reads of consecutive rows land in different banks
template <int ROWB>
DEVINLINE int swz(int row, int colbyte) {
  return colbyte ^ ((row & (ROWB >= 256 ? 15 : 7)) << 4);
}

// The transposed V tile (rows = value entries, 128 bytes of keys each) is
// WRITTEN by lanes whose rows differ by multiples of 8 and READ by lanes on
// 16 consecutive rows; folding both the low and the next three row bits
// into the 16-byte chunk index keeps either access to two lanes per bank.
DEVINLINE int swz_vt(int row, int colbyte) {
  return colbyte ^ ((((row & 7) ^ ((row >> 3) & 7))) << 4);
}

DEVINLINE float tanh_fast(float x) {
  return 1.0f - 2.0f * __frcp_rn(1.0f + __expf(2.0f * x));
}

constexpr int SA_BM = 64;
constexpr int SA_BN = 64;
constexpr int SA_BT_LDS = 1024;   // page numbers kept in LDS per sequence

template <int NP, int PP, bool HEADS_ROWS>
__global__ __launch_bounds__(256, 2) void softcap_attention_mfma_kernel(
    uint16_t* __restrict__ out, const uint16_t* __restrict__ q, int64_t q_rs,
    const uint16_t* __restrict__ kcache, const uint16_t* __restrict__ vcache,
    const int32_t* __restrict__ block_table, int max_blocks,
    const int32_t* __restrict__ seq_cu, const int32_t* __restrict__ seq_start,
    int nprompt, int H, int G, int N, int P, int BS, float scale,
    float softcap,
    float temp_coef, int temp_every, int window,
    const float* __restrict__ slopes, int chunk, int keep,
    const float* __restrict__ sinks, const uint16_t* __restrict__ gate,
    int64_t gate_rs, int gate_w) {
  constexpr int BM = SA_BM, BN = SA_BN;
  constexpr int KROWB = NP * 2;          // bytes per staged Q / K row
  // K tile (shared with the Q staging) | V^T tile | per-wave P tiles
  __shared__ __attribute__((aligned(16)))
  uint16_t smem[BN * NP + PP * BN + 4 * 16 * BN];
  uint16_t* k_s = smem;
  uint16_t* vt_s = smem + BN * NP;
  uint16_t* p_s = vt_s + PP * BN;

  int seq = nprompt + blockIdx.x, qoff = 0;
  if (!HEADS_ROWS && !ft_find_tile<BM>(seq_cu, nprompt, blockIdx.x, &seq, &qoff))
    return;
  const int q0 = seq_cu[seq];
  const int Lq = HEADS_ROWS ? 1 : seq_cu[seq + 1] - q0;
  const int P0 = seq_start[seq];
  const int KVL = P0 + Lq;
  const int rep = H / G;
  const int kvh = HEADS_ROWS ? blockIdx.y : blockIdx.y / rep;
  const int nrows = HEADS_ROWS ? rep : min(BM, Lq - qoff);  // valid rows
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  uint16_t* pw_s = p_s + wave * 16 * BN;
  // the sequence's page numbers sit in LDS when they fit, so that a K/V
  // address does not wait on a second global load
  __shared__ int32_t bt_s[SA_BT_LDS];
  const int32_t* bt_row = block_table + (int64_t)seq * max_blocks;
  const int nblk = (KVL + BS - 1) / BS;
  if (nblk <= SA_BT_LDS) {
    for (int i = tid; i < nblk; i += 256) bt_s[i] = bt_row[i];
    bt_row = bt_s;      // visible after the barrier that follows Q staging
  }

  // ---- Q tile -> LDS (the K region) -> A fragments ----
  for (int it = 0; it < BM * NP / 8 / 256; ++it) {
    const int idx = tid + it * 256;
    const int row = idx / (NP / 8);
    const int d8 = (idx % (NP / 8)) * 8;
    const int r = min(row, nrows - 1);
    const int64_t tok = HEADS_ROWS ? q0 : q0 + qoff + r;
    const int head = HEADS_ROWS ? kvh * rep + r : blockIdx.y;
    ushort8 val;
    if (d8 < N) {
      val = *reinterpret_cast<const ushort8*>(q + tok * q_rs + head * N + d8);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) val.v[e] = 0;
    }
    *reinterpret_cast<ushort8*>(reinterpret_cast<char*>(k_s) + row * KROWB +
                                swz<KROWB>(row, d8 * 2)) = val;
  }
  const int frag_m = lane & 15;
  const int frag_k8 = (lane >> 4) * 8;
  const int crow0 = (lane >> 4) * 4;
  const int ccol = lane & 15;
  __syncthreads();
  short8v qfrag[NP / 32];
  {
    const int row = wave * 16 + frag_m;
#pragma unroll
    for (int kk = 0; kk < NP / 32; ++kk)
      qfrag[kk] = *reinterpret_cast<const short8v*>(
          reinterpret_cast<char*>(k_s) + row * KROWB +
          swz<KROWB>(row, (kk * 32 + frag_k8) * 2));
  }

  float m[4], l[4], rscale[4], slope[4];
  int qpos[4], klo[4];
  float4v acc_o[PP / 16];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    m[r] = -INFINITY;
    l[r] = 0.0f;
    qpos[r] = HEADS_ROWS ? P0 : P0 + qoff + wave * 16 + crow0 + r;
    rscale[r] = scale * (1.0f + temp_coef * logf((float)((qpos[r] + 1) /
                                                         temp_every) + 1.0f));
    // first visible key of the row: window and position chunk
    klo[r] = window > 0 ? qpos[r] - window + 1 : 0;
    if (chunk > 0) klo[r] = max(klo[r], qpos[r] / chunk * chunk);
    const int head_r =
        HEADS_ROWS ? kvh * rep + min(wave * 16 + crow0 + r, rep - 1)
                   : (int)blockIdx.y;
    slope[r] = slopes ? slopes[head_r] : 0.0f;
  }
#pragma unroll
  for (int nt = 0; nt < PP / 16; ++nt) acc_o[nt] = {0.f, 0.f, 0.f, 0.f};
  const float inv_cap = softcap > 0.0f ? 1.0f / softcap : 0.0f;

  // keys [kfirst, kend): up to the tile's last row, from its first row's
  // window start
  const int kend = HEADS_ROWS ? KVL : min(KVL, P0 + qoff + BM);
  int kfirst = window > 0 ? max(0, P0 + qoff - window + 1) : 0;
  if (chunk > 0) kfirst = max(kfirst, (P0 + qoff) / chunk * chunk);
  kfirst = kfirst / BN * BN;
  // kept first keys: their tiles come first, then the loop jumps to the
  // window
  const int kkept = keep > 0 ? min((keep + BN - 1) / BN * BN, kfirst) : 0;
  const int kbegin = kkept > 0 ? 0 : kfirst;
  auto next_tile = [&](int kb) {
    kb += BN;
    return kb >= kkept && kb < kfirst ? kfirst : kb;
  };

  // the next K/V tile travels in registers while the current one is used
  // (a second tile in flight costs more in occupancy than it hides)
  constexpr int KIT = BN * NP / 8 / 256, VIT = BN * PP / 8 / 256;
  ushort8 kreg[KIT], vreg[VIT];
  auto fetch = [&](int kbase) {
#pragma unroll
    for (int it = 0; it < KIT; ++it) {
      const int idx = tid + it * 256;
      const int row = idx / (NP / 8);
      const int d8 = (idx % (NP / 8)) * 8;
      if (d8 < N) {
        const int gpos = min(kbase + row, KVL - 1);
        const int64_t blk = bt_row[gpos / BS];
        kreg[it] = *reinterpret_cast<const ushort8*>(
            kcache + ((blk * G + kvh) * BS + (gpos % BS)) * N + d8);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) kreg[it].v[e] = 0;
      }
    }
#pragma unroll
    for (int it = 0; it < VIT; ++it) {
      const int idx = tid + it * 256;
      const int key = idx / (PP / 8);
      const int d8 = (idx % (PP / 8)) * 8;
      if (d8 < P) {
        const int gpos = min(kbase + key, KVL - 1);
        const int64_t blk = bt_row[gpos / BS];
        vreg[it] = *reinterpret_cast<const ushort8*>(
            vcache + ((blk * G + kvh) * BS + (gpos % BS)) * P + d8);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) vreg[it].v[e] = 0;
      }
    }
  };
  if (kbegin < kend) fetch(kbegin);

  for (int kbase = kbegin; kbase < kend; kbase = next_tile(kbase)) {
    __syncthreads();
#pragma unroll
    for (int it = 0; it < KIT; ++it) {
      const int idx = tid + it * 256;
      const int row = idx / (NP / 8);
      const int d8 = (idx % (NP / 8)) * 8;
      *reinterpret_cast<ushort8*>(reinterpret_cast<char*>(k_s) + row * KROWB +
                                  swz<KROWB>(row, d8 * 2)) = kreg[it];
    }
#pragma unroll
    for (int it = 0; it < VIT; ++it) {
      const int idx = tid + it * 256;
      const int key = idx / (PP / 8);
      const int d8 = (idx % (PP / 8)) * 8;
#pragma unroll
      for (int e = 0; e < 8; ++e)
        *reinterpret_cast<uint16_t*>(reinterpret_cast<char*>(vt_s) +
                                     (d8 + e) * (BN * 2) +
                                     swz_vt(d8 + e, key * 2)) =
            vreg[it].v[e];
    }
    __syncthreads();
    if (next_tile(kbase) < kend) fetch(next_tile(kbase));
    // a wave none of whose 16 rows exists only helps with the staging
    if (wave * 16 >= nrows) continue;

    float4v acc_s[4];
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) {
      acc_s[nt] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < NP / 32; ++kk) {
        const int krow = nt * 16 + frag_m;
        short8v bfrag = *reinterpret_cast<const short8v*>(
            reinterpret_cast<char*>(k_s) + krow * KROWB +
            swz<KROWB>(krow, (kk * 32 + frag_k8) * 2));
        acc_s[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qfrag[kk], bfrag,
                                                            acc_s[nt], 0, 0, 0);
      }
    }

    float pmax[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int lo = klo[r];
      float mx = -INFINITY;
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) {
        const int kpos = kbase + nt * 16 + ccol;
        float s = acc_s[nt][r] * rscale[r];
        if (softcap > 0.0f) s = softcap * tanh_fast(s * inv_cap);
        s -= slope[r] * (float)(qpos[r] - kpos);
        if (kpos > qpos[r] || kpos >= KVL || (kpos < lo && kpos >= keep))
          s = -INFINITY;
        acc_s[nt][r] = s;
        mx = fmaxf(mx, s);
      }
      pmax[r] = group_reduce_max<16>(mx);
    }
    float alpha[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float mn = fmaxf(m[r], pmax[r]);
      alpha[r] = (m[r] == -INFINITY) ? 0.0f : __expf(m[r] - mn);
      m[r] = mn;
      float rowsum = 0.0f;
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) {
        const float s = acc_s[nt][r];
        const float p = (s == -INFINITY) ? 0.0f : __expf(s - mn);
        rowsum += p;
        const int prow = crow0 + r;
        *reinterpret_cast<uint16_t*>(reinterpret_cast<char*>(pw_s) +
                                     prow * (BN * 2) +
                                     swz<128>(prow, (nt * 16 + ccol) * 2)) =
            f32_to_bf16(p);
      }
      l[r] = l[r] * alpha[r] + group_reduce_sum<16>(rowsum);
    }
#pragma unroll
    for (int nt = 0; nt < PP / 16; ++nt) {
#pragma unroll
      for (int r = 0; r < 4; ++r) acc_o[nt][r] *= alpha[r];
    }
#pragma unroll
    for (int kk2 = 0; kk2 < BN / 32; ++kk2) {
      short8v pfrag = *reinterpret_cast<const short8v*>(
          reinterpret_cast<char*>(pw_s) + frag_m * (BN * 2) +
          swz<128>(frag_m, (kk2 * 32 + frag_k8) * 2));
#pragma unroll
      for (int nt = 0; nt < PP / 16; ++nt) {
        const int vrow = nt * 16 + frag_m;
        short8v vfrag = *reinterpret_cast<const short8v*>(
            reinterpret_cast<char*>(vt_s) + vrow * (BN * 2) +
            swz_vt(vrow, (kk2 * 32 + frag_k8) * 2));
        acc_o[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pfrag, vfrag,
                                                            acc_o[nt], 0, 0, 0);
      }
    }
  }

#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int row = wave * 16 + crow0 + r;
    if (row >= nrows) continue;
    const int64_t tok = HEADS_ROWS ? q0 : q0 + qoff + row;
    const int head = HEADS_ROWS ? kvh * rep + row : blockIdx.y;
    // the sink's term relative to the running maximum (an overflow to
    // infinity gives the right limit, an all-zero row)
    const float lsum = sinks ? l[r] + __expf(sinks[head] - m[r]) : l[r];
    const float inv = 1.0f / lsum;
    uint16_t* o = out + (tok * H + head) * P;
    const uint16_t* gt = gate ? gate + tok * gate_rs + head * gate_w : nullptr;
#pragma unroll
    for (int nt = 0; nt < PP / 16; ++nt) {
      const int c = nt * 16 + ccol;
      if (c < P) {
        float y = acc_o[nt][r] * inv;
        if (gt) y *= sigmoid_fast(bf16_to_f32(gt[gate_w == 1 ? 0 : c]));
        o[c] = f32_to_bf16(y);
      }
    }
  }
}

struct SoftcapArgs {
  uint16_t* out;             // [T, H * P]
  const uint16_t* q;         // [T, H * N], row stride q_rs
  int64_t q_rs;
  const uint16_t *kcache, *vcache;
  const int32_t *block_table, *seq_cu, *seq_start;
  int max_blocks, nprompt, ntiles, H, G, N, P, BS;
  float scale, softcap, temp_coef;
  int temp_every, window, chunk, keep;
  const float *slopes, *sinks;
  const uint16_t* gate;      // [T, H * gate_w], row stride gate_rs
  int64_t gate_rs;
  int gate_w;
};

template <int NP, int PP>
__global__ __launch_bounds__(64 * FT_WAVES, 2) void softcap_prompt_kernel(
    SoftcapArgs a) {
  __shared__ __attribute__((aligned(1024))) uint8_t k_s0[FT_BN * NP * 2];
  __shared__ __attribute__((aligned(1024))) uint8_t k_s1[FT_BN * NP * 2];
  __shared__ __attribute__((aligned(1024))) uint8_t v_s0[FT_BN * PP * 2];
  __shared__ __attribute__((aligned(1024))) uint8_t v_s1[FT_BN * PP * 2];
  const int lane = threadIdx.x & 63, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

  int head, tile, seq, qoff;
  ft_head_and_tile(a.H, a.ntiles, &head, &tile);
  if (!ft_find_tile<FT_BM>(a.seq_cu, a.nprompt, tile, &seq, &qoff)) return;
  const int q0 = a.seq_cu[seq];
  const int Lq = a.seq_cu[seq + 1] - q0;
  const int P0 = a.seq_start[seq];
  const int KVL = P0 + Lq;

  const int row = qoff + wave * 32 + (lane & 31);
  ft_bf16x8 qf[NP / 16];
  const uint16_t* qp = a.q + (int64_t)(q0 + min(row, Lq - 1)) * a.q_rs +
                       (int64_t)head * a.N;
#pragma unroll
  for (int s = 0; s < NP / 16; ++s) {
    const int d = 16 * s + 8 * half;
    ft_bf16x8 f{};
    if (d < a.N) f = *reinterpret_cast<const ft_bf16x8*>(qp + d);
    qf[s] = f;
  }

  auto first_key = [&](int pos) {   // window and position chunk
    int lo = a.window > 0 ? max(0, pos - a.window + 1) : 0;
    return a.chunk > 0 ? max(lo, pos / a.chunk * a.chunk) : lo;
  };
  FlashScore sc{};
  sc.pos = P0 + row;
  sc.lo = first_key(sc.pos);
  sc.keep = a.keep;
  sc.wave_pos = P0 + qoff + wave * 32;
  sc.wave_lo[0] = first_key(sc.wave_pos);
  sc.wave_lo[1] = first_key(sc.wave_pos + 31);
  sc.c = a.scale * FT_LOG2E *
         (1.0f + a.temp_coef *
                     logf((float)((sc.pos + 1) / a.temp_every) + 1.0f));
  sc.cap = a.softcap > 0.0f ? a.softcap * FT_LOG2E : 0.0f;
  sc.slope = a.slopes ? a.slopes[head] * FT_LOG2E : 0.0f;
  FlashSpan span;
  span.kv_len = KVL;
  span.first = first_key(P0 + qoff) / FT_BN * FT_BN;
  span.kept =
      a.keep > 0 ? min((a.keep + FT_BN - 1) / FT_BN * FT_BN, span.first) : 0;
  span.end = min(KVL, P0 + qoff + FT_BM);

  PagedRows rows{a.kcache, a.vcache,
                 a.block_table + (int64_t)seq * a.max_blocks,
                 head / (a.H / a.G), a.G, a.BS, a.N, a.P, KVL};
  ft_f32x16 o[PP / 32];
  float m, l;
  flash_tiles<NP, PP, false>(rows, span, sc, qf, k_s0, k_s1, v_s0, v_s1, o, m,
                             l);
  if (row >= Lq) return;
  // the sink's term relative to the running maximum (an overflow to
  // infinity gives the right limit, an all-zero row)
  if (a.sinks)
    l += __builtin_amdgcn_exp2f(fmaf(a.sinks[head], FT_LOG2E, -m));
  const float inv = 1.0f / l;
  const uint16_t* gt =
      a.gate ? a.gate + (q0 + row) * a.gate_rs + head * a.gate_w : nullptr;
  uint16_t* out = a.out + ((int64_t)(q0 + row) * a.H + head) * a.P;
  if (gt && a.gate_w > 1)
    flash_store<PP>(out, o, a.P, half, [&](int d) {
      return inv * sigmoid_fast(bf16_to_f32(gt[d]));
    });
  else {
    const float f = gt ? inv * sigmoid_fast(bf16_to_f32(gt[0])) : inv;
    flash_store<PP>(out, o, a.P, half, [&](int) { return f; });
  }
}

// Decoded rows: the heads that share a key/value head (32 of them at most per
// workgroup) are the 32 query rows of all four waves, which take a quarter of
// the value dims each; no probabilities are exchanged, and scoring four times
// costs less than HBM takes to deliver the keys.
// ONCE: nontemporal loads, where one workgroup reads a key head's rows (us, eight
// caches in turn, plain and so: 32 heads on 8, 16 of 500 tokens 14.4 and 14.5, of 2000
// 31.2 and 28.1, 48 of 700 to 3500 95.3 and 89.9, 256 of 2048 374 and 335; 32 on 4, the
// last 512 keys, 48 of 2000 19.6 and 18.2).  Of more heads several do, and find them in
// the memory side's cache (64 on 1, 48 of 2000 25.0 and 25.7, 128 of 700 24.6 and 25.6,
// 256 of 2048 79.5 and 80.8).
template <int NP, bool ONCE>
__global__ __launch_bounds__(64 * FT_WAVES, 2) void softcap_decode_kernel(
    SoftcapArgs a, FlashClose close, FlashParts parts) {
  constexpr int PP = 128, VD = PP / FT_WAVES;
  __shared__ __attribute__((aligned(1024))) uint8_t k_s0[FT_BN * NP * 2];
  __shared__ __attribute__((aligned(1024))) uint8_t k_s1[FT_BN * NP * 2];
  __shared__ __attribute__((aligned(1024))) uint8_t v_s0[FT_BN * PP * 2];
  __shared__ __attribute__((aligned(1024))) uint8_t v_s1[FT_BN * PP * 2];
  const int lane = threadIdx.x & 63, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int seq = a.nprompt + blockIdx.x;
  const int rep = a.H / a.G;
  const int kvh = blockIdx.y % a.G;
  const int in_group = blockIdx.y / a.G * 32 + (lane & 31);
  const bool real = in_group < rep;
  const int head = kvh * rep + (real ? in_group : 0);
  const int64_t tok = a.seq_cu[seq];
  const int pos = a.seq_start[seq];

  ft_bf16x8 qf[NP / 16];
  const uint16_t* qp = a.q + tok * a.q_rs + (int64_t)head * a.N;
#pragma unroll
  for (int s = 0; s < NP / 16; ++s) {
    const int d = 16 * s + 8 * half;
    ft_bf16x8 f{};
    if (real && d < a.N) f = *reinterpret_cast<const ft_bf16x8*>(qp + d);
    qf[s] = f;
  }
  FlashScore sc{};
  sc.pos = sc.wave_pos = pos;
  sc.lo = a.window > 0 ? max(0, pos - a.window + 1) : 0;
  if (a.chunk > 0) sc.lo = max(sc.lo, pos / a.chunk * a.chunk);
  sc.wave_lo[0] = sc.wave_lo[1] = sc.lo;
  sc.keep = a.keep;
  sc.c = a.scale * FT_LOG2E *
         (1.0f +
          a.temp_coef * logf((float)((pos + 1) / a.temp_every) + 1.0f));
  sc.cap = a.softcap > 0.0f ? a.softcap * FT_LOG2E : 0.0f;
  sc.slope = a.slopes ? a.slopes[head] * FT_LOG2E : 0.0f;
  FlashSpan span{pos + 1, 0, sc.lo / FT_BN * FT_BN, pos + 1};
  span.kept =
      a.keep > 0 ? min((a.keep + FT_BN - 1) / FT_BN * FT_BN, span.first) : 0;
  span = flash_part(span, blockIdx.z, parts.nsplit);
  PagedRows rows{a.kcache, a.vcache,
                 a.block_table + (int64_t)seq * a.max_blocks, kvh, a.G, a.BS,
                 a.N, a.P, pos + 1};
  ft_f32x16 o[VD / 32];
  float m, l;
  flash_tiles<NP, PP, false, PagedRows, VD, ONCE>(
      rows, span, sc, qf, k_s0, k_s1, v_s0, v_s1, o, m, l, wave * VD);
  if (!real) return;
  if (parts.nsplit > 1) {
    flash_store_part<VD>(parts, (int64_t)blockIdx.x * a.H + head, blockIdx.z,
                         a.P, o, wave * VD, m, l, half);
    return;
  }
  const float inv = 1.0f / close.sum(head, m, l);
  flash_store<VD>(a.out + (tok * a.H + head) * a.P + wave * VD, o,
                  a.P - wave * VD, half, [&](int d) {
                    return inv * close.factor(tok, head, wave * VD + d);
                  });
}

// Decoded rows of keys and values of 128 entries in pages of 16 tokens, up to eight
// heads on a key head: every wave walks pages of its own, two at a time, K to
// registers in whole lines (LineTurn), V by DMA to LDS, both one step ahead, as in
// the engine's own decode attention (csrc/paged_attn_decode.hip, whose walk this
// repeats: what is mended in one is looked for in the other): nothing waits for another wave until the
// end, and 128 KB are under way on a compute unit where the tiles above have 64.
// S^T = K Q^T with the heads in the columns of mfma 16x16x32; the order of its
// rows is the one that V is read in (ds_read_b64_tr_b16), so weights stay in their
// lanes.  The waves' sums meet in LDS once.
//
// Bound by the cache's bytes where there are workgroups for the chip, else by a walk's
// latency.  Measured, the tiles above and this (us, eight caches in turn, 32 heads
// on 8, distance bias and head gate): 48 of 700 to 3500, the last 1024 and the first
// 16 keys, 49.7 and 38.2, all 94.5 and 83.6, of 2000 with a score cap 93.6 and 70.2,
// 128 of 100 to 1000 77.2 and 57.3, 256 of 2048 356 and 336 (6.4 TB/s), 700 of 200
// 178 and 112, one of 3000 15.5 and 13.3, 64 of 20 10.7 and 6.6; 32 on 4, the last
// 512, 48 of 2000 21.0 and 19.2.  Of 2700 mixes of 1 to 600 tokens of 20 to 4000 keys,
// one to eight heads a key head, whole, windowed or in chunks, the tiles are ahead only
// where few parts of 1000 keys are one round (16 of 1000, 40 on 8 20.4 and 21.6; 64 of
// 1000, 16 on 2 21.2 and 22.4).  With 16 on 1, where a page's bytes are a 32nd of
// a workgroup's, they are behind (48 of 2000 21.4 and 22.5).
constexpr int SD_HD = 128, SD_BS = 16, SD_PAGE = SD_HD * SD_BS;

DEVINLINE float sd_quads(float x, bool max) {   // of lanes l, l ^ 16, l ^ 32
  float a = x, b = x;
  asm("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 0" : "+v"(a), "+v"(b));
  x = max ? fmaxf(a, b) : a + b;
  ft_both_halves(x, a, b);
  return max ? fmaxf(a, b) : a + b;
}

DEVINLINE void softcap_pages_body(const SoftcapArgs& a, const FlashClose& close,
                                  const FlashParts& parts) {
  typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
  constexpr int HD = SD_HD, BS = SD_BS, PAGE = SD_PAGE, WAVES = FT_WAVES;
  // two objects, so that reads of one do not wait for loads to the other
  __shared__ __attribute__((aligned(1024))) uint16_t v_s0[WAVES][2 * PAGE];
  __shared__ __attribute__((aligned(1024))) uint16_t v_s1[WAVES][2 * PAGE];
  __shared__ __attribute__((aligned(1024))) u32x4 k_s[WAVES][128];
  __shared__ float m_s[WAVES][16], l_s[WAVES][16];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, quad = lane >> 4;
  const int row = blockIdx.x, seq = a.nprompt + row;
  const int rep = a.H / a.G, kvh = blockIdx.y;
  const int64_t tok = a.seq_cu[seq];
  const int pos = __builtin_amdgcn_readfirstlane(a.seq_start[seq]);

  // visible pages: the kept ones, then from the window's first on; this part's
  int lo = a.window > 0 ? max(0, pos - a.window + 1) : 0;
  if (a.chunk > 0) lo = max(lo, pos / a.chunk * a.chunk);
  const int first = lo / BS;
  const int kept = a.keep > 0 ? min((a.keep + BS - 1) / BS, first) : 0;
  const int pages = kept + pos / BS + 1 - first;
  const int per = ((pages + parts.nsplit - 1) / parts.nsplit + 1) & ~1;
  const int page0 = blockIdx.z * per, page1 = min(page0 + per, pages);
  const int pairs = (page1 - page0 + 1) >> 1;   // wave, wave + WAVES, ...
  auto page_at = [&](int i) FT_INLINE { return i < kept ? i : first + i - kept; };

  // page numbers of this wave's next 32 pairs, one per lane
  const int32_t* table = a.block_table + (int64_t)seq * a.max_blocks;
  int ids = 0;
  auto load_ids = [&](int u) FT_INLINE {
    const int i = page0 + 2 * (u + (lane >> 1) * WAVES) + (lane & 1);
    ids = table[page_at(min(i, page1 - 1))];
    __builtin_amdgcn_s_waitcnt(0x0f70);   // here, not at every use
  };
  if (wave < pairs) load_ids(wave);

  // the heads as columns, dims 32 kk + 8 quad ..; past the last the first one's
  const int head = kvh * rep + (r16 < rep ? r16 : 0);
  ft_bf16x8 qf[4];
  const uint16_t* qp = a.q + tok * a.q_rs + (int64_t)head * HD + quad * 8;
#pragma unroll
  for (int kk = 0; kk < 4; ++kk)
    qf[kk] = *reinterpret_cast<const ft_bf16x8*>(qp + kk * 32);
  const float c =
      a.scale * FT_LOG2E *
      (1.0f + a.temp_coef * logf((float)((pos + 1) / a.temp_every) + 1.0f));
  const float cap = a.softcap > 0.0f ? a.softcap * FT_LOG2E : 0.0f;
  // tanh by exp2: cap - 2 cap / (1 + 2^(cap_k s))
  const float cap_k = cap > 0.0f ? 2.0f * FT_LOG2E * c / cap : 0.0f;
  const float slope = a.slopes ? a.slopes[head] * FT_LOG2E : 0.0f;

  // lane offsets into a page, bytes: K half a row of eight rows a load; V four rows
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
    u32x4 k[2][4];
  };
  typedef __attribute__((address_space(3))) void lds_void;
  // pair u; rows past the part's end or the row's position read as zeros
  auto fetch = [&](int u, Keys& K, uint16_t* vs) FT_INLINE {
    const int at = (u - wave) / WAVES;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int i = page0 + 2 * u + h;
      const int64_t id = __builtin_amdgcn_readlane(ids, (at & 31) * 2 + h);
      const int64_t base = (id * a.G + kvh) * PAGE;
      const int rows = __builtin_amdgcn_readfirstlane(
          i < page1 ? max(0, min(BS, pos + 1 - page_at(i) * BS)) : 0);
      const auto kr = __builtin_amdgcn_make_buffer_rsrc(
          (void*)(a.kcache + base), 0, rows * HD * 2, 0x00020000);
      const auto vr = __builtin_amdgcn_make_buffer_rsrc(
          (void*)(a.vcache + base), 0, rows * HD * 2, 0x00020000);
#pragma unroll
      for (int kk = 0; kk < 4; ++kk)
        K.k[h][kk] = __builtin_amdgcn_raw_buffer_load_b128(
            kr, kx + (kk >> 1) * 128 + (kk & 1) * 8 * HD * 2, 0, 2);
#pragma unroll
      for (int j = 0; j < 4; ++j)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            vr, (lds_void*)(vs + h * PAGE + j * 512), 16, vx[j], 0, 0, 2);
    }
  };

  // O^T: column r16, dims 16 d + 4 quad ..; m in log2, l of this lane's tokens
  typedef __attribute__((ext_vector_type(4))) float f32x4;
  f32x4 acc[8];
#pragma unroll
  for (int d = 0; d < 8; ++d) acc[d] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  float m = -INFINITY, l = 0.0f;
  // V's rows as operands: dims 16 d + r16, tokens 4 quad ..
  const int vrow = 4 * quad + (r16 >> 2);
  const int vat = vrow * HD + ((r16 & 3) >> 1) * 8 + (r16 & 1) * 4;
  auto use = [&](int u, const Keys& K, uint16_t* vs) FT_INLINE {
    f32x4 s[2];
    u32x4 kf[2][4];
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        turn(k_s[wave], K.k[h][2 * e], K.k[h][2 * e + 1], kf[h][2 * e],
             kf[h][2 * e + 1]);
#pragma unroll
    for (int h = 0; h < 2; ++h) s[h] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int kk = 0; kk < 4; ++kk)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        s[h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            __builtin_bit_cast(ft_bf16x8, kf[h][kk]), qf[kk], s[h], 0, 0, 0);
    // token 4 quad + j % 4 of page j / 4
    float t[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) t[j] = s[j >> 2][j & 3];
    if (cap > 0.0f) {
#pragma unroll
      for (int j = 0; j < 8; ++j)
        t[j] = fmaf(-2.0f * cap,
                    __builtin_amdgcn_rcpf(
                        1.0f + __builtin_amdgcn_exp2f(t[j] * cap_k)),
                    cap);
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) t[j] *= c;
    }
    const int i = page0 + 2 * u;
    const int key0 = page_at(i) * BS, key1 = page_at(i + 1) * BS;
#pragma unroll
    for (int j = 0; j < 8; ++j)
      t[j] = fmaf((float)((j < 4 ? key0 : key1) + 4 * quad + (j & 3) - pos),
                  slope, t[j]);
    if (i + 1 >= page1 || key1 + BS > pos + 1 || key0 < lo || key1 < lo) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int key = (j < 4 ? key0 : key1) + 4 * quad + (j & 3);
        if ((j >= 4 && i + 1 >= page1) || key > pos ||
            (key < lo && key >= a.keep))
          t[j] = -INFINITY;
      }
    }
    float mx = t[0];
#pragma unroll
    for (int j = 1; j < 8; ++j) mx = fmaxf(mx, t[j]);
    mx = sd_quads(mx, true);
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
    for (int j = 0; j < 8; ++j) p[j] = __builtin_amdgcn_exp2f(t[j] - mc);
    l += ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
    union {
      uint32_t u[4];
      ft_bf16x8 v;
    } w;
#pragma unroll
    for (int e = 0; e < 4; ++e) w.u[e] = ft_pack_bf16(p[2 * e], p[2 * e + 1]);
    typedef __attribute__((address_space(3))) ft_short4 lds_short4;
#pragma unroll
    for (int d = 0; d < 8; ++d) {
      union {
        ft_short4 h[2];
        ft_bf16x8 v;
      } vf;
#pragma unroll
      for (int h = 0; h < 2; ++h)
        vf.h[h] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (lds_short4*)(vs + h * PAGE + vat + ((d ^ (vrow & 7)) << 4)));
      acc[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf.v, w.v, acc[d], 0, 0,
                                                       0);
    }
  };

  Keys k0, k1;
  auto ahead = [&](int u, Keys& K, uint16_t* vs) FT_INLINE {
    if ((((u - wave) / WAVES) & 31) == 0 && u < pairs) load_ids(u);
    fetch(u, K, vs);
  };
  if (wave < pairs) {
    fetch(wave, k0, v_s0[wave]);
    for (int u = wave;; u += 2 * WAVES) {
      ahead(u + WAVES, k1, v_s1[wave]);
      use(u, k0, v_s0[wave]);
      if (u + WAVES >= pairs) break;
      ahead(u + 2 * WAVES, k0, v_s0[wave]);
      use(u + WAVES, k1, v_s1[wave]);
      if (u + 2 * WAVES >= pairs) break;
    }
  }
  l = sd_quads(l, false);

  // the waves' sums meet in the memory of the V tiles (loads that are still
  // under way there read nothing, and are waited for first)
  float* sums = reinterpret_cast<float*>(&v_s0[0][0]);   // [WAVES][16][HD]
  static_assert(sizeof(v_s0) == WAVES * 16 * HD * sizeof(float));
  __builtin_amdgcn_s_waitcnt(0x0f70);
  __syncthreads();
  if (quad == 0) {
    m_s[wave][r16] = m;
    l_s[wave][r16] = l;
  }
  if (r16 < rep) {
#pragma unroll
    for (int d = 0; d < 8; ++d)
      *reinterpret_cast<f32x4*>(sums + (wave * 16 + r16) * HD + d * 16 +
                                quad * 4) = acc[d];
  }
  __syncthreads();
  for (int i = tid; i < rep * (HD / 4); i += 64 * WAVES) {
    const int j = i / (HD / 4), d = i % (HD / 4) * 4;
    float M = m_s[0][j], L = 0.0f;
#pragma unroll
    for (int w = 1; w < WAVES; ++w) M = fmaxf(M, m_s[w][j]);
    float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      const float f = m_s[w][j] == -INFINITY
                          ? 0.0f
                          : __builtin_amdgcn_exp2f(m_s[w][j] - M);
      const float4 x =
          *reinterpret_cast<const float4*>(sums + (w * 16 + j) * HD + d);
      L = fmaf(f, l_s[w][j], L);
      o.x = fmaf(f, x.x, o.x);
      o.y = fmaf(f, x.y, o.y);
      o.z = fmaf(f, x.z, o.z);
      o.w = fmaf(f, x.w, o.w);
    }
    const int at = kvh * rep + j;
    if (parts.nsplit > 1) {
      const int64_t slot =
          ((int64_t)row * a.H + at) * parts.nsplit + blockIdx.z;
      *reinterpret_cast<float4*>(parts.o + slot * HD + d) = o;
      if (d == 0) {
        parts.ml[2 * slot] = M;
        parts.ml[2 * slot + 1] = L;
      }
    } else {
      const float inv = 1.0f / close.sum(at, M, L);
      uint2 y;
      y.x = ft_pack_bf16(o.x * (inv * close.factor(tok, at, d)),
                         o.y * (inv * close.factor(tok, at, d + 1)));
      y.y = ft_pack_bf16(o.z * (inv * close.factor(tok, at, d + 2)),
                         o.w * (inv * close.factor(tok, at, d + 3)));
      *reinterpret_cast<uint2*>(a.out + (tok * a.H + at) * HD + d) = y;
    }
  }
}

__global__ __launch_bounds__(64 * FT_WAVES, 2) void softcap_pages_kernel(
    SoftcapArgs a, FlashClose close, FlashParts parts) {
  softcap_pages_body(a, close, parts);
}

// prompt_rows: row counts of the first sequences of the batch; the other
// sequences bring one decoded row each.  Returns false when the sizes do not
// fit the tile kernels.
bool softcap_attention_mfma(torch::Tensor out, torch::Tensor q,
                            torch::Tensor kcache, torch::Tensor vcache,
                            torch::Tensor block_table, torch::Tensor seq_cu,
                            torch::Tensor seq_start,
                            std::vector<int64_t> prompt_rows, double scale,
                            double softcap, double temp_coef,
                            int64_t temp_every, int64_t window,
                            c10::optional<torch::Tensor> slopes,
                            int64_t chunk, c10::optional<torch::Tensor> sinks,
                            c10::optional<torch::Tensor> gate, int64_t keep) {
  TORCH_CHECK(q.is_cuda() && q.dim() == 2 && q.stride(1) == 1);
  if (q.scalar_type() != torch::kBFloat16) return false;
  TORCH_CHECK(kcache.is_contiguous() && kcache.dim() == 4 &&
              vcache.is_contiguous() && vcache.dim() == 4 &&
              kcache.dtype() == q.dtype() && vcache.dtype() == q.dtype());
  const int T = q.size(0), G = kcache.size(1), BS = kcache.size(2);
  const int N = kcache.size(3), P = vcache.size(3);
  TORCH_CHECK(q.size(1) % N == 0);
  const int H = q.size(1) / N;
  TORCH_CHECK(H % G == 0 && vcache.size(0) == kcache.size(0) &&
              vcache.size(1) == G && vcache.size(2) == BS);
  const int S = seq_start.numel(), nprompt = prompt_rows.size();
  TORCH_CHECK(nprompt <= S);
  const int ndec = S - nprompt;
  if (N % 8 || P % 8 || N > 128 || P > 256 || q.stride(0) % 8 ||
      (reinterpret_cast<uintptr_t>(q.data_ptr()) & 15) ||
      (reinterpret_cast<uintptr_t>(kcache.data_ptr()) & 15) ||
      (reinterpret_cast<uintptr_t>(vcache.data_ptr()) & 15) ||
      (ndec > 0 && H / G > SA_BM))
    return false;
  TORCH_CHECK(out.is_contiguous() && out.dtype() == q.dtype() &&
              out.numel() == (int64_t)T * H * P);
  TORCH_CHECK(block_table.dtype() == torch::kInt32 &&
              block_table.is_contiguous() && block_table.dim() == 2);
  TORCH_CHECK(seq_cu.dtype() == torch::kInt32 && seq_cu.numel() == S + 1 &&
              seq_start.dtype() == torch::kInt32 && block_table.size(0) >= S);
  TORCH_CHECK(temp_every >= 1 && chunk >= 0 && keep >= 0);
  if (slopes.has_value())
    TORCH_CHECK(slopes->dtype() == torch::kFloat32 &&
                slopes->is_contiguous() && slopes->numel() == H);
  if (sinks.has_value())
    TORCH_CHECK(sinks->dtype() == torch::kFloat32 && sinks->is_contiguous() &&
                sinks->numel() == H);
  if (gate.has_value())
    TORCH_CHECK(gate->dtype() == q.dtype() && gate->dim() == 2 &&
                gate->stride(1) == 1 && gate->size(0) == T &&
                (gate->size(1) == (int64_t)H * P || gate->size(1) == H));
  const int gate_w = gate.has_value() ? (int)(gate->size(1) / H) : 1;
  hipStream_t stream = at::cuda::getCurrentCUDAStream();
  auto tiles = [&](int bm) {
    int64_t n = 0;
    for (int64_t len : prompt_rows) n += (len + bm - 1) / bm;
    return n;
  };
  SoftcapArgs a{(uint16_t*)out.data_ptr(), (const uint16_t*)q.data_ptr(),
                q.stride(0), (const uint16_t*)kcache.data_ptr(),
                (const uint16_t*)vcache.data_ptr(),
                (const int32_t*)block_table.data_ptr(),
                (const int32_t*)seq_cu.data_ptr(),
                (const int32_t*)seq_start.data_ptr(),
                (int)block_table.size(1), nprompt, (int)tiles(FT_BM), H, G, N,
                P, BS, (float)scale, (float)softcap, (float)temp_coef,
                (int)temp_every, (int)window, (int)chunk, (int)keep,
                slopes.has_value() ? (const float*)slopes->data_ptr() : nullptr,
                sinks.has_value() ? (const float*)sinks->data_ptr() : nullptr,
                gate.has_value() ? (const uint16_t*)gate->data_ptr() : nullptr,
                gate.has_value() ? (int64_t)gate->stride(0) : 0, gate_w};
#define LAUNCH_SP(NPV, PPV)                                                   \
  hipLaunchKernelGGL((softcap_prompt_kernel<NPV, PPV>),                       \
                     dim3((int64_t)a.ntiles * H), dim3(64 * FT_WAVES), 0,     \
                     stream, a)
#define LAUNCH_SA(NPV, PPV, HR, GRID)                                         \
  hipLaunchKernelGGL(                                                         \
      (softcap_attention_mfma_kernel<NPV, PPV, HR>), GRID, dim3(256), 0,      \
      stream, a.out, a.q, a.q_rs, a.kcache, a.vcache, a.block_table,          \
      a.max_blocks, a.seq_cu, a.seq_start, nprompt, H, G, N, P, BS, a.scale,  \
      a.softcap, a.temp_coef, a.temp_every, a.window, a.slopes, a.chunk,      \
      a.keep, a.sinks, a.gate, a.gate_rs, gate_w)
  if (a.ntiles > 0) {
    if (N <= 64 && P <= 64) LAUNCH_SP(64, 64);
    else if (N <= 64 && P <= 128) LAUNCH_SP(64, 128);
    else if (P <= 64) LAUNCH_SP(128, 64);
    else if (P <= 128) LAUNCH_SP(128, 128);
    else if (N <= 64) LAUNCH_SA(64, 256, false, dim3(tiles(SA_BM), H));
    else LAUNCH_SA(128, 256, false, dim3(tiles(SA_BM), H));
    HIP_CHECK_KERNEL();
  }
  if (ndec > 0 && P <= 128) {
    const int64_t groups = (int64_t)G * ((H / G + 31) / 32);
    // two workgroups per compute unit; a part has at least four tiles of the
    // longest context that the block table holds
    const int64_t cus =
        at::cuda::getCurrentDeviceProperties()->multiProcessorCount;
    const int64_t longest = (int64_t)a.max_blocks * BS;
    const int64_t keys =
        window > 0 ? std::min<int64_t>(longest, window + keep) : longest;
    const int64_t nsplit = std::max<int64_t>(
        1, std::min<int64_t>({32, 2 * cus / std::max<int64_t>(1, ndec * groups),
                              keys / (4 * FT_BN)}));
    const FlashClose close{a.out, H, P, a.sinks, nullptr, a.gate, a.gate_rs,
                           gate_w};
    FlashParts parts{nullptr, nullptr, (int)nsplit};
    torch::Tensor part;
    if (nsplit > 1) {
      const int64_t slots = (int64_t)ndec * H * nsplit;
      part = torch::empty({slots * (P + 2)},
                          q.options().dtype(torch::kFloat32));
      parts.o = part.data_ptr<float>();
      parts.ml = parts.o + slots * P;
    }
    const dim3 grid(ndec, groups, nsplit), block(64 * FT_WAVES);
    const bool once = H / G <= 32;
    const bool in_pages = N == SD_HD && P == SD_HD && BS == SD_BS && H / G <= 8;
    auto* kern = in_pages  ? softcap_pages_kernel
                 : N <= 64 ? once ? softcap_decode_kernel<64, true>
                                  : softcap_decode_kernel<64, false>
                 : once    ? softcap_decode_kernel<128, true>
                           : softcap_decode_kernel<128, false>;
    hipLaunchKernelGGL(kern, grid, block, 0, stream, a, close, parts);
    HIP_CHECK_KERNEL();
    if (nsplit > 1) {
      hipLaunchKernelGGL(flash_merge_kernel, dim3((int64_t)ndec * H),
                         dim3(P / 4), 0, stream, close, parts,
                         a.seq_cu + nprompt);
      HIP_CHECK_KERNEL();
    }
  } else if (ndec > 0) {
    if (N <= 64) LAUNCH_SA(64, 256, true, dim3(ndec, G));
    else LAUNCH_SA(128, 256, true, dim3(ndec, G));
    HIP_CHECK_KERNEL();
  }
#undef LAUNCH_SA
#undef LAUNCH_SP
  return true;
}

}  // namespace igw
