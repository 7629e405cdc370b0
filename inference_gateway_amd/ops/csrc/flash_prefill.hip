// Varlen causal flash attention for prompt rows, gfx950 (MI355X), bf16.
//
// One kernel, two sources of keys and values: the freshly projected dense
// K/V of whole prompts (flash_prefill), or the paged cache (flash_prefill_
// paged: chunked prefill and prefix reuse, where the q rows are a chunk
// behind `prefix` cached tokens and row r sits at position prefix + r; the
// chunk's own keys are already appended).
//
// What bounds it: per score two MFMA multiply-adds over 128 dims, and on the
// vector units one max, one multiply-add, one exponential (quarter rate), one
// add and half a conversion, about as many cycles as the MFMAs take.  The
// design keeps everything else off those two units:
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
//   * K and V tiles go from global memory straight to LDS, the tile after
//     next being fetched while this one is used: two buffers, one barrier a
//     tile, four LDS objects so that the reads of one buffer do not wait for
//     the writes to the other;
//   * 16-byte chunks are XOR-swizzled by row (on the global side, a DMA
//     writes LDS linearly): K by row & 15, V by the two row fields that the
//     transposing read spreads over lanes, both free of bank conflicts;
//   * the running maximum is raised, and the accumulators rescaled, only
//     when a row outgrows it by more than 2^8 (exact: every term carries
//     the same factor, which the division by the sum takes out again);
//   * masks are evaluated only in tiles that reach past a wave's first row,
//     and a wave skips tiles past its last row.
//
// Two waves per SIMD (256 registers, 64 KB of LDS per workgroup) let one
// wave's softmax run beside the other's MFMAs.  Measured with 32 heads on 8:
// one prompt of 16000 tokens 2065 us, 1016 TFLOP/s (64 x 64 tiles of
// 16x16x32 MFMAs with V transposed by the stores and P through LDS: 12518
// us); 16 prompts of 512 72 us (416); 2000 rows behind 6000 cached ones 281
// us, 816 TFLOP/s (1552).  GQA heads that share keys run
// on one XCD: workgroup ids go round-robin over the 8 XCDs, so heads are
// dealt to id % 8 and the tiles of a head follow each other there, the
// longest (last) tiles of each prompt first.

#include <ATen/cuda/CUDAContext.h>
#include <torch/extension.h>

#include "common.h"

namespace igw {

typedef __attribute__((ext_vector_type(4))) short fp_short4;
typedef __attribute__((ext_vector_type(8))) short fp_short8;
typedef __attribute__((ext_vector_type(8))) __bf16 fp_bf16x8;
typedef __attribute__((ext_vector_type(16))) float fp_f32x16;

constexpr int FP_HD = 128;   // head dim
constexpr int FP_BN = 64;    // keys per tile
constexpr int FP_WAVES = 4;  // waves per workgroup, 32 query rows each
constexpr int FP_BM = 32 * FP_WAVES;
constexpr int FP_PAGE = 16;  // tokens per cache page

// two floats -> packed bf16 pair, round to nearest even
DEVINLINE uint32_t fp_pack_bf16(float a, float b) {
  typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2_t;
  typedef __attribute__((ext_vector_type(2))) float f32x2_t;
  const f32x2_t v = {a, b};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
}

// x of lane i and of lane i ^ 32, in both lanes: a = lower half's value, b =
// upper half's.  Written out because the compiler folds the builtin's two
// results into one when its operands are equal; the s_nop is the wait that
// the swap needs behind the instruction that wrote its operands.
DEVINLINE void fp_both_halves(float x, float& a, float& b) {
  a = b = x;
  asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 0" : "+v"(a), "+v"(b));
}

struct FlashArgs {
  uint16_t* out;              // [T, NQ, HD]
  const uint16_t* q;          // [T, NQ, HD], row stride q_rs
  const uint16_t* k;          // dense [T, NKV, HD] or pages
  const uint16_t* v;
  const int32_t* block_table; // paged only: [B, max_blocks]
  const int32_t* prefix;      // paged only: [B]
  const int32_t* cu;          // [B + 1]
  int64_t q_rs, k_rs, v_rs;
  int B, ntiles, nq, nkv, max_blocks;
  float scale;
};

// Sequence and row offset of tile `t` when every sequence of cu takes
// ceil(rows / BM) tiles (found here: a tile map made on the host costs two
// copies that wait for the stream).  One step per 64 sequences; false when
// there is no such tile.
DEVINLINE bool fp_find_tile(const FlashArgs& a, int t, int* seq, int* off) {
  const int lane = threadIdx.x & 63;
  int before = 0;
  for (int base = 0; base < a.B; base += 64) {
    const int i = base + lane;
    const int n = i < a.B ? (a.cu[i + 1] - a.cu[i] + FP_BM - 1) / FP_BM : 0;
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
          (t - before - __shfl(sum - n, w, 64)) * FP_BM);
      return true;
    }
    before += __builtin_amdgcn_readfirstlane(__shfl(sum, 63, 64));
  }
  return false;
}

template <bool PAGED>
__global__ __launch_bounds__(64 * FP_WAVES, 2) void flash_prefill_kernel(
    FlashArgs a) {
  constexpr int HD = FP_HD, BN = FP_BN, BM = FP_BM;
  // [64 keys][16 chunks of 16 bytes], chunks swizzled per row
  __shared__ __attribute__((aligned(1024))) uint8_t k_s0[BN * HD * 2];
  __shared__ __attribute__((aligned(1024))) uint8_t k_s1[BN * HD * 2];
  __shared__ __attribute__((aligned(1024))) uint8_t v_s0[BN * HD * 2];
  __shared__ __attribute__((aligned(1024))) uint8_t v_s1[BN * HD * 2];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int half = lane >> 5;
  const int col = lane & 31;

  // heads dealt to XCDs (a multiple of 8 heads), longest tiles first
  int qh, tile;
  if (a.nq % 8 == 0) {
    const int hp = a.nq >> 3, local = blockIdx.x >> 3;
    qh = (blockIdx.x & 7) * hp + local % hp;
    tile = local / hp;
  } else {
    qh = blockIdx.x % a.nq;
    tile = blockIdx.x / a.nq;
  }
  int seq, qoff;
  if (!fp_find_tile(a, a.ntiles - 1 - tile, &seq, &qoff)) return;
  const int kvh = qh / (a.nq / a.nkv);
  const int q0 = a.cu[seq];
  const int Lq = a.cu[seq + 1] - q0;
  const int P = PAGED ? a.prefix[seq] : 0;
  const int KVL = P + Lq;
  const int32_t* bt = PAGED ? a.block_table + (int64_t)seq * a.max_blocks
                            : nullptr;

  // ---- Q: B operand, this lane's query row, dims 16 s + 8 half .. + 7 ----
  const int row = qoff + wave * 32 + col;  // row within the sequence
  const int qpos = P + row;
  fp_bf16x8 qf[HD / 16];
  {
    const uint16_t* qp = a.q + (int64_t)(q0 + min(row, Lq - 1)) * a.q_rs +
                         (int64_t)qh * HD + 8 * half;
#pragma unroll
    for (int s = 0; s < HD / 16; ++s)
      qf[s] = *reinterpret_cast<const fp_bf16x8*>(qp + 16 * s);
    // the running maximum is of raw scores: a negative scale turns q round
    if (a.scale < 0.0f) {
#pragma unroll
      for (int s = 0; s < HD / 16; ++s) qf[s] = -qf[s];
    }
  }

  // ---- staging: wave w moves rows RW w .. of the tile, 4 rows a load ----
  constexpr int RW = BN / FP_WAVES;
  const int sub = lane >> 4;  // row within a load
  // the wave's pages of the tile to be staged next: their numbers are
  // requested one tile ahead
  int page[PAGED ? RW / FP_PAGE : 1];
  auto next_pages = [&](int kbase) {
#pragma unroll
    for (int g = 0; g < RW / FP_PAGE; ++g)
      page[g] = bt[min((kbase + wave * RW) / FP_PAGE + g,
                       (KVL - 1) / FP_PAGE)];
  };
  auto stage = [&](int kbase, uint8_t* kd, uint8_t* vd) {
#pragma unroll
    for (int p = 0; p < RW / 4; ++p) {
      const int r0 = wave * RW + 4 * p;       // tile row of lane 0
      const int r = r0 + sub;
      const int kc = ((lane & 15) ^ (r & 15)) * 8;
      const int vc = ((lane & 15) ^ ((sub << 2) | (p & 3))) * 8;
      const uint16_t *ks, *vs;
      if (PAGED) {
        // rows past the last key repeat it (they are masked)
        const int last = KVL - 1 - (kbase + wave * RW + (p >> 2) * FP_PAGE);
        const int in_page = min(4 * (p & 3) + sub,
                                last >= 0 ? last : (KVL - 1) % FP_PAGE);
        const int64_t base =
            ((int64_t)page[p >> 2] * a.nkv + kvh) * (FP_PAGE * HD) +
            in_page * HD;
        ks = a.k + base + kc;
        vs = a.v + base + vc;
      } else {
        const int64_t tok = q0 + min(kbase + r, KVL - 1);
        ks = a.k + tok * a.k_rs + kvh * HD + kc;
        vs = a.v + tok * a.v_rs + kvh * HD + vc;
      }
      __builtin_amdgcn_global_load_lds(
          reinterpret_cast<const uint32_t*>(ks),
          reinterpret_cast<uint32_t*>(kd + r0 * HD * 2), 16, 0, 0);
      __builtin_amdgcn_global_load_lds(
          reinterpret_cast<const uint32_t*>(vs),
          reinterpret_cast<uint32_t*>(vd + r0 * HD * 2), 16, 0, 0);
    }
    if (PAGED) next_pages(kbase + BN);
  };

  // ---- LDS offsets of this lane's fragments ----
  int koff[HD / 16];  // K row `col` (+ 32 per sub-tile), dims 16 s + 8 half
#pragma unroll
  for (int s = 0; s < HD / 16; ++s)
    koff[s] = col * (HD * 2) + (((2 * s + half) ^ (col & 15)) << 4);
  int voff[HD / 32][2];  // V^T: dims 32 dt + 16 (lane bit 4), keys 4 half + 8 e
#pragma unroll
  for (int dt = 0; dt < HD / 32; ++dt)
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int i = lane & 15, r = 4 * half + 8 * e + (i >> 2);
      const int c = 4 * dt + 2 * ((lane >> 4) & 1) + ((i & 3) >> 1);
      voff[dt][e] = r * (HD * 2) +
                    ((c ^ (((r & 3) << 2) | ((r >> 2) & 3))) << 4) +
                    8 * (i & 1);
    }

  // scores in log2; not 0, so that a masked score stays -inf
  const float c = fmaxf(fabsf(a.scale) * 1.44269504088896340736f, 1e-37f);
  float m = -INFINITY;  // running maximum of the raw scores, this lane's row
  float l = 0.0f;       // sum over this lane half's keys
  fp_f32x16 o[HD / 32];
#pragma unroll
  for (int dt = 0; dt < HD / 32; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[dt][i] = 0.0f;

  const int first_pos = P + qoff + wave * 32;  // of the wave's rows
  const int kend = min(KVL, P + qoff + BM);
  const int nkt = (kend + BN - 1) / BN;

  auto step = [&](int kt, uint8_t* kb, uint8_t* vb, uint8_t* kn,
                  uint8_t* vn) {
    const int kbase = kt * BN;
    // this wave's loads of the tile have arrived; behind the barrier all
    // have, and nobody reads the other buffer any more
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (kt + 1 < nkt) stage(kbase + BN, kn, vn);
    if (kbase > first_pos + 31) return;  // past the wave's last row

    fp_f32x16 s[2];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) s[t][i] = 0.0f;
#pragma unroll
    for (int d = 0; d < HD / 16; ++d)
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const fp_bf16x8 kf = *reinterpret_cast<const fp_bf16x8*>(
            kb + koff[d] + t * 32 * HD * 2);
        s[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[d], s[t], 0, 0,
                                                       0);
      }

    if (kbase + BN - 1 > first_pos) {
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int kpos = kbase + 32 * t + (i & 3) + 8 * (i >> 2) + 4 * half;
          if (kpos > qpos || kpos >= KVL) s[t][i] = -INFINITY;
        }
    }

    float mx = s[0][0];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[t][i]);
    {
      float lo, hi;
      fp_both_halves(mx, lo, hi);
      mx = fmaxf(lo, hi);
    }
    // mx <= m + 8 for all rows of the wave: keep the old maximum
    if (__any((mx - m) * c > 8.0f)) {
      const float mn = fmaxf(m, mx);
      const float alpha = __builtin_amdgcn_exp2f((m - mn) * c);
      m = mn;
      l *= alpha;
#pragma unroll
      for (int dt = 0; dt < HD / 32; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[dt][i] *= alpha;
    }
    const float mc = m == -INFINITY ? 0.0f : m * c;
    float sum = 0.0f;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float p = __builtin_amdgcn_exp2f(fmaf(s[t][i], c, -mc));
        s[t][i] = p;
        sum += p;
      }
    l += sum;

#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        union {
          uint32_t u[4];
          fp_bf16x8 v;
        } pf;
#pragma unroll
        for (int e = 0; e < 4; ++e)
          pf.u[e] = fp_pack_bf16(s[t][8 * ks + 2 * e],
                                 s[t][8 * ks + 2 * e + 1]);
#pragma unroll
        for (int dt = 0; dt < HD / 32; ++dt) {
          typedef __attribute__((address_space(3))) fp_short4 lds_short4;
          union {
            fp_short4 h[2];
            fp_bf16x8 v;
          } vf;
#pragma unroll
          for (int e = 0; e < 2; ++e)
            vf.h[e] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (lds_short4*)(vb + voff[dt][e] + (32 * t + 16 * ks) * HD * 2));
          o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf.v, pf.v, o[dt],
                                                          0, 0, 0);
        }
      }
  };

  if (PAGED) next_pages(0);
  stage(0, k_s0, v_s0);
  for (int kt = 0; kt < nkt; kt += 2) {
    step(kt, k_s0, v_s0, k_s1, v_s1);
    if (kt + 1 < nkt) step(kt + 1, k_s1, v_s1, k_s0, v_s0);
  }

  // ---- both halves' sums, normalise, store 4 dims at a time ----
  {
    float lo, hi;
    fp_both_halves(l, lo, hi);
    l = lo + hi;
  }
  if (row < Lq) {
    const float inv = 1.0f / l;
    uint16_t* op = a.out + ((int64_t)(q0 + row) * a.nq + qh) * HD + 4 * half;
#pragma unroll
    for (int dt = 0; dt < HD / 32; ++dt)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        uint2 w;
        w.x = fp_pack_bf16(o[dt][4 * g] * inv, o[dt][4 * g + 1] * inv);
        w.y = fp_pack_bf16(o[dt][4 * g + 2] * inv, o[dt][4 * g + 3] * inv);
        *reinterpret_cast<uint2*>(op + 32 * dt + 8 * g) = w;
      }
  }
}

template <bool PAGED>
static void flash_launch(FlashArgs& a, const std::vector<int64_t>& seq_lens,
                         hipStream_t stream) {
  int64_t tiles = 0;
  for (int64_t len : seq_lens) tiles += (len + FP_BM - 1) / FP_BM;
  if (tiles == 0) return;
  a.ntiles = (int)tiles;
  hipLaunchKernelGGL((flash_prefill_kernel<PAGED>), dim3(tiles * a.nq),
                     dim3(64 * FP_WAVES), 0, stream, a);
  HIP_CHECK_KERNEL();
}

static void flash_check(const torch::Tensor& out, const torch::Tensor& q,
                        const torch::Tensor& cu_seqlens,
                        const std::vector<int64_t>& seq_lens, int64_t nkv) {
  TORCH_CHECK(q.is_cuda() && q.dtype() == torch::kBFloat16 && q.dim() == 3);
  TORCH_CHECK(q.stride(2) == 1 && q.stride(1) == q.size(2));
  TORCH_CHECK(out.is_contiguous() && out.sizes() == q.sizes() &&
              out.dtype() == q.dtype());
  TORCH_CHECK(cu_seqlens.dtype() == torch::kInt32 &&
              cu_seqlens.is_contiguous() &&
              cu_seqlens.numel() > (int64_t)seq_lens.size());
  TORCH_CHECK(q.size(2) == FP_HD, "only head_dim=128 supported");
  TORCH_CHECK(nkv > 0 && q.size(1) % nkv == 0);
}

void flash_prefill_paged(torch::Tensor out, torch::Tensor q,
                         torch::Tensor kcache, torch::Tensor vcache,
                         torch::Tensor block_table, torch::Tensor prefix_lens,
                         torch::Tensor cu_seqlens,
                         std::vector<int64_t> seq_lens, double scale) {
  TORCH_CHECK(kcache.is_contiguous() && vcache.is_contiguous() &&
              kcache.dtype() == q.dtype() && vcache.dtype() == q.dtype());
  TORCH_CHECK(block_table.dtype() == torch::kInt32 &&
              block_table.is_contiguous());
  TORCH_CHECK(prefix_lens.dtype() == torch::kInt32);
  TORCH_CHECK(kcache.size(2) == FP_PAGE, "cache block size must be 16");
  flash_check(out, q, cu_seqlens, seq_lens, kcache.size(1));
  FlashArgs a{};
  a.out = (uint16_t*)out.data_ptr();
  a.q = (const uint16_t*)q.data_ptr();
  a.k = (const uint16_t*)kcache.data_ptr();
  a.v = (const uint16_t*)vcache.data_ptr();
  a.block_table = (const int32_t*)block_table.data_ptr();
  a.prefix = (const int32_t*)prefix_lens.data_ptr();
  a.cu = (const int32_t*)cu_seqlens.data_ptr();
  a.q_rs = q.stride(0);
  a.B = (int)seq_lens.size();
  a.nq = q.size(1);
  a.nkv = kcache.size(1);
  a.max_blocks = block_table.size(1);
  a.scale = (float)scale;
  flash_launch<true>(a, seq_lens, at::cuda::getCurrentCUDAStream());
}

void flash_prefill(torch::Tensor out, torch::Tensor q, torch::Tensor k,
                   torch::Tensor v, torch::Tensor cu_seqlens,
                   std::vector<int64_t> seq_lens, double scale) {
  for (auto* t : {&k, &v})
    TORCH_CHECK(t->dtype() == q.dtype() && t->dim() == 3 &&
                t->stride(2) == 1 && t->stride(1) == t->size(2));
  flash_check(out, q, cu_seqlens, seq_lens, k.size(1));
  FlashArgs a{};
  a.out = (uint16_t*)out.data_ptr();
  a.q = (const uint16_t*)q.data_ptr();
  a.k = (const uint16_t*)k.data_ptr();
  a.v = (const uint16_t*)v.data_ptr();
  a.cu = (const int32_t*)cu_seqlens.data_ptr();
  a.q_rs = q.stride(0);
  a.k_rs = k.stride(0);
  a.v_rs = v.stride(0);
  a.B = (int)seq_lens.size();
  a.nq = q.size(1);
  a.nkv = k.size(1);
  a.scale = (float)scale;
  flash_launch<false>(a, seq_lens, at::cuda::getCurrentCUDAStream());
}

}  // namespace igw
