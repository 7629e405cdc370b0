// Varlen causal flash attention for prompt rows, gfx950 (MI355X), bf16.
//
// One kernel (the tile walk is flash_tile.h), two sources of keys and values:
// the freshly projected dense K/V of whole prompts (flash_prefill), or the
// paged cache (flash_prefill_paged: chunked prefill and prefix reuse, where
// the q rows are a chunk behind `prefix` cached tokens and row r sits at
// position prefix + r; the chunk's own keys are already appended).
//
// Measured with 32 heads on 8 (cards differ by 10 %), alone and between the other
// kernels of a step: one prompt of 16000 tokens 1979 us, 1060 TFLOP/s, and 2130 (64
// x 64 tiles of 16x16x32 MFMAs with V transposed by the stores and P through LDS:
// 12518 us); 16 prompts of 512 71 us, 487 TFLOP/s, and 84; 2000 rows behind 6000
// cached ones 236 us, 974 TFLOP/s, and 279.

#include <ATen/cuda/CUDAContext.h>
#include <torch/extension.h>

#include "flash_tile.h"

namespace igw {

constexpr int FP_HD = 128;   // head dim
constexpr int FP_PAGE = 16;  // tokens per cache page

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

template <bool PAGED>
__global__ __launch_bounds__(64 * FT_WAVES, 2) void flash_prefill_kernel(
    FlashArgs a) {
  constexpr int HD = FP_HD;
  __shared__ __attribute__((aligned(1024))) uint8_t k_s0[FT_BN * HD * 2];
  __shared__ __attribute__((aligned(1024))) uint8_t k_s1[FT_BN * HD * 2];
  __shared__ __attribute__((aligned(1024))) uint8_t v_s0[FT_BN * HD * 2];
  __shared__ __attribute__((aligned(1024))) uint8_t v_s1[FT_BN * HD * 2];
  const int lane = threadIdx.x & 63, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

  int qh, tile, seq, qoff;
  ft_head_and_tile(a.nq, a.ntiles, &qh, &tile);
  if (!ft_find_tile<FT_BM>(a.cu, a.B, tile, &seq, &qoff)) return;
  const int kvh = qh / (a.nq / a.nkv);
  const int q0 = a.cu[seq];
  const int Lq = a.cu[seq + 1] - q0;
  const int P = PAGED ? a.prefix[seq] : 0;
  const int KVL = P + Lq;

  // this lane's query row: dims 16 s + 8 half .. + 7
  const int row = qoff + wave * 32 + (lane & 31);
  ft_bf16x8 qf[HD / 16];
  const uint16_t* qp = a.q + (int64_t)(q0 + min(row, Lq - 1)) * a.q_rs +
                       (int64_t)qh * HD + 8 * half;
#pragma unroll
  for (int s = 0; s < HD / 16; ++s)
    qf[s] = *reinterpret_cast<const ft_bf16x8*>(qp + 16 * s);
  // the running maximum is of raw scores: a negative scale turns q round
  if (a.scale < 0.0f) {
#pragma unroll
    for (int s = 0; s < HD / 16; ++s) qf[s] = -qf[s];
  }

  const FlashSpan span{KVL, 0, 0, min(KVL, P + qoff + FT_BM)};
  FlashScore sc{};
  sc.pos = P + row;
  sc.wave_pos = P + qoff + wave * 32;
  // not 0, so that a masked score stays -inf
  sc.c = fmaxf(fabsf(a.scale) * FT_LOG2E, 1e-37f);
  ft_f32x16 o[HD / 32];
  float m, l;
  if constexpr (PAGED) {
    PagedRows rows{a.k, a.v, a.block_table + (int64_t)seq * a.max_blocks,
                   kvh, a.nkv, FP_PAGE, HD, HD, KVL};
    flash_tiles<HD, HD, true>(rows, span, sc, qf, k_s0, k_s1, v_s0, v_s1, o,
                              m, l);
  } else {
    DenseRows rows{a.k + q0 * a.k_rs + kvh * HD, a.v + q0 * a.v_rs + kvh * HD,
                   (int)a.k_rs, (int)a.v_rs, KVL};
    flash_tiles<HD, HD, true>(rows, span, sc, qf, k_s0, k_s1, v_s0, v_s1, o,
                              m, l);
  }
  if (row < Lq) {
    const float inv = 1.0f / l;
    flash_store<HD>(a.out + ((int64_t)(q0 + row) * a.nq + qh) * HD, o, HD,
                    half, [&](int) { return inv; });
  }
}

template <bool PAGED>
static void flash_launch(FlashArgs& a, const std::vector<int64_t>& seq_lens,
                         hipStream_t stream) {
  int64_t tiles = 0;
  for (int64_t len : seq_lens) tiles += (len + FT_BM - 1) / FT_BM;
  if (tiles == 0) return;
  a.ntiles = (int)tiles;
  hipLaunchKernelGGL((flash_prefill_kernel<PAGED>), dim3(tiles * a.nq),
                     dim3(64 * FT_WAVES), 0, stream, a);
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

// The tile loads move 16 bytes to LDS at a time and want them aligned, at
// 32-bit offsets within a tile: views that are not (never the model's) are
// copied.
static torch::Tensor flash_aligned(const torch::Tensor& t) {
  bool ok = (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0;
  for (int64_t d = 0; d + 1 < t.dim(); ++d)
    ok = ok && (t.stride(d) % 8 == 0 || t.size(d) == 1);
  ok = ok && (t.dim() != 3 || (t.stride(0) >= 0 && t.stride(0) < 1 << 24));
  return ok ? t : t.clone(at::MemoryFormat::Contiguous);
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
  kcache = flash_aligned(kcache);
  vcache = flash_aligned(vcache);
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
  k = flash_aligned(k);
  v = flash_aligned(v);
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
