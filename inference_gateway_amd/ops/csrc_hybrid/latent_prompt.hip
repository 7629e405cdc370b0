// Latent attention of prompt rows with the keys and values written out
// (gfx950, bf16).
//
// In absorbed form (latent_attn_mfma.hip) a score costs kv_rank + rot_dim
// multiply-adds and its value kv_rank more: at rank 512 that is 3.4 times the
// work of heads of 128 + 64 key and 128 value entries.  A prompt pays for the
// up-projections of its keys once (two library products of rows x kv_rank x
// heads x dim, as the absorbed form runs them on queries and results) and its
// rows x keys scores then run at the head's own widths on the tile walk of
// flash_tile.h: 128 rows of one head per workgroup, keys of NK = 192 padded
// entries from two sources, each head's own unrotated part and the rotated
// part that all heads share.
//
// Decoded tokens, and portions whose earlier tokens are only in the cache,
// stay absorbed: they would expand the whole context for a few rows.
//
// Measured with 32 heads, rank 512, 2 prompts of 3000 tokens, all the steps
// between the query and the value rows: absorbed 4563 us, written out 347 us,
// 125 of them the two products; 16 prompts of 512: 1650 and 241; one of 128:
// 72 and 62 (launches).
#include "../csrc/flash_tile.h"
#include "act_types.h"

namespace igw {

// Keys in two parts: kn [rows, heads * dn] (this head) | kr [rows, rd]
// (shared); values v [rows, vd] of this head.  Value chunks past the width
// repeat the first one, they are not stored.
struct LatentRows {
  const uint16_t *kn, *kr, *v;
  int kn_rs, kr_rs, v_rs;
  int dn, dk, vd, kv_len;
  const uint16_t *knt = nullptr, *krt = nullptr, *vt = nullptr;
  int last = 0;
  DEVINLINE void prefetch(int, int) {}
  DEVINLINE void begin(int kbase, int) {
    knt = kn + (int64_t)kbase * kn_rs;
    krt = kr + (int64_t)kbase * kr_rs;
    vt = v + (int64_t)kbase * v_rs;
    last = kv_len - 1 - kbase;
  }
  static constexpr bool STRAIGHT = false;   // keys from two places
  DEVINLINE int key_width() const { return dk; }
  template <bool PAD>
  DEVINLINE const uint16_t* kp(int r, int c) const {
    const int d = c * 8, in = min(r, last);
    return d < dn            ? knt + (uint32_t)(in * kn_rs + d)
           : !PAD || d < dk ? krt + (uint32_t)(in * kr_rs + (d - dn))
                             : ft_zeros;
  }
  DEVINLINE const uint16_t* vp(int r, int c) const {
    return vt + (uint32_t)(min(r, last) * v_rs + (c * 8 < vd ? c * 8 : 0));
  }
};

struct LatentPromptArgs {
  uint16_t* out;          // [P, H, vd]
  const uint16_t* q;      // [P, H, dn + rd], strides q_s0, q_s1
  int64_t q_s0, q_s1;
  const uint16_t* kn;     // [P, H * dn]
  const uint16_t* kr;     // [P, rd], row stride kr_rs
  int64_t kr_rs;
  const uint16_t* v;      // [H, P, vd]
  const int32_t* cu;      // [B + 1]
  const float *sink, *gate;  // [H], [P, H]
  int B, ntiles, H, P, dn, rd, vd, window;
  float scale;
};

constexpr int LP_NK = 192, LP_NV = 128;

__global__ __launch_bounds__(64 * FT_WAVES, 2) void latent_prompt_kernel(
    LatentPromptArgs a) {
  constexpr int NK = LP_NK, NV = LP_NV;
  __shared__ __attribute__((aligned(1024))) uint8_t k_s0[FT_BN * NK * 2];
  __shared__ __attribute__((aligned(1024))) uint8_t k_s1[FT_BN * NK * 2];
  __shared__ __attribute__((aligned(1024))) uint8_t v_s0[FT_BN * NV * 2];
  __shared__ __attribute__((aligned(1024))) uint8_t v_s1[FT_BN * NV * 2];
  const int lane = threadIdx.x & 63, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

  int head, tile, seq, qoff;
  ft_head_and_tile(a.H, a.ntiles, &head, &tile);
  if (!ft_find_tile<FT_BM>(a.cu, a.B, tile, &seq, &qoff)) return;
  const int q0 = a.cu[seq];
  const int L = a.cu[seq + 1] - q0;

  const int row = qoff + wave * 32 + (lane & 31);   // = position
  const int dk = a.dn + a.rd;
  ft_bf16x8 qf[NK / 16];
  const uint16_t* qp = a.q + (int64_t)(q0 + min(row, L - 1)) * a.q_s0 +
                       (int64_t)head * a.q_s1;
#pragma unroll
  for (int s = 0; s < NK / 16; ++s) {
    const int d = 16 * s + 8 * half;
    ft_bf16x8 f{};
    if (d < dk) f = *reinterpret_cast<const ft_bf16x8*>(qp + d);
    qf[s] = f;
  }

  auto first_key = [&](int pos) {
    return a.window > 0 ? max(0, pos - a.window + 1) : 0;
  };
  FlashScore sc{};
  sc.pos = row;
  sc.lo = first_key(row);
  sc.wave_pos = qoff + wave * 32;
  sc.wave_lo[0] = first_key(sc.wave_pos);
  sc.wave_lo[1] = first_key(sc.wave_pos + 31);
  sc.c = a.scale * FT_LOG2E;
  const FlashSpan span{L, 0, first_key(qoff) / FT_BN * FT_BN,
                       min(L, qoff + FT_BM)};
  LatentRows rows{a.kn + (int64_t)q0 * a.H * a.dn + head * a.dn,
                  a.kr + q0 * a.kr_rs,
                  a.v + ((int64_t)head * a.P + q0) * a.vd,
                  a.H * a.dn, (int)a.kr_rs, a.vd, a.dn, dk, a.vd, L};
  ft_f32x16 o[NV / 32];
  float m, l;
  flash_tiles<NK, NV, false>(rows, span, sc, qf, k_s0, k_s1, v_s0, v_s1, o, m,
                             l);
  if (row >= L) return;
  if (a.sink)   // a key with that score and no value
    l += __builtin_amdgcn_exp2f(fmaf(a.sink[head], FT_LOG2E, -m));
  const int64_t pair = (int64_t)(q0 + row) * a.H + head;
  const float f = (a.gate ? a.gate[pair] : 1.0f) / l;
  flash_store<NV>(a.out + pair * a.vd, o, a.vd, half, [&](int) { return f; });
}

// Whether latent_prompt takes these widths.
bool latent_prompt_fits(int64_t dn, int64_t rd, int64_t vd) {
  return dn > 0 && dn % 8 == 0 && rd % 8 == 0 && vd > 0 && vd % 8 == 0 &&
         dn + rd <= LP_NK && vd <= LP_NV;
}

// Rows of whole prompts: sequence i has rows cu[i] .. cu[i + 1] at positions
// 0, 1, ...; rows: their counts.  q [P, H, dn + rd] (strided ok), kn [P, H *
// dn], kr [P, rd] (strided rows ok), v [H, P, vd] -> out [P, H, vd].
void latent_prompt(torch::Tensor out, torch::Tensor q, torch::Tensor kn,
                   torch::Tensor kr, torch::Tensor v, torch::Tensor cu,
                   std::vector<int64_t> rows,
                   c10::optional<torch::Tensor> sink, double scale,
                   int64_t window, c10::optional<torch::Tensor> gate) {
  TORCH_CHECK(q.is_cuda() && q.dim() == 3 && q.stride(2) == 1 &&
              kr.dim() == 2 && kr.stride(1) == 1 && v.dim() == 3);
  for (auto* t : {&out, &q, &kn, &kr, &v})
    TORCH_CHECK(t->dtype() == torch::kBFloat16 &&
                (reinterpret_cast<uintptr_t>(t->data_ptr()) & 15) == 0);
  const int64_t P = q.size(0), H = q.size(1), rd = kr.size(1);
  const int64_t dn = q.size(2) - rd, vd = v.size(2);
  TORCH_CHECK(latent_prompt_fits(dn, rd, vd));
  TORCH_CHECK(q.stride(0) % 8 == 0 && q.stride(1) % 8 == 0 &&
              kr.stride(0) % 8 == 0 && kr.stride(0) < 1 << 24 &&
              H * dn < 1 << 24);
  TORCH_CHECK(kn.is_contiguous() && kn.numel() == P * H * dn &&
              kr.size(0) == P && v.is_contiguous() && v.size(0) == H &&
              v.size(1) == P && out.is_contiguous() &&
              out.numel() == P * H * vd);
  TORCH_CHECK(cu.dtype() == torch::kInt32 && cu.is_contiguous() &&
              cu.numel() > (int64_t)rows.size());
  for (auto* t : {&out, &kn, &kr, &v, &cu})
    TORCH_CHECK(t->device() == q.device(), "tensors on different devices");
  int64_t tiles = 0, total = 0;
  for (int64_t n : rows) {
    tiles += (n + FT_BM - 1) / FT_BM;
    total += n;
  }
  TORCH_CHECK(total == P, "row counts do not add up");
  if (sink.has_value())
    TORCH_CHECK(sink->dtype() == torch::kFloat32 && sink->is_contiguous() &&
                sink->numel() == H && sink->device() == q.device());
  if (gate.has_value())
    TORCH_CHECK(gate->dtype() == torch::kFloat32 && gate->is_contiguous() &&
                gate->numel() >= P * H && gate->device() == q.device());
  if (tiles == 0) return;
  LatentPromptArgs a{
      (uint16_t*)out.data_ptr(), (const uint16_t*)q.data_ptr(), q.stride(0),
      q.stride(1), (const uint16_t*)kn.data_ptr(),
      (const uint16_t*)kr.data_ptr(), kr.stride(0),
      (const uint16_t*)v.data_ptr(), (const int32_t*)cu.data_ptr(),
      sink.has_value() ? (const float*)sink->data_ptr() : nullptr,
      gate.has_value() ? (const float*)gate->data_ptr() : nullptr,
      (int)rows.size(), (int)tiles, (int)H, (int)P, (int)dn, (int)rd, (int)vd,
      (int)window, (float)scale};
  hipStream_t stream = at::cuda::getCurrentCUDAStream();
  hipLaunchKernelGGL(latent_prompt_kernel, dim3(tiles * H),
                     dim3(64 * FT_WAVES), 0, stream, a);
  HIP_CHECK_KERNEL();
}

}  // namespace igw
