// Products of a few rows with a matrix per head (gfx950, bf16): the absorbed halves
// of latent attention around its decoded tokens,
//
//   out[t, h, :] = x[t, h, :] W[h]        W [heads, K, N] as it is held, K-major
//
// and, in the same launch, the in-place rotation of the queries' other part.
//
// Bound by latency: 4 MB of W for 32 heads are 16 KB a compute unit, so all of a
// wave's loads are sent at once and used once.  A wave owns 32 columns and up to 128
// rows of K of one head: out^T = W^T x^T on mfma 32x32x16, W by DMA to a part of LDS
// of its own and transposed by the read (ds_read_b64_tr_b16; rows of 64 bytes, so
// that four neighbouring ones fill the banks), tokens as columns straight from
// memory.  The waves of a workgroup lie side by side along N, or, where N alone
// gives too few workgroups, one behind the other along K with their sums added
// through LDS in fp32.
//
// Measured in a step of 48 tokens, 32 heads, W cold (us): 128 x 512 with the rotation
// 13.2 and 4.1 as two launches, 6.1 here; 512 x 128 7.3 and 5.8.
#include "../csrc/flash_tile.h"
#include "../csrc/plain_call.h"
#include "act_types.h"

namespace igw {

constexpr int HP_ROWS = 128;   // tokens of a call at most: four tiles of columns

struct HeadProducts {
  uint16_t* out;        // [T, H, N], row strides o0, o1
  int64_t o0, o1;
  const uint16_t* x;    // [T, H, K], row strides x0, x1
  int64_t x0, x1;
  const uint16_t* w;    // [H, K, N]
  int T, H, K, N;
  // rotation of turn[t, h, 0 .. 2 pairs), or null; strides x0, x1
  uint16_t* turn;
  const int32_t* positions;
  const float* inv_freq;
  int pairs;
  bool half;
  float mag;
};

// KC: rows of K that a wave holds at a time.  NT: tiles of 32 tokens.  BY_K: the
// waves cut K.
template <int KC, int NT, bool BY_K>
__global__ __launch_bounds__(64 * FT_WAVES, 1) void head_products_kernel(
    HeadProducts a) {
  __shared__ __attribute__((aligned(1024))) uint8_t w_s[FT_WAVES * KC * 64];
  const int lane = threadIdx.x & 63, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h = blockIdx.x;
  const int cols = BY_K ? 32 : 32 * FT_WAVES;
  if ((int)blockIdx.y * cols >= a.N) {   // the workgroup that turns this head
    for (int i = threadIdx.x; i < a.T * a.pairs; i += 64 * FT_WAVES) {
      const int t = i / a.pairs, p = i - t * a.pairs;
      float s, c;
      sincosf((float)a.positions[t] * a.inv_freq[p], &s, &c);
      c *= a.mag;
      s *= a.mag;
      const int lo = a.half ? p : 2 * p, hi = a.half ? p + a.pairs : lo + 1;
      uint16_t* e = a.turn + t * a.x0 + h * a.x1;
      const float u = bf16_to_f32(e[lo]), v = bf16_to_f32(e[hi]);
      e[lo] = f32_to_bf16(u * c - v * s);
      e[hi] = f32_to_bf16(v * c + u * s);
    }
    return;
  }
  const int n0 = blockIdx.y * cols + (BY_K ? 0 : wave * 32);
  const int kper = BY_K ? a.K / FT_WAVES : a.K;
  const int k0 = BY_K ? wave * kper : 0;
  const uint16_t* w = a.w + ((int64_t)h * a.K + k0 + (lane >> 2)) * a.N + n0 +
                      (lane & 3) * 8;
  uint8_t* ws = w_s + wave * KC * 64;
  const uint16_t* x = a.x + h * a.x1 + k0 + 8 * half;
  const uint16_t* xr[NT];
  ft_f32x16 acc[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    xr[nt] = x + min(nt * 32 + (lane & 31), a.T - 1) * a.x0;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[nt][i] = 0.0f;
  }
  const int i16 = lane & 15;
  const int voff = (8 * half + (i16 >> 2)) * 64 + ((lane >> 4) & 1) * 32 +
                   (i16 & 3) * 8;
  for (int k = 0; k < kper; k += KC) {
#pragma unroll
    for (int i = 0; i < KC / 16; ++i)
      __builtin_amdgcn_global_load_lds(
          reinterpret_cast<const uint32_t*>(w + (int64_t)(k + 16 * i) * a.N),
          reinterpret_cast<uint32_t*>(ws + i * 1024), 16, 0, 0);
    ft_bf16x8 xf[KC / 16][NT];
#pragma unroll
    for (int s = 0; s < KC / 16; ++s)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
        xf[s][nt] =
            *reinterpret_cast<const ft_bf16x8*>(xr[nt] + k + 16 * s);
    // the rows are this wave's own: no barrier
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
    for (int s = 0; s < KC / 16; ++s) {
      typedef __attribute__((address_space(3))) ft_short4 lds_short4;
      union {
        ft_short4 h[2];
        ft_bf16x8 v;
      } wf;
#pragma unroll
      for (int e = 0; e < 2; ++e)
        wf.h[e] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (lds_short4*)(ws + voff + s * 1024 + e * 256));
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
        acc[nt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf.v, xf[s][nt],
                                                          acc[nt], 0, 0, 0);
    }
  }
  if constexpr (BY_K) {
    // wave g adds the entries 8 g .. + 7 of all
    __shared__ float4 sum_s[FT_WAVES][NT][4][64];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        sum_s[wave][nt][g][lane] =
            make_float4(acc[nt][4 * g], acc[nt][4 * g + 1],
                        acc[nt][4 * g + 2], acc[nt][4 * g + 3]);
    __syncthreads();
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const int t = nt * 32 + (lane & 31);
      float4 y = sum_s[0][nt][wave][lane];
#pragma unroll
      for (int v = 1; v < FT_WAVES; ++v) {
        const float4 z = sum_s[v][nt][wave][lane];
        y.x += z.x;
        y.y += z.y;
        y.z += z.z;
        y.w += z.w;
      }
      if (t < a.T) {
        uint2 o;
        o.x = ft_pack_bf16(y.x, y.y);
        o.y = ft_pack_bf16(y.z, y.w);
        *reinterpret_cast<uint2*>(a.out + t * a.o0 + h * a.o1 + n0 + 8 * wave +
                                  4 * half) = o;
      }
    }
  } else {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const int t = nt * 32 + (lane & 31);
      const ft_f32x16 o[1] = {acc[nt]};
      if (t < a.T)
        flash_store<32>(a.out + t * a.o0 + h * a.o1 + n0, o, 32, half,
                        [](int) { return 1.0f; });
    }
  }
}

// Whether the kernel is ahead of the library's batched product (and, of `pairs`
// turned pairs, of that and rope_pairs).  It sends a wave's loads once, tokens with
// them: its time grows with the tokens a wave has, and with the rounds of workgroups,
// where the library's hardly does (us, it and this):
//  * by columns, 1 / 32 / 48 / 64 / 96 tokens of 32 heads: 64 x 128 4.9 4.2 4.7 4.5
//    4.9 and 2.4 2.9 3.8 4.0 5.2, 128 x 128 5.6 4.7 5.3 5.1 5.6 and 2.7 3.7 4.7 5.1
//    7.0, 128 x 256 5.3 5.7 6.7 6.4 8.2 and 3.2 4.0 5.0 5.5 7.5, 64 x 512 6.9 4.5 4.9
//    and 3.0 3.5 4.1, 128 x 512 of four heads 3.8 3.9 4.0 and 2.6 3.7 4.6, of 128
//    heads, 16 / 32 tokens 7.4 7.9 and 6.8 8.3;
//  * with 32 pairs a head turned, 32 heads, 48 / 64 / 96 / 128 tokens: 128 x 128 8.0
//    7.8 8.3 8.8 and 4.8 5.2 7.0 8.1, 128 x 512 8.3 8.3 8.8 and 5.3 5.8 7.7, of four
//    heads 6.1 6.6 6.4 and 4.7 5.1 6.9, 128 x 256 of 128 heads 12.4 12.3 14.2 14.2 and
//    7.6 8.9 13.1 17.4.  One workgroup turns a head, which takes 8 us of 4096 pairs;
//  * cut by K, 1 / 32 / 64 / 128 tokens: 512 x 128, 32 heads 9.9 8.8 9.1 10.7 and 3.6
//    4.2 5.4 8.2, 128 heads 12.7 12.1 12.5 and 6.2 7.6 10.3, 768 x 128, 128 heads 12.4
//    11.5 12.1 and 7.2 9.4 13.5, 1024 x 128, 16 heads 6.3 6.5 6.7 8.6 and 4.6 5.8 8.0
//    12.5, 512 x 256, 128 heads, 1 / 32 / 48 tokens 13.7 13.7 14.7 and 8.8 11.7 14.8.
//    Of wider ones the library is ahead early (512 x 512, 64 heads, 16 tokens 10.5 and
//    10.7, 1024 x 1024, 16 heads, one token 10.3 and 11.4);
//  * of more than 128 heads the library is ahead early (128 x 256, 160 heads, 32 / 64
//    tokens 7.5 7.5 and 6.9 9.4).
static bool hp_ahead(int64_t T, int64_t H, int64_t K, int64_t N,
                     int64_t pairs) {
  if (T * pairs > 3072 || H > 128) return false;
  if (K > 128)
    return N <= 256 && K * N <= 131072 && (K <= 768 || T <= 32) &&
           T * H * N * std::max<int64_t>(K, 512) <= (int64_t)1 << 29;
  if (pairs > 0) return T * N <= 49152 && T <= (N > 256 ? 64 : 96);
  if (N > 256)
    return T * N <= 24576 &&
           T <= (K <= 64 ? 48 : H * N < 65536 ? 32 : 16);
  return T <= 96 && (N > 128 || (T <= 64 && T * K <= 6144));
}

// x [T, H, K] times W [H, K, N] per head, in `out` [T, H, N] where it is given; with
// `turn` [T, H, 2 pairs] (the same strides as x) its rotation in place, as
// rope_pairs does it.  Nothing, and nothing done, when the call does not fit: the
// caller then runs the library's batched product.
c10::optional<torch::Tensor> head_products(
    c10::optional<torch::Tensor> given, torch::Tensor x, torch::Tensor w,
    c10::optional<torch::Tensor> turn, c10::optional<torch::Tensor> positions,
    c10::optional<torch::Tensor> inv_freq, bool half, double mag) {
  if (!x.is_cuda() || !call_is_plain() || !plain_bf16(x, x.device()) ||
      !plain_bf16(w, x.device()) || x.dim() != 3 || w.dim() != 3 ||
      (given.has_value() &&
       (!plain_bf16(*given, x.device()) || given->dim() != 3)))
    return c10::nullopt;
  const int64_t T = x.size(0), H = x.size(1), K = x.size(2), N = w.size(2);
  TORCH_CHECK(w.size(0) == H && w.size(1) == K &&
                  (!given.has_value() ||
                   (given->size(0) == T && given->size(1) == H &&
                    given->size(2) == N)),
              "head_products: sizes");
  auto on = [](const torch::Tensor& t, int64_t bytes) {
    return reinterpret_cast<uintptr_t>(t.data_ptr()) % bytes == 0 &&
           t.stride(2) == 1 && t.stride(0) % (bytes / 2) == 0 &&
           t.stride(1) % (bytes / 2) == 0;
  };
  if (T < 1 || T > HP_ROWS || H < 1 || K < 64 || K > 1024 || N < 128 ||
      N > 4096 || N % 128 || K % 64 || !w.is_contiguous() || !on(x, 16) ||
      !on(w, 16) || (given.has_value() && !on(*given, 8)))
    return c10::nullopt;
  // By columns where a wave can have all of K at once; longer ones are cut over the
  // waves.
  const bool by_k = K > 128;
  if (!hp_ahead(T, H, K, N, turn.has_value() ? turn->size(2) / 2 : 0))
    return c10::nullopt;
  const int64_t kper = by_k ? K / FT_WAVES : K;
  if (kper * (by_k ? FT_WAVES : 1) != K || kper % 64) return c10::nullopt;
  const torch::Tensor out =
      given.has_value() ? *given : torch::empty({T, H, N}, x.options());
  HeadProducts a{(uint16_t*)out.data_ptr(), out.stride(0), out.stride(1),
                 (const uint16_t*)x.data_ptr(), x.stride(0), x.stride(1),
                 (const uint16_t*)w.data_ptr(), (int)T, (int)H, (int)K, (int)N,
                 nullptr, nullptr, nullptr, 0, half, (float)mag};
  if (turn.has_value()) {
    TORCH_CHECK(positions.has_value() && inv_freq.has_value() &&
                positions->dtype() == torch::kInt32 &&
                positions->is_contiguous() && positions->numel() == T &&
                inv_freq->dtype() == torch::kFloat32 &&
                inv_freq->is_contiguous());
    a.pairs = inv_freq->numel();
    TORCH_CHECK(turn->dtype() == x.dtype() && turn->dim() == 3 &&
                turn->size(0) == T && turn->size(1) == H &&
                turn->size(2) == 2 * a.pairs && turn->stride(2) == 1 &&
                turn->stride(0) == x.stride(0) &&
                turn->stride(1) == x.stride(1));
    a.turn = (uint16_t*)turn->data_ptr();
    a.positions = (const int32_t*)positions->data_ptr();
    a.inv_freq = (const float*)inv_freq->data_ptr();
  }
  hipStream_t stream = at::cuda::getCurrentCUDAStream();
  const dim3 grid(H, N / (by_k ? 32 : 32 * FT_WAVES) + (a.pairs > 0 ? 1 : 0));
#define LAUNCH_HP(KC, NT, BY_K)                                            \
  hipLaunchKernelGGL((head_products_kernel<KC, NT, BY_K>), grid,           \
                     dim3(64 * FT_WAVES), 0, stream, a)
#define LAUNCH_HP_NT(KC, BY_K)                                             \
  do {                                                                     \
    if (T <= 32) LAUNCH_HP(KC, 1, BY_K);                                   \
    else if (T <= 64) LAUNCH_HP(KC, 2, BY_K);                              \
    else LAUNCH_HP(KC, 4, BY_K);                                           \
  } while (0)
  if (by_k) {
    if (kper % 128 == 0) LAUNCH_HP_NT(128, true);
    else LAUNCH_HP_NT(64, true);
  } else {
    if (kper % 128 == 0) LAUNCH_HP_NT(128, false);
    else LAUNCH_HP_NT(64, false);
  }
#undef LAUNCH_HP_NT
#undef LAUNCH_HP
  HIP_CHECK_KERNEL();
  return out;
}

}  // namespace igw
