// Absorbed latent attention of decoded tokens (gfx950, bf16).
//
// All heads of a token read the same cached rows (latent | rotated key), so 32
// heads are the 32 query rows of one MFMA tile and a row of the cache is its
// own key AND value: tiles of 64 rows go to LDS once, by DMA and double
// buffered, K fragments and transposed V fragments are read from the same
// image (flash_tile.h, SHARED).  The four waves of a workgroup score the same
// rows and take a quarter of the value dims each: scores are computed four
// times, which costs 9 MFLOP per 73 KB tile beside 2 for the values and is
// still far above what HBM delivers (both the MFMAs and the LDS reads of a
// tile take about 2800 cycles, 26 bytes per cycle and compute unit against 10
// from HBM), and there is no exchange of probabilities and one barrier a tile.
// One workgroup per compute unit (147 KB of LDS); contexts are cut to give
// every compute unit one.
//
// Measured with 32 heads, rank 512 + 64, against the tiles that stage rows
// twice (row-major and transposed by 2-byte stores): 48 tokens of 700 to 3500
// keys 262 and 67 us, 256 of 2048 538 and 187 (3.2 TB/s), one of 3000 125 and
// 35; rank 256, 16 heads, 256 of 2048: 241 and 109.
#include "../csrc/flash_tile.h"
#include "act_types.h"

namespace igw {

struct LatentDecodeArgs {
  const uint16_t *qa, *qr;   // [T, H, R], [T, H, RD]
  int64_t qa_s0, qa_s1, qr_s0, qr_s1;
  const uint16_t* cache;     // [pages, size, R + RD]
  const int32_t *block_table, *row_seq, *positions;
  int max_blocks, RD, size, window;
  float scale;
  FlashClose close;
  FlashParts parts;
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

template <int NK, int R, bool ONCE>
__global__ __launch_bounds__(64 * FT_WAVES, 1) void latent_decode_kernel(
    LatentDecodeArgs a) {
  constexpr int VD = R / FT_WAVES;
  __shared__ __attribute__((aligned(1024))) uint8_t k_s0[FT_BN * NK * 2];
  __shared__ __attribute__((aligned(1024))) uint8_t k_s1[FT_BN * NK * 2];
  const int lane = threadIdx.x & 63, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t t = blockIdx.x;
  const int H = a.close.heads;
  const int head = blockIdx.y * 32 + (lane & 31);
  const int pos = a.positions[t];

  ft_bf16x8 qf[NK / 16];
#pragma unroll
  for (int s = 0; s < NK / 16; ++s) {
    const int d = 16 * s + 8 * half;
    ft_bf16x8 f{};
    if (head < H && d < R + a.RD)
      f = *reinterpret_cast<const ft_bf16x8*>(
          d < R ? a.qa + t * a.qa_s0 + head * a.qa_s1 + d
                : a.qr + t * a.qr_s0 + head * a.qr_s1 + (d - R));
    qf[s] = f;
  }
  FlashScore sc{};
  sc.pos = sc.wave_pos = pos;
  sc.lo = sc.wave_lo[0] = sc.wave_lo[1] =
      a.window > 0 ? max(0, pos - a.window + 1) : 0;
  sc.c = a.scale * FT_LOG2E;
  const FlashSpan span = flash_part(
      FlashSpan{pos + 1, 0, sc.lo / FT_BN * FT_BN, pos + 1}, blockIdx.z,
      a.parts.nsplit);
  PagedRows rows{a.cache, nullptr,
                 a.block_table + (int64_t)a.row_seq[t] * a.max_blocks, 0, 1,
                 a.size, R + a.RD, 0, pos + 1};
  ft_f32x16 o[VD / 32];
  float m, l;
  flash_tiles<NK, R, false, PagedRows, VD, true, ONCE>(
      rows, span, sc, qf, k_s0, k_s1, nullptr, nullptr, o, m, l, wave * VD);
  if (head >= H) return;
  if (a.parts.nsplit > 1) {
    flash_store_part<VD>(a.parts, t * H + head, blockIdx.z, R, o, wave * VD, m,
                         l, half);
    return;
  }
  const float f = a.close.factor(t, head, 0) / a.close.sum(head, m, l);
  flash_store<VD>(a.close.out + (t * H + head) * R + wave * VD, o, VD, half,
                  [&](int) { return f; });
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
  // Parts of at least four tiles, of the longest context as many as give the
  // fewest rounds of workgroups, one per compute unit, times the tiles of a
  // part and about two for a workgroup's start and end (48 tokens of 2000, 32
  // heads, rank 512: six parts, a round and an eighth, 62 us, five parts 51).
  int64_t nsplit = 1, least = INT64_MAX;
  for (int64_t n = 1; n <= std::min<int64_t>(32, std::max<int64_t>(
                               1, tiles / 4)); ++n) {
    const int64_t rounds = (T * groups * n + cus - 1) / cus;
    const int64_t cost = rounds * ((tiles + n - 1) / n + 2);
    if (cost < least) {
      least = cost;
      nsplit = n;
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
      FlashParts{nullptr, nullptr, (int)nsplit}};
  if (nsplit > 1) {
    const int64_t slots = T * H * nsplit;
    part = torch::empty({slots * (R + 2)},
                        q_abs.options().dtype(torch::kFloat32));
    a.parts.o = part.data_ptr<float>();
    a.parts.ml = a.parts.o + slots * R;
  }
  hipStream_t stream = at::cuda::getCurrentCUDAStream();
  const dim3 grid(T, groups, nsplit), block(64 * FT_WAVES);
  const bool once = T * max_keys * (R + RD) * 2 >= LD_ONCE;
  auto* kern = R == 512 ? once ? latent_decode_kernel<576, 512, true>
                               : latent_decode_kernel<576, 512, false>
               : once   ? latent_decode_kernel<320, 256, true>
                        : latent_decode_kernel<320, 256, false>;
  hipLaunchKernelGGL(kern, grid, block, 0, stream, a);
  HIP_CHECK_KERNEL();
  if (nsplit > 1) {
    hipLaunchKernelGGL(flash_merge_kernel, dim3(T * H), dim3(R / 4), 0, stream,
                       a.close, a.parts, (const int32_t*)nullptr);
    HIP_CHECK_KERNEL();
  }
  return true;
}

}  // namespace igw
