// Products of hundreds to thousands of rows on the tiles of wide_tile.h: which tile a
// product takes and where it is ahead of the library, and the grouped products of
// a mixture of experts.
#include <ATen/cuda/CUDAContext.h>
#include <c10/cuda/CUDAGuard.h>
#include <torch/extension.h>

#include <cmath>

#include "wide_tile.h"

namespace igw {

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

// Up to this many rows, and entries of a row of W, a gated product reads W once and by
// nontemporal loads (us, plain and so: 28672 x 4096, 200 / 256 rows 70.4 73.3 and 66.8
// 69.4, 35840 x 5120 103 113 and 98.4 100).  384 and 512 rows gain or lose (28672 x 4096
// 82.9 96.7 and 80.2 94.1, 35840 x 5120 153 169 and 160 165), 8192 do not, where W comes
// back from the caches for every patch of tiles (1 % behind); longer rows of W are slower
// so (28672 x 14336, 134 rows, 218 and 257, 18560 x 11008, 138 rows, 154 and 179).
constexpr int64_t WIDE_ONCE = 256, WIDE_ONCE_K = 8192;

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
  const bool once = M <= WIDE_ONCE && K <= WIDE_ONCE_K;
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

// From this many entries of W, in rows of 4 KB and more, a grouped product of few rows
// an expert reads it by nontemporal loads and from turned starts (us, without and so; 2
// / 64 rows an expert: 8 x 4096 x 2048 as SwiGLU 32.5 37.1 and 26.4 30.1, 8 x 4096 x 4096
// 58 69 and 49 55).  Smaller W gains nothing (8 x 2048 x 2048 24.0 27.1 and 23.5 26.6; 4 x
// 4096 x 1024, 13.3 15.1 and 14.2 15.9), nor do shorter rows (64 x 1024 x 1024 as SwiGLU, 8
// rows, 28.8 and 32.1, 8 x 8192 x 1024 29.1 and 32.4).
constexpr int64_t GROUPED_ONCE = 48 << 20;

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
  // nontemporal W where half a patch of tiles has an expert's rows: three prompts of
  // 560 to 700 tokens on eight experts of 14336 x 4096, a step 1442 and 1330 us; with 790
  // rows an expert, some of which have more than a patch, 2484 and 2522
  const bool once = K >= 2048 && w.numel() >= GROUPED_ONCE;
#define LAUNCH_GROUPED_AS(...)                                                \
  hipLaunchKernelGGL((wide_gemm_kernel<__VA_ARGS__>), dim3(WG_BLOCKS),        \
                     dim3(256), 0, stream, a)
#define LAUNCH_GROUPED(MT, NT)                                                \
  case MT * 16 + NT:                                                          \
    if (swiglu && once && R <= E * 2 * 32 * MT)                               \
      LAUNCH_GROUPED_AS(MT, NT, 1, true, false, true);                        \
    else if (swiglu)                                                          \
      LAUNCH_GROUPED_AS(MT, NT, 1, true, false, false);                       \
    else if (once && R <= E * 2 * 32 * MT)                                    \
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
