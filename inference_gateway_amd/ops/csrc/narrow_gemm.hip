// Products of a few to hundreds of rows on the tiles of wide_tile.h: with K in parts,
// or on tiles of fewer columns, where the whole K of wide tiles would leave compute
// units without one.
#include <ATen/cuda/CUDAContext.h>
#include <c10/cuda/CUDAGuard.h>
#include <torch/extension.h>

#include <cmath>

#include "wide_tile.h"

namespace igw {

bool wide_gemm_fits(int64_t x_rs, int64_t N, int64_t K, bool swiglu);
int64_t wide_gemm_tile(int64_t M, int64_t N, int64_t K, bool swiglu);

// Products of rows that leave the chip idle, K in parts.
//
// Tiles with a part of K each, their fp32 sums to memory, and a second kernel to add
// them (with the residual and the norm behind it where there is one).  wide_split picks
// the tile and the parts by what they cost: rounds of 256 items at `step` us a K step of
// 64, against W from HBM, and the sums' way to memory and back.  Of 1044 measured pairs
// of a tile and parts the model is off by 12 % on average (10 % too low: it leaves out
// what a launch costs whatever its size), and its choice is 1 % behind the best, 7 % at
// worst.
struct SplitTile {
  int MT, NT;
  double step;
};
// us for `work` us of steps beside `mb` MB of W from HBM: about the longer of the two.
// 4.6 TB/s was fitted with plain loads; read once by nontemporal ones W comes at up to
// 6.4 (128256 x 4096, 16 rows), for which the choices here are priced too high alike.
static double split_cost(double work, double mb) {
  const double stream = mb / 4.6, a = work * work, b = stream * stream;
  return std::sqrt(std::sqrt(a * a + b * b));
}
static constexpr SplitTile split_tiles[] = {
    {3, 4, 0.500}, {4, 4, 0.567}, {4, 6, 0.712}, {6, 4, 0.671}, {6, 6, 0.845},
    {6, 8, 1.069}, {8, 4, 0.799}, {8, 6, 1.049}, {8, 8, 1.387}};

// 256 times the tile (16 MT + NT) and the parts of K, at least two; 0: cannot be.
int64_t wide_split(int64_t M, int64_t N, int64_t K) {
  if (M < 65 || M > (1 << 16) || N < 8 || N % 8 != 0 || N > (1 << 20) ||
      K % (2 * WG_BK) != 0 || K > (1 << 20))
    return 0;
  int64_t best = 0;
  double least = 0.0;
  const int64_t pairs = K / (2 * WG_BK);
  for (const auto& c : split_tiles)
    for (int64_t S = 2; S <= 16 && 3 * S <= pairs; ++S) {
      const int64_t items = (M + 32 * c.MT - 1) / (32 * c.MT) *
                            ((N + 32 * c.NT - 1) / (32 * c.NT)) * S;
      const int64_t rounds = (items + WG_BLOCKS - 1) / WG_BLOCKS;
      const double work =
          rounds * (2 * ((pairs + S - 1) / S) * c.step + 0.11);
      const double cost =
          split_cost(work, N * K * 2e-6) + S * M * N * 4e-6 * 0.36;
      if (best == 0 || cost < least) {
        best = (c.MT * 16 + c.NT) * 256 + S;
        least = cost;
      }
    }
  return best;
}

// What wide_split says where that is ahead of the library, else 0; norm: where the
// norm that follows adds the parts, of the library and fused_add_rmsnorm.  Measured at
// 29 sizes of W by 24 of 65 to 2048 rows (us, library and here; then with the norm).
// Over a long K the library's tiles are few: 4096 x 14336, 65 / 128 / 256 / 512 / 1024 /
// 2033 rows 47.7 75.0 61.2 88.2 130 205 and 30.3 37.3 48.2 61.9 108 181; 5120 x 17920,
// 65 / 256 / 1024 rows 145 220 246 and 42.9 60.8 156, but 2033 rows 290 and 311; 8192 x
// 28672, 512 / 640 rows 312 265 and 183 271.  Of squarer W the parts' way to memory
// weighs more: 4096 x 4096, 128 / 256 / 512 / 1024 / 1600 rows 24.2 22.4 29.2 40.7 54.0
// and 17.8 21.3 29.7 41.7 64.1 (with the norm 27.3 25.9 33.8 46.9 62.6 and 19.0 22.5 31.6
// 44.3 68.1), 5120 x 5120, 256 / 640 / 1024 rows 49.6 50.4 62.1 and 29.0 45.7 58.9, 7680
// x 5120, 128 / 512 / 640 rows 33.4 52.1 58.2 and 27.3 50.1 60.1, 6144 x 4096, 128 / 160
// / 200 rows 25.4 27.8 25.4 and 21.0 23.7 25.2, 8192 x 8192, 128 rows 47.4 and 36.1 (65
// rows, which the line leaves to the library, 36.9 and 32.8).  Small W and a short K pay
// for the second launch: 1024 x 4096, 128 rows, 11.8 and 12.2, 4096 x 2048 14.6 and 15.4,
// as do wide ones: 16384 x 4096 36.8 and 38.1.  Without the norm the library is ahead
// where its tiles come out even: 5120 x 4096, 65 / 80 rows 16.5 16.9 and 18.3 17.4; 9216
// x 6144, 257 / 384 rows 49.9 60.0 and 59.8 66.3, 10240 x 5120, 257 rows 43.6 and 49.9.
int64_t wide_split_ahead(int64_t M, int64_t N, int64_t K, bool norm) {
  const int64_t least = N > 7680 && K < 2 * N            ? 128
                        : !norm && N <= 5120 && K < N ? 81
                                                      : 65;
  int64_t most;
  if (norm) {
    if (K < 3584 || N * K < (int64_t)12 << 20 || N > 16384) return 0;
    most = K >= 3 * N   ? N > 5120 ? 512 : N > 4096 ? 1600 : 2048
           : K >= 2 * N ? N > 5120 ? 512 : 1600
           : K >= N     ? N > 7680 ? 512 : 1024
                        : 512;
  } else {
    if (K < 4096 || N * K < (int64_t)16 << 20 || N < 2048 || N > 10240) return 0;
    most = K >= 3 * N   ? N > 5120 ? 512 : N > 4096 ? 1600 : 2048
           : K >= 2 * N ? N > 5120 ? 512 : 1300
           : K >= 5120  ? N > 7680 && K < 8192 ? 256 : 512
           : K >= N     ? 256
                        : 160;
  }
  return M >= least && M <= most ? wide_split(M, N, K) : 0;
}

// W from this many entries on is read by nontemporal loads where one patch of tiles
// has all rows (us, plain and so: 8192 x 28672, 65 / 256 / 512 rows 105.3 148.6 201
// and 88.0 119.5 187.5; 4096 x 14336, 65 / 128 rows 35.2 39.4 and 30.4 36.4, most of it
// the turned K, 256 rows 47.5 and 48.6; 12288 x 4096, 128 / 256 rows 34.7 41.7 and 33.6
// 42.0).  Less of it is slower so: 4096 x 4096, 65 / 128 / 256 rows 15.4 17.6 21.3 and
// 16.2 19.2 25.5; 7680 x 5120, 128 / 256 rows 27.1 38.4 and 29.8 39.9; 4096 x 8192 25.0
// 32.1 and 27.0 32.6.
constexpr int64_t SPLIT_ONCE = 48 << 20;

// The sums [S, M, N] of the parts that wide_split says.
torch::Tensor split_parts(const torch::Tensor& x, const torch::Tensor& w,
                          int64_t tile, int64_t S) {
  TORCH_CHECK(x.is_cuda() && x.dim() == 2 && x.stride(1) == 1 &&
              x.dtype() == torch::kBFloat16 && w.dtype() == x.dtype() &&
              w.dim() == 2 && w.is_contiguous());
  const int64_t M = x.size(0), K = x.size(1), N = w.size(0);
  TORCH_CHECK(M >= 1 && N >= 8 && N % 8 == 0 && S >= 1 && S <= 64 &&
              K / (2 * WG_BK) >= 3 * S && K % (2 * WG_BK) == 0 &&
              M <= (1 << 20) && N <= (1 << 20) && K <= (1 << 20) &&
              wide_gemm_fits(x.stride(0), N, K, false));
  TORCH_CHECK(w.size(1) == K && x.stride(0) % 8 == 0);
  TORCH_CHECK(w.device() == x.device(), "tensors on different devices");
  for (const auto* t : {&x, &w})
    TORCH_CHECK((reinterpret_cast<uintptr_t>(t->data_ptr()) & 15) == 0);
  const at::cuda::CUDAGuard guard(x.device());
  hipStream_t stream = at::cuda::getCurrentCUDAStream();
  auto part = torch::empty({S, M, N}, x.options().dtype(torch::kFloat32));
  const WideArgs a{nullptr, (const uint16_t*)x.data_ptr(),
                   (const uint16_t*)w.data_ptr(), (int)M, (int)N, (int)K,
                   x.stride(0), nullptr, 0, part.data_ptr<float>(), (int)S};
  const bool once = N * K >= SPLIT_ONCE;
#define LAUNCH_SPLIT_AS(...)                                                  \
  hipLaunchKernelGGL((wide_gemm_kernel<__VA_ARGS__>), dim3(WG_BLOCKS),        \
                     dim3(256), 0, stream, a)
#define LAUNCH_SPLIT(MT, NT)                                                  \
  case MT * 16 + NT:                                                          \
    if (once && M <= 4 * 32 * MT)                                             \
      LAUNCH_SPLIT_AS(MT, NT, 0, false, true, true);                          \
    else                                                                      \
      LAUNCH_SPLIT_AS(MT, NT, 0, false, true, false);                         \
    break
  switch (tile) {
    LAUNCH_SPLIT(3, 4);
    LAUNCH_SPLIT(4, 4);
    LAUNCH_SPLIT(4, 6);
    LAUNCH_SPLIT(6, 4);
    LAUNCH_SPLIT(6, 6);
    LAUNCH_SPLIT(6, 8);
    LAUNCH_SPLIT(8, 4);
    LAUNCH_SPLIT(8, 6);
    LAUNCH_SPLIT(8, 8);
    default: TORCH_CHECK(false, "no such tile: ", tile);
  }
#undef LAUNCH_SPLIT
#undef LAUNCH_SPLIT_AS
  HIP_CHECK_KERNEL();
  return part;
}

// Gated products of up to 384 rows, and plain ones of many outputs of up to 256, on
// tiles of 64 to 128 columns.
//
// So few rows are bound by streaming W, and wider tiles leave compute units without
// one: 28672 rows of W are 112 tiles of 256 and 224 of 128.  Measured, what a call would
// have else (the library with silu_mul, rows_gemm, held_gemm or the tiles of
// wide_gemm_tile) and here (us): 28672 x 4096 as SwiGLU, 61 / 65 / 128 / 200 / 256 rows
// 44.8 60.6 61.1 64.9 66.3 and 41.5 42.9 48.6 59.7 60.8; 35840 x 5120, 16 / 48 / 65 / 128 /
// 256 / 384 rows 91.2 98.1 80.5 86.8 93.1 154 and 62.1 66.6 64.8 72.8 86.1 138; 57344 x
// 8192, 61 rows, 174 and 153, but 160 and 256, which wide_gemm_tile's tiles keep, 162 190
// and 206 231; 14336 x 4096, 160 / 256 rows 42.8 54.9 and 37.8 42.8, but 96 rows, with 112
// tiles, 36.4 and 39.3; 128256 x 4096, 9 / 32 / 61 / 65 / 128 / 256 rows 167 180 194 230
// 237 302 and 164 171 176 172 169 242; 32064 x 5120, 16 / 48 / 65 / 256 rows 69.1 80.7 68.8
// 94.6 and 53.6 55.2 57.9 84.9; 28672 x 4096, 61 rows 45.7 and 43.5, but 24 and 48 rows
// 39.6 41.0 and 41.6 42.6; 24576 x 5120, with 192 tiles, 64 rows 51.4 and 52.0 (as SwiGLU
// 24576 x 4096 53.8 and 39.3); 65536 x 2048 and 152064 x 3584, 32 rows 67.3 262 and 44.7
// 190, and 16 rows, which held_gemm keeps, 48.5 186 and 43.9 180; 49152 x 6144, 65 / 160 /
// 256 rows 151 163 200 and 107 107 136; 32768 x 8192 126 134 158 and 88.7 103 123; 128256 x
// 8192 425 457 546 and 339 391 474.
// Of more than 128 rows the library is ahead where its tiles, 256 wide, are one round,
// ours of 192 more, and rows of W do not lie a multiple of 4 KB apart (57344 x 3584, 129 /
// 160 / 256 rows 90.4 90.0 95.3 and 97.5 100 111; 65536 x 2560 77 77 83 and 83 84 93; but
// 65536 x 4096 151 138 149 and 107 110 125), of more than 192 also where they do, over a
// long K or where they leave a part of the round (65536 x 8192, 200 / 256 rows, 224 246 and
// 247 245; 57344 x 4096, 193 / 256 rows 111 113 and 117 121; but 98304 x 8192, 200 / 256
// rows 403 410 and 347 352).
static constexpr SplitTile two_tiles[] = {
    {2, 4, 0.450}, {2, 5, 0.500}, {2, 8, 0.850}};  // up to 64 rows
static constexpr SplitTile narrow_tiles[] = {
    {3, 4, 0.500}, {4, 4, 0.567}, {3, 5, 0.560}, {4, 5, 0.640}, {6, 4, 0.671},
    {6, 5, 0.758}, {8, 4, 0.799}, {8, 5, 0.920}};
static constexpr SplitTile few_wide_tiles[] = {
    {3, 4, 0.500}, {4, 4, 0.567}, {6, 4, 0.671}, {8, 4, 0.799}, {3, 8, 0.769},
    {4, 8, 0.864}, {6, 6, 0.845}, {8, 6, 1.049}};
// the tiles that a gated product of more than 64 rows would have else
static constexpr SplitTile gated_tiles[] = {
    {4, 8, 0.864}, {6, 8, 1.069}, {8, 6, 1.049}, {8, 7, 1.220}, {8, 8, 1.387}};

// Gated products of a K above 2048 that the library would have else (wide_gemm_tile does
// not take them): it is ahead where the second row of tiles is filled to a third, or the
// third to a half, as W is read again for it (us, library with silu_mul and here: 16384 x
// 5120, 107 rows, 47.7 and 53.4, 12288 x 8192 59.4 and 64.9; 8192 x 5120, 200 rows, 40.0
// and 44.3, 12288 x 6144, 239 rows, 64.0 and 68.8; but 16384 x 6144, whose rows of W lie a
// multiple of 4 KB apart, 107 rows, 0.98 of the library's time, and 10240 x 5120, whose
// tiles fill a round, 193 and 239 rows, 0.93 and 0.89).
static bool mostly_empty(int64_t M, int64_t N, int64_t K, int64_t tile,
                         int64_t tiles) {
  const int64_t tm = 32 * (tile >> 4), last = (M - 1) % tm + 1;
  if (K <= 2048) return false;
  if (M > tm && M <= 2 * tm)
    return 3 * last <= tm && (K % 2048 != 0 || N < 8192);
  return M > 2 * tm && M <= 3 * tm && 2 * last <= tm &&
         tiles < WG_BLOCKS * 15 / 16;
}

// 16 MT + NT of the tile, or 0.
int64_t narrow_tile(int64_t M, int64_t N, int64_t K, bool gated) {
  if (M < 7 || M > (gated ? 384 : 256) || N < 8 || N % 8 != 0 ||
      N > (1 << 24) || K < 2048 || K > 8192 || K % (2 * WG_BK) != 0 ||
      (!gated && M > 64 && N < 32000))
    return 0;
  auto price = [&](const SplitTile& c, int64_t* items) {
    const int64_t tn = (gated ? 16 : 32) * c.NT;
    *items = (M + 32 * c.MT - 1) / (32 * c.MT) * ((N + tn - 1) / tn);
    const int64_t rounds = (*items + WG_BLOCKS - 1) / WG_BLOCKS;
    return split_cost(rounds * (K / WG_BK) * c.step,
                      (gated ? 2 : 1) * N * K * 2e-6);
  };
  int64_t best = 0, tiles = 0, items = 0;
  double least = 0.0;
  for (int i = 0; i < (M <= 64 ? 3 : 8); ++i) {
    const auto& c = M <= 64 ? two_tiles[i] : gated ? narrow_tiles[i] : few_wide_tiles[i];
    if (!gated && c.NT % 2 != 0) continue;
    const double cost = price(c, &items);
    if (best == 0 || cost < least) {
      best = c.MT * 16 + c.NT;
      least = cost;
      tiles = items;
    }
  }
  if (!gated && M > 64) {
    const int64_t its = (N + 255) / 256;   // the library's tiles
    const bool round = N > 192 * WG_BLOCKS && its <= WG_BLOCKS;
    const bool even = K % 2048 == 0 &&
                      (M <= 192 || (K <= 6144 && its > WG_BLOCKS * 15 / 16));
    return M > 128 && round && !even ? 0 : best;
  }
  if (M > 64)
    for (const auto& c : gated_tiles)
      if (price(c, &items) <= least) return 0;
  if (M > 64 && wide_gemm_tile(M, N, K, true) == 0 && mostly_empty(M, N, K, best, tiles))
    return 0;
  return tiles >= WG_BLOCKS * (gated ? 6 : 7) / 8 ? best : 0;
}

void narrow_gemm(torch::Tensor out, torch::Tensor x, torch::Tensor w,
                 int64_t gate, int64_t tile) {
  const bool swiglu = gate != 0;
  TORCH_CHECK(gate >= 0 && gate <= 2);
  TORCH_CHECK(x.is_cuda() && x.dim() == 2 && x.stride(1) == 1 &&
              x.dtype() == torch::kBFloat16 && w.dtype() == x.dtype() &&
              w.dim() == 2 && w.is_contiguous() && out.dim() == 2 &&
              out.is_contiguous() && out.dtype() == x.dtype());
  const int64_t M = x.size(0), K = x.size(1), N = out.size(1);
  TORCH_CHECK(M >= 1 && N >= 8 && N % 8 == 0 && K >= 6 * WG_BK &&
              K % (2 * WG_BK) == 0 && M <= (1 << 20) && N <= (1 << 24) &&
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
#define LAUNCH_NARROW_AS(...)                                                 \
  hipLaunchKernelGGL((wide_gemm_kernel<__VA_ARGS__, false, false, true>),     \
                     dim3(WG_BLOCKS), dim3(256), 0, stream, a)
#define LAUNCH_GATED(MT, NT)                                                  \
  case MT * 16 + NT:                                                          \
    if (gate == 2) LAUNCH_NARROW_AS(MT, NT, 2);                               \
    else LAUNCH_NARROW_AS(MT, NT, 1);                                         \
    break
#define LAUNCH_PLAIN(MT, NT)                                                  \
  case MT * 16 + NT:                                                          \
    LAUNCH_NARROW_AS(MT, NT, 0);                                              \
    break
  if (swiglu) {
    switch (tile) {
      LAUNCH_GATED(2, 4);
      LAUNCH_GATED(2, 5);
      LAUNCH_GATED(2, 8);
      LAUNCH_GATED(3, 4);
      LAUNCH_GATED(4, 4);
      LAUNCH_GATED(3, 5);
      LAUNCH_GATED(4, 5);
      LAUNCH_GATED(6, 4);
      LAUNCH_GATED(6, 5);
      LAUNCH_GATED(8, 4);
      LAUNCH_GATED(8, 5);
      default: TORCH_CHECK(false, "no such tile: ", tile);
    }
  } else {
    switch (tile) {
      LAUNCH_PLAIN(2, 4);
      LAUNCH_PLAIN(2, 8);
      LAUNCH_PLAIN(3, 4);
      LAUNCH_PLAIN(4, 4);
      LAUNCH_PLAIN(6, 4);
      LAUNCH_PLAIN(8, 4);
      LAUNCH_PLAIN(3, 8);
      LAUNCH_PLAIN(4, 8);
      LAUNCH_PLAIN(6, 6);
      LAUNCH_PLAIN(8, 6);
      default: TORCH_CHECK(false, "no such tile: ", tile);
    }
  }
#undef LAUNCH_PLAIN
#undef LAUNCH_GATED
#undef LAUNCH_NARROW_AS
  HIP_CHECK_KERNEL();
}

}  // namespace igw
