// y = x W^T for the tens of rows of x of a decode step or a short prompt,
// gfx950, bf16, products and sums in fp32 (16x16x32 matrix instructions).
//
// Bound by streaming W once from HBM.  A wave owns 16 rows of W and takes them
// from memory straight to registers, 512 bytes of each per slice of K, two
// slices on their way while one is multiplied; the slice's rows of x go
// through LDS once for the eight waves of a workgroup.  Loads take whole
// 128-byte lines, and workgroups start at different slices, waves at different
// lines: rows of W lie a multiple of 4 KB apart and would meet in the same
// memory channels (28672 x 4096, 16 rows: 52.0 us, with the starts apart 48.0,
// with whole lines as well 47.1).  A workgroup draws about 28 KB a microsecond
// whatever its depth, so the launch has to fill the compute units evenly.
//
// SWIGLU: a wave's 16 rows are eight gate rows and the up rows of the same
// outputs, and the result is silu(gate) * up of the fp32 sums.
//
// Measured, library and here (us, W cold; 16 / 32 / 48 / 64 rows): 28672 x 4096
// 65 56 64 55 and 48 48 50 52 (5.0 TB/s at 32 rows), as SwiGLU with the
// activation 70 58 70 58 and 47 48 50 52; 128256 x 4096 182 200 210 213 and
// 190 193 198 204; 4096 x 14336 27 34 40 41 and 30 31 33 35; 5120 x 17920
// 118 125 130 135 and 43 44 47 51.
#include <ATen/cuda/CUDAContext.h>
#include <torch/extension.h>

#include "common.h"

namespace igw {

typedef __attribute__((ext_vector_type(8))) __bf16 rg_bf16x8;
typedef __attribute__((ext_vector_type(4))) float rg_f32x4;
typedef __attribute__((ext_vector_type(4))) uint32_t rg_u32x4;

constexpr int RG_BK = 256;     // entries of a K slice
constexpr int RG_WAVES = 8;

struct RowsArgs {
  uint16_t* out;         // [M, N]
  float* part;           // [S, M, N] sums of a split K, or null
  const uint16_t* x;
  const uint16_t* w;
  const uint16_t* bias;
  int M, N, K;
  int64_t x_rs;
};

template <int MT, bool SWIGLU>
__global__ __launch_bounds__(64 * RG_WAVES, 2) void rows_gemm_kernel(
    RowsArgs a) {
  __shared__ __attribute__((aligned(1024))) uint16_t xs[3][MT * 16 * RG_BK];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, quad = lane >> 4;
  const int slices = a.K / RG_BK;
  const int s0 = slices * blockIdx.y / gridDim.y;
  const int last = slices * (blockIdx.y + 1) / gridDim.y - 1;
  const int rot = (blockIdx.x + (blockIdx.x >> 3)) % (last + 1 - s0);
  constexpr int COLS = SWIGLU ? 8 : 16;    // outputs of a wave
  const int n0 = (blockIdx.x * RG_WAVES + wave) * COLS;

  // Matrix row r of a wave's tile is this row of W; with SWIGLU four of them
  // are two gate rows and the up rows of the same two outputs.
  auto w_row = [&](int r) {
    return a.w + (int64_t)(SWIGLU ? min(n0 + (r >> 2) * 2 + (r & 1), a.N - 1) +
                                        ((r >> 1) & 1) * a.N
                                  : min(n0 + r, a.N - 1)) *
                     a.K;
  };
  // A load takes whole 128-byte lines: eight rows, eight lanes a row.
  const int piece = (quad + 4 * (r16 >> 3)) * 8;
  const uint16_t* w_lo = w_row(r16 & 7) + piece;
  const uint16_t* w_hi = w_row(8 + (r16 & 7)) + piece;
  // rows of x: 512 bytes of a row per 32 lanes, its 16-byte pieces permuted by
  // the row so that the 16 rows of a matrix operand lie in different banks
  constexpr int XR = MT * 8 / RG_WAVES;    // 16-byte pieces of x per lane
  const uint16_t* xp[XR];
#pragma unroll
  for (int i = 0; i < XR; ++i) {
    const int row = (i * RG_WAVES + wave) * 2 + (lane >> 5);
    xp[i] = a.x + min(row, a.M - 1) * a.x_rs + (lane & 31) * 8;
  }
  // a slice of x and of W, x first as it is waited for first; past the end the
  // last slice once more, so that the loop is the same to its end
  auto load = [&](rg_u32x4 (&xr)[XR], rg_u32x4 (&wr)[8], int sl) {
    int at = min(sl, last) + rot;
    at = at > last ? at - (last + 1 - s0) : at;
    const int k = at * RG_BK;
#pragma unroll
    for (int i = 0; i < XR; ++i)
      xr[i] = *reinterpret_cast<const rg_u32x4*>(xp[i] + k);
    asm volatile("" ::: "memory");
#pragma unroll
    for (int j = 0; j < 8; ++j)
      wr[j] = *reinterpret_cast<const rg_u32x4*>(
          (j & 1 ? w_hi : w_lo) + k + ((j / 2 + wave) & 3) * 64);
    asm volatile("" ::: "memory");
  };
  auto put_x = [&](const rg_u32x4 (&xr)[XR], uint16_t* s) {
#pragma unroll
    for (int i = 0; i < XR; ++i) {
      const int row = (i * RG_WAVES + wave) * 2 + (lane >> 5);
      *reinterpret_cast<rg_u32x4*>(
          s + row * RG_BK + ((lane & 31) ^ (row & 15)) * 8) = xr[i];
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  rg_f32x4 acc[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) acc[m] = rg_f32x4{0.f, 0.f, 0.f, 0.f};
  // Two loads hold rows 0..7 and 8..15 of the same line, first half in lanes
  // 0..7 of 16 and second half in 8..15; a matrix operand is one half of all
  // 16 rows, so the inner quarters change places.
  auto compute = [&](const rg_u32x4 (&wr)[8], const uint16_t* s) {
#pragma unroll
    for (int j = 0; j < 8; j += 2) {
      rg_u32x4 half[2];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        half[0][e] = __builtin_amdgcn_update_dpp(wr[j][e], wr[j + 1][e], 0x128,
                                                 0xf, 0xc, false);
        half[1][e] = __builtin_amdgcn_update_dpp(wr[j + 1][e], wr[j][e], 0x128,
                                                 0xf, 0x3, false);
      }
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          const int chunk =
              (((j / 2 + wave) & 3) * 8 + h * 4 + quad) ^ r16;
          const rg_bf16x8 xv = *reinterpret_cast<const rg_bf16x8*>(
              s + (m * 16 + r16) * RG_BK + chunk * 8);
          acc[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(rg_bf16x8, half[h]), xv, acc[m], 0, 0, 0);
        }
    }
  };

  // Past the barrier of put_x a slice's rows of x are there for every wave; the
  // buffer that they go to was last read two barriers before.
  rg_u32x4 x0[XR], x1[XR], x2[XR], w0[8], w1[8], w2[8];
  load(x0, w0, s0);
  load(x1, w1, s0 + 1);
  put_x(x0, xs[0]);
  for (int sl = s0;; sl += 3) {
    load(x2, w2, sl + 2);
    compute(w0, xs[0]);
    if (sl >= last) break;
    put_x(x1, xs[1]);
    load(x0, w0, sl + 3);
    compute(w1, xs[1]);
    if (sl + 1 >= last) break;
    put_x(x2, xs[2]);
    load(x1, w1, sl + 4);
    compute(w2, xs[2]);
    if (sl + 2 >= last) break;
    put_x(x0, xs[0]);
  }

#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const int row = m * 16 + r16;
    if (row >= a.M) continue;
    const rg_f32x4 y = acc[m];
    if (SWIGLU) {
      const int n = n0 + quad * 2;
      if (n >= a.N) continue;
      const uint32_t lo = f32_to_bf16(y[0] / (1.0f + __expf(-y[0])) * y[2]);
      const uint32_t hi = f32_to_bf16(y[1] / (1.0f + __expf(-y[1])) * y[3]);
      *reinterpret_cast<uint32_t*>(a.out + (int64_t)row * a.N + n) =
          lo | hi << 16;
    } else {
      const int n = n0 + quad * 4;
      if (n >= a.N) continue;
      if (a.part) {
        *reinterpret_cast<rg_f32x4*>(
            a.part + ((int64_t)blockIdx.y * a.M + row) * a.N + n) = y;
      } else {
        ushort4x o;
#pragma unroll
        for (int e = 0; e < 4; ++e)
          o.v[e] = f32_to_bf16(
              y[e] + (a.bias ? bf16_to_f32(a.bias[n + e]) : 0.0f));
        *reinterpret_cast<ushort4x*>(a.out + (int64_t)row * a.N + n) = o;
      }
    }
  }
}

// sum of the splits' parts, with the bias
__global__ __launch_bounds__(256) void rows_gemm_sum_kernel(RowsArgs a,
                                                            int S) {
  const int n = (blockIdx.x * 256 + threadIdx.x) * 4;
  const int row = blockIdx.y;
  if (n >= a.N) return;
  const float* p = a.part + (int64_t)row * a.N + n;
  const int64_t step = (int64_t)a.M * a.N;
  rg_f32x4 y = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
  for (int s = 0; s < S; ++s)
    y += *reinterpret_cast<const rg_f32x4*>(p + s * step);
  ushort4x o;
#pragma unroll
  for (int e = 0; e < 4; ++e)
    o.v[e] = f32_to_bf16(y[e] + (a.bias ? bf16_to_f32(a.bias[n + e]) : 0.0f));
  *reinterpret_cast<ushort4x*>(a.out + (int64_t)row * a.N + n) = o;
}

// In how many parts K is split for M rows of x and N outputs; 0: not taken.
//
// A workgroup holds a compute unit (registers), so the 256 of them have to be
// evenly used: 224 workgroups take 49.0 us for 28672 x 4096 where the library
// has 54.3, 280 take 108 for 35840 x 5120 where it has 96, 160 take 47 for
// 20480 x 4096 where it has 43 (40 rows).  Splitting K to get there pays for
// the sums only over a long K: 4096 x 14336 32.2 and 39.4, but 8192 x 8192
// 33.7 and 32.8, 8192 x 4096 22.8 and 18.8.  Up to 16 rows the library is
// ahead on 128256 x 4096 (182 and 190) and 4096 x 14336 (27 and 30); with the
// activation inside it is behind from 9 rows on (69 and 46).
int64_t rows_gemm_splits(int64_t M, int64_t N, int64_t K, bool swiglu) {
  if (M < (swiglu ? 9 : 17) || M > 64 || K < RG_BK || K % RG_BK != 0 ||
      N <= 0 || N % 4 != 0)
    return 0;
  const int64_t cols = RG_WAVES * (swiglu ? 8 : 16);
  const int64_t blocks = (N + cols - 1) / cols;
  const int64_t S = std::max<int64_t>(1, 256 / blocks);
  if (S > 1 && (swiglu || K < 3 * N || K < 6 * S * RG_BK)) return 0;
  const int64_t total = blocks * S, rounds = (total + 255) / 256;
  return total * 20 >= rounds * 256 * 17 ? S : 0;
}

void rows_gemm(torch::Tensor out, torch::Tensor x, torch::Tensor w,
               c10::optional<torch::Tensor> bias, bool swiglu) {
  TORCH_CHECK(x.is_cuda() && x.dim() == 2 && x.stride(1) == 1 &&
              x.dtype() == torch::kBFloat16 && w.dtype() == x.dtype() &&
              w.dim() == 2 && w.is_contiguous() && out.is_contiguous() &&
              out.dtype() == x.dtype());
  const int64_t M = x.size(0), K = x.size(1), N = out.size(1);
  const int64_t S = rows_gemm_splits(M, N, K, swiglu);
  TORCH_CHECK(S >= 1);
  TORCH_CHECK(out.size(0) == M && w.size(1) == K &&
              w.size(0) == (swiglu ? 2 * N : N) && x.stride(0) % 8 == 0);
  TORCH_CHECK((reinterpret_cast<uintptr_t>(x.data_ptr()) & 15) == 0 &&
              (reinterpret_cast<uintptr_t>(w.data_ptr()) & 15) == 0);
  if (bias.has_value())
    TORCH_CHECK(!swiglu && bias->dtype() == x.dtype() &&
                bias->is_contiguous() && bias->numel() == N);
  hipStream_t stream = at::cuda::getCurrentCUDAStream();
  const int64_t cols = RG_WAVES * (swiglu ? 8 : 16);
  const int64_t blocks = (N + cols - 1) / cols;
  torch::Tensor part;
  if (S > 1)
    part = torch::empty({S, M, N}, x.options().dtype(torch::kFloat32));
  RowsArgs a{(uint16_t*)out.data_ptr(),
             S > 1 ? part.data_ptr<float>() : nullptr,
             (const uint16_t*)x.data_ptr(),
             (const uint16_t*)w.data_ptr(),
             bias.has_value() ? (const uint16_t*)bias->data_ptr() : nullptr,
             (int)M, (int)N, (int)K, x.stride(0)};
  const dim3 grid(blocks, S);
#define LAUNCH_RG(MT, SW)                                                    \
  hipLaunchKernelGGL((rows_gemm_kernel<MT, SW>), grid, dim3(64 * RG_WAVES),  \
                     0, stream, a)
#define LAUNCH_RG_M(MT)                                                      \
  do {                                                                       \
    if (swiglu) LAUNCH_RG(MT, true);                                         \
    else LAUNCH_RG(MT, false);                                               \
  } while (0)
  if (M <= 16) LAUNCH_RG(1, true);
  else if (M <= 32) LAUNCH_RG_M(2);
  else if (M <= 48) LAUNCH_RG_M(3);
  else LAUNCH_RG_M(4);
#undef LAUNCH_RG_M
#undef LAUNCH_RG
  HIP_CHECK_KERNEL();
  if (S > 1) {
    hipLaunchKernelGGL(rows_gemm_sum_kernel, dim3((N / 4 + 255) / 256, M),
                       dim3(256), 0, stream, a, (int)S);
    HIP_CHECK_KERNEL();
  }
}

}  // namespace igw
