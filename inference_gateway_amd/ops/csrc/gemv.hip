// y = x W^T for the one to eight rows of x of a small decode step, gfx950,
// bf16.
//
// Bound by streaming W once from HBM.  x sits in LDS (staged by DMA while the
// first rows of W are on their way); a wave takes R rows of W at a time and
// reads 1 KB of a row per load, 64 lanes x 16 bytes, U loads per row in flight
// before the first is used: 16 waves per compute unit then keep 128 to 256 KB
// in flight, well past HBM latency times bandwidth.  Products and sums are
// fp32 (v_dot2_f32_bf16), a row's sum is completed across the wave.  Two
// workgroups of eight waves per compute unit stay for the whole of W, so x is
// staged 512 times at most.
//
// SWIGLU: the rows of a wave are the same rows of the gate and of the up half
// of W; the result is silu(gate) * up of the fp32 sums, one rounding where the
// separate activation has two.
//
// Measured, library and here (us; W cold, one row of x unless said): 6144 x
// 4096 14.2 and 10.7, 4096 x 4096 14.9 and 8.0, 28672 x 4096 with SwiGLU 69.1
// (two launches) and 38.6, 4096 x 14336 26.7 and 21.5, 128256 x 4096 187 and
// 161 (6.5 TB/s).  At 6 rows 15.5 / 14.0, 15.1 / 11.4, 69.8 / 41.8 and, 4 rows,
// 26.9 / 24.1; at 8 rows the library is level or ahead without the SwiGLU
// (15.6 / 16.6, 187 / 192; with it 69.9 / 50.8), so the line lies at 6 and 8.
#include <ATen/cuda/CUDAContext.h>
#include <torch/extension.h>

#include "common.h"

namespace igw {

typedef __attribute__((ext_vector_type(2))) __bf16 gv_bf16x2;

constexpr int GV_WAVES = 8;
constexpr int GV_ROWS = 2;              // of W per wave (SWIGLU: gate and up)
constexpr int64_t GV_MAX_X = 64 * 1024; // entries of x: 128 KB of LDS

template <int M, int R, bool SWIGLU>
__global__ __launch_bounds__(64 * GV_WAVES, 4) void gemv_kernel(
    uint16_t* __restrict__ out, const uint16_t* __restrict__ x,
    const uint16_t* __restrict__ w, const uint16_t* __restrict__ bias,
    int rows, int N, int K, int64_t x_rs) {
  extern __shared__ __attribute__((aligned(16))) uint16_t xs[];   // [M][K]
  // 16-byte loads in flight per row and lane: what 128 registers leave room
  // for (two workgroups per compute unit)
  constexpr int GV_U = M <= 3 ? 8 : 4;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int chunks = (K + 511) >> 9;
  constexpr int STEP = SWIGLU ? R / 2 : R;   // output columns per group
  const int groups = (N + STEP - 1) / STEP;
  const int stride = gridDim.x * GV_WAVES;

  uint4 buf[R][GV_U];
  auto load = [&](int grp, int c0) {
#pragma unroll
    for (int t = 0; t < R; ++t) {
      int n = SWIGLU ? grp * STEP + (t % STEP) : grp * STEP + t;
      n = min(n, N - 1) + (SWIGLU && t >= STEP ? N : 0);
      const uint16_t* row = w + (int64_t)n * K;
#pragma unroll
      for (int u = 0; u < GV_U; ++u) {
        const int k = ((c0 + u) << 9) + lane * 8;
        uint4 v = {0, 0, 0, 0};
        if (k < K) {
          typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
          const u32x4 q = __builtin_nontemporal_load(
              reinterpret_cast<const u32x4*>(row + k));
          v = {q.x, q.y, q.z, q.w};
        }
        buf[t][u] = v;
      }
    }
  };
  // x to LDS, linearly, all of it in flight at once; a 1 KB piece may cross
  // rows, lanes past the end repeat the last entries
  const int total = M * K;
  for (int base = wave * 512; base < total; base += GV_WAVES * 512) {
    const int i = min(base + lane * 8, total - 8);
    const int m = i / K;
    __builtin_amdgcn_global_load_lds(
        reinterpret_cast<const uint32_t*>(x + min(m, rows - 1) * x_rs +
                                          (i - m * K)),
        reinterpret_cast<uint32_t*>(xs + base), 16, 0, 0);
  }
  int grp = blockIdx.x * GV_WAVES + wave;
  // the first rows of W are on their way meanwhile
  if (grp < groups) load(grp, 0);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();

  for (; grp < groups; grp += stride) {
    float acc[R][M];
#pragma unroll
    for (int t = 0; t < R; ++t)
#pragma unroll
      for (int m = 0; m < M; ++m) acc[t][m] = 0.0f;
    for (int c0 = 0; c0 < chunks; c0 += GV_U) {
      if (!(c0 == 0 && grp < stride)) load(grp, c0);
#pragma unroll
      for (int u = 0; u < GV_U; ++u) {
        const int k = ((c0 + u) << 9) + lane * 8;
        if (((c0 + u) << 9) >= K) break;
        const int kx = k < K ? k : 0;   // W is zero there
#pragma unroll
        for (int m = 0; m < M; ++m) {
          const uint4 xv = *reinterpret_cast<const uint4*>(xs + m * K + kx);
#pragma unroll
          for (int t = 0; t < R; ++t)
#pragma unroll
            for (int e = 0; e < 4; ++e)
              acc[t][m] = __builtin_amdgcn_fdot2_f32_bf16(
                  __builtin_bit_cast(gv_bf16x2, (&buf[t][u].x)[e]),
                  __builtin_bit_cast(gv_bf16x2, (&xv.x)[e]), acc[t][m],
                  false);
        }
      }
    }
#pragma unroll
    for (int t = 0; t < R; ++t)
#pragma unroll
      for (int m = 0; m < M; ++m) acc[t][m] = wave_reduce_sum(acc[t][m]);
    if (lane == 0) {
#pragma unroll
      for (int t = 0; t < STEP; ++t) {
        const int n = grp * STEP + t;
        if (n < N) {
#pragma unroll
          for (int m = 0; m < M; ++m) {
            if (m >= rows) break;
            float y = acc[t][m];
            if (SWIGLU) y = y / (1.0f + __expf(-y)) * acc[t + STEP][m];
            else if (bias) y += bf16_to_f32(bias[n]);
            out[(int64_t)m * N + n] = f32_to_bf16(y);
          }
        }
      }
    }
  }
}

// Whether gemv takes M rows of x with K entries against this many outputs.
bool gemv_fits(int64_t M, int64_t K, bool swiglu) {
  const int64_t mp = M <= 4 ? M : M <= 6 ? 6 : 8;
  return M >= 1 && M <= (swiglu ? 8 : 6) && K >= 8 && K % 8 == 0 &&
         mp * K <= GV_MAX_X;
}

// out [M, N] = x [M, K] W^T (+ bias [N]); swiglu: W [2 N, K], out = silu(x
// Wg^T) * (x Wu^T).  Rows of x and W 16-byte aligned.
void gemv(torch::Tensor out, torch::Tensor x, torch::Tensor w,
          c10::optional<torch::Tensor> bias, bool swiglu) {
  TORCH_CHECK(x.is_cuda() && x.dim() == 2 && x.stride(1) == 1 &&
              x.dtype() == torch::kBFloat16 && w.dtype() == x.dtype() &&
              w.dim() == 2 && w.is_contiguous() && out.is_contiguous() &&
              out.dtype() == x.dtype());
  const int64_t M = x.size(0), K = x.size(1), N = out.size(1);
  TORCH_CHECK(gemv_fits(M, K, swiglu) && out.size(0) == M && w.size(1) == K &&
              w.size(0) == (swiglu ? 2 * N : N) && x.stride(0) % 8 == 0);
  TORCH_CHECK((reinterpret_cast<uintptr_t>(x.data_ptr()) & 15) == 0 &&
              (reinterpret_cast<uintptr_t>(w.data_ptr()) & 15) == 0);
  const uint16_t* b = nullptr;
  if (bias.has_value()) {
    TORCH_CHECK(!swiglu && bias->dtype() == x.dtype() &&
                bias->is_contiguous() && bias->numel() == N);
    b = (const uint16_t*)bias->data_ptr();
  }
  if (N == 0) return;
  hipStream_t stream = at::cuda::getCurrentCUDAStream();
  const int64_t mp = M <= 4 ? M : M <= 6 ? 6 : 8;
  const size_t shmem = (size_t)(mp * K + 511) / 512 * 1024;
  const int64_t step = swiglu ? GV_ROWS / 2 : GV_ROWS;
  const int64_t need = ((N + step - 1) / step + GV_WAVES - 1) / GV_WAVES;
  const dim3 grid(std::min<int64_t>(need, 512));
#define LAUNCH_GV(MV)                                                         \
  do {                                                                        \
    auto kern = swiglu ? gemv_kernel<MV, GV_ROWS, true>                       \
                       : gemv_kernel<MV, GV_ROWS, false>;                     \
    if (shmem > 64 * 1024)                                                    \
      TORCH_CHECK(hipFuncSetAttribute(                                        \
                      (const void*)kern,                                      \
                      hipFuncAttributeMaxDynamicSharedMemorySize,             \
                      (int)shmem) == hipSuccess);                             \
    hipLaunchKernelGGL(kern, grid, dim3(64 * GV_WAVES), shmem, stream,        \
                       (uint16_t*)out.data_ptr(),                             \
                       (const uint16_t*)x.data_ptr(),                         \
                       (const uint16_t*)w.data_ptr(), b, (int)M, (int)N,      \
                       (int)K, x.stride(0));                                  \
  } while (0)
  switch (mp) {
    case 1: LAUNCH_GV(1); break;
    case 2: LAUNCH_GV(2); break;
    case 3: LAUNCH_GV(3); break;
    case 4: LAUNCH_GV(4); break;
    case 6: LAUNCH_GV(6); break;
    default: LAUNCH_GV(8); break;
  }
#undef LAUNCH_GV
  HIP_CHECK_KERNEL();
}

}  // namespace igw
