// y = x W^T for the one to eight rows of x of a small decode step, gfx950,
// bf16.
//
// Bound by streaming W once from HBM.  x sits in LDS (staged by DMA while the
// first rows of W are on their way); a wave takes R rows of W at a time and
// reads 1 KB of a row per load, 64 lanes x 16 bytes, U loads per row in flight
// before the first is used.  Products and sums are fp32 (v_dot2_f32_bf16), a
// row's sum is completed across the wave.  Workgroups of eight waves stay for
// the whole of W, so x is staged 512 times at most; up to 80 KB of x two of
// them share a compute unit and keep 128 KB in flight, well past HBM latency
// times bandwidth, with more x one keeps half of that.
//
// GATE: the rows of a wave are the same rows of the gate and of the up half of W;
// the result is act(gate) * up of the fp32 sums, one rounding where the separate
// activation has two.
//
// Measured, library and here (us; W cold, one row of x unless said): 6144 x
// 4096 14.2 and 10.7, 4096 x 4096 14.9 and 8.0, 28672 x 4096 with SwiGLU 69.1
// (two launches) and 38.6, 4096 x 14336 26.7 and 21.5, 128256 x 4096 187 and
// 161 (6.5 TB/s).  gemv_ahead says where the library takes over.
#include <ATen/cuda/CUDAContext.h>
#include <c10/cuda/CUDAGuard.h>
#include <torch/extension.h>

#include "common.h"

namespace igw {

typedef __attribute__((ext_vector_type(2))) __bf16 gv_bf16x2;

constexpr int GV_WAVES = 8;
constexpr int GV_ROWS = 2;              // of W per wave (SWIGLU: gate and up)
constexpr int64_t GV_MAX_X = 64 * 1024; // entries of x: 128 KB of LDS

// A wave's walk over the row groups first, first + stride, ... below `groups`
// of W [N (or 2 N), K] against the M rows of x in LDS.  stage() puts x there,
// after the first rows of W have been asked for (ahead() is called before); store(n,
// sums of W row n, of its up row) is called by lane 0.
// U is the 16-byte loads in flight per row and lane (gemv_deep says when eight).
// TAIL: K is not a multiple of the 512 entries of a load, and lanes lie past a
// row's end.
template <int M, int R, bool SWIGLU, bool TAIL, int U, class Stage, class Store,
          class Ahead>
DEVINLINE void gemv_walk(const uint16_t* xs, const uint16_t* __restrict__ w,
                         int N, int K, int first, int groups, int stride,
                         Stage stage, Store store, Ahead ahead) {
  const int lane = threadIdx.x & 63;
  const int chunks = (K + 511) >> 9;
  constexpr int STEP = SWIGLU ? R / 2 : R;   // output columns per group

  uint4 buf[R][U];
  auto load = [&](int grp, int c0) {
#pragma unroll
    for (int t = 0; t < R; ++t) {
      int n = SWIGLU ? grp * STEP + (t % STEP) : grp * STEP + t;
      n = min(n, N - 1) + (SWIGLU && t >= STEP ? N : 0);
      const uint16_t* row = w + (int64_t)n * K;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k = ((c0 + u) << 9) + lane * 8;
        uint4 v = {0, 0, 0, 0};
        if (TAIL ? k < K : (c0 + u) << 9 < K) {
          typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
          const u32x4 q = __builtin_nontemporal_load(
              reinterpret_cast<const u32x4*>(row + k));
          v = {q.x, q.y, q.z, q.w};
        }
        buf[t][u] = v;
      }
    }
  };
  ahead();
  if (first < groups) load(first, 0);
  stage();

  for (int grp = first; grp < groups; grp += stride) {
    float acc[R][M];
#pragma unroll
    for (int t = 0; t < R; ++t)
#pragma unroll
      for (int m = 0; m < M; ++m) acc[t][m] = 0.0f;
    for (int c0 = 0; c0 < chunks; c0 += U) {
      if (c0 > 0 || grp > first) load(grp, c0);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k = ((c0 + u) << 9) + lane * 8;
        if (((c0 + u) << 9) >= K) break;
        if (!TAIL || k < K) {   // past the end nothing is added, not even 0 * x
#pragma unroll
          for (int m = 0; m < M; ++m) {
            const uint4 xv = *reinterpret_cast<const uint4*>(xs + m * K + k);
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
    }
#pragma unroll
    for (int t = 0; t < R; ++t)
#pragma unroll
      for (int m = 0; m < M; ++m) acc[t][m] = wave_reduce_sum(acc[t][m]);
    if (lane == 0) {
#pragma unroll
      for (int t = 0; t < STEP; ++t)
        if (grp * STEP + t < N)
          store(grp * STEP + t, acc[t], acc[SWIGLU ? t + STEP : t]);
    }
  }
}

// Rows of x to LDS, linearly, all of it in flight at once; row(m) is the m-th
// row.  A 1 KB piece may cross rows, lanes past the end repeat the last
// entries.
template <class Row>
DEVINLINE void gemv_stage(uint16_t* xs, int total, int K, Row row) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  for (int base = wave * 512; base < total; base += GV_WAVES * 512) {
    const int i = min(base + lane * 8, total - 8);
    const int m = i / K;
    __builtin_amdgcn_global_load_lds(
        reinterpret_cast<const uint32_t*>(row(m) + (i - m * K)),
        reinterpret_cast<uint32_t*>(xs + base), 16, 0, 0);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
}

template <int M, int R, int GATE, bool TAIL, int U>
__global__ __launch_bounds__(64 * GV_WAVES, 4) void gemv_kernel(
    uint16_t* __restrict__ out, const uint16_t* __restrict__ x,
    const uint16_t* __restrict__ w, const uint16_t* __restrict__ bias,
    int rows, int N, int K, int64_t x_rs) {
  extern __shared__ __attribute__((aligned(16))) uint16_t xs[];   // [M][K]
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  constexpr bool SWIGLU = GATE != 0;
  constexpr int STEP = SWIGLU ? R / 2 : R;
  gemv_walk<M, R, SWIGLU, TAIL, U>(
      xs, w, N, K, blockIdx.x * GV_WAVES + wave, (N + STEP - 1) / STEP,
      gridDim.x * GV_WAVES,
      [&] {
        gemv_stage(xs, M * K, K,
                   [&](int m) { return x + min(m, rows - 1) * x_rs; });
      },
      [&](int n, const float* a, const float* up) {
#pragma unroll
        for (int m = 0; m < M; ++m) {
          if (m >= rows) break;
          float y = a[m];
          if (SWIGLU) y = gate_act<GATE>(y) * up[m];
          else if (bias) y += bf16_to_f32(bias[n]);
          out[(int64_t)m * N + n] = f32_to_bf16(y);
        }
      },
      [] {});
}

// The same with the norm before it: x = rmsnorm(residual + delta) * weight, rows of
// K entries.  Every workgroup norms for itself (24 KB a row from L2, 512 times) while
// its first rows of W are on their way, which takes longer; a launch of the norm's
// own is 2.5 to 3 us of a decode step, twice a layer.  The first workgroup writes the
// new residual, to other memory, as the others still read the old one.
// A thread has 8 entries of a row in each of IT turns; sums wait in LDS.
struct GemvNorm {
  const uint16_t *delta, *residual, *weight;   // delta may be null
  uint16_t* sum;                               // residual + delta, where there is one
  float eps;
};

template <int M, int R, int GATE, int IT, int U>
__global__ __launch_bounds__(64 * GV_WAVES, 4) void gemv_norm_kernel(
    uint16_t* __restrict__ out, GemvNorm g, const uint16_t* __restrict__ w,
    const uint16_t* __restrict__ bias, int rows, int N, int K) {
  extern __shared__ __attribute__((aligned(16))) uint16_t xs[];   // [M][K]
  __shared__ float red[GV_WAVES][M];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  constexpr bool SWIGLU = GATE != 0;
  constexpr int STEP = SWIGLU ? R / 2 : R;
  // Loads return in order: what the norm needs is asked for before W where it fits
  // the registers, else two or three rows at a time behind it.
  constexpr bool AHEAD = M * IT <= 4;
  constexpr int G = M <= 4 && (AHEAD || M == 3) ? M : 2, TURNS = AHEAD ? IT : 1;
  static_assert(M % G == 0);
  ushort8 s[TURNS][G], d[TURNS][G];
  auto fetch = [&](int it, int m0, int t) {
    const int i = (it * 64 * GV_WAVES + threadIdx.x) * 8;
    if (i >= K) return;
#pragma unroll
    for (int m = 0; m < G; ++m) {
      const int64_t at = (int64_t)min(m0 + m, rows - 1) * K + i;
      s[t][m] = *reinterpret_cast<const ushort8*>(g.residual + at);
      if (g.delta) d[t][m] = *reinterpret_cast<const ushort8*>(g.delta + at);
    }
  };
  auto ahead = [&] {
    if (!AHEAD) return;
#pragma unroll
    for (int it = 0; it < IT; ++it) fetch(it, 0, it);
    asm volatile("" ::: "memory");
  };
  auto stage = [&] {
    float ss[M];
#pragma unroll
    for (int m = 0; m < M; ++m) ss[m] = 0.0f;
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      const int i = (it * 64 * GV_WAVES + threadIdx.x) * 8;
#pragma unroll
      for (int m0 = 0; m0 < M; m0 += G) {
        const int t = AHEAD ? it : 0;
        if (!AHEAD) fetch(it, m0, 0);
        if (i < K) {
#pragma unroll
          for (int m = 0; m < G; ++m) {
            ushort8& v = s[t][m];
            if (g.delta) {
#pragma unroll
              for (int j = 0; j < 8; ++j)
                v.v[j] = f32_to_bf16(bf16_to_f32(d[t][m].v[j]) +
                                     bf16_to_f32(v.v[j]));
              if (blockIdx.x == 0 && m0 + m < rows)
                *reinterpret_cast<ushort8*>(g.sum + (int64_t)(m0 + m) * K + i) =
                    v;
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) {
              const float f = bf16_to_f32(v.v[j]);
              ss[m0 + m] += f * f;
            }
            *reinterpret_cast<ushort8*>(xs + (m0 + m) * K + i) = v;
          }
        }
        asm volatile("" ::: "memory");
      }
    }
#pragma unroll
    for (int m = 0; m < M; ++m) {
      ss[m] = wave_reduce_sum(ss[m]);
      if (lane == 0) red[wave][m] = ss[m];
    }
    __syncthreads();
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      const int i = (it * 64 * GV_WAVES + threadIdx.x) * 8;
      if (i >= K) continue;
      const ushort8 wv = *reinterpret_cast<const ushort8*>(g.weight + i);
#pragma unroll 2
      for (int m = 0; m < M; ++m) {
        float all = 0.0f;
#pragma unroll
        for (int v = 0; v < GV_WAVES; ++v) all += red[v][m];
        const float inv = rsqrtf(all / K + g.eps);
        ushort8 o = *reinterpret_cast<const ushort8*>(xs + m * K + i);
#pragma unroll
        for (int j = 0; j < 8; ++j)
          o.v[j] = f32_to_bf16(bf16_to_f32(o.v[j]) * inv *
                               bf16_to_f32(wv.v[j]));
        *reinterpret_cast<ushort8*>(xs + m * K + i) = o;
      }
    }
    __syncthreads();
  };
  gemv_walk<M, R, SWIGLU, false, U>(
      xs, w, N, K, blockIdx.x * GV_WAVES + wave, (N + STEP - 1) / STEP,
      gridDim.x * GV_WAVES, stage, [&](int n, const float* a, const float* up) {
#pragma unroll
        for (int m = 0; m < M; ++m) {
          if (m >= rows) break;
          float y = a[m];
          if (SWIGLU) y = gate_act<GATE>(y) * up[m];
          else if (bias) y += bf16_to_f32(bias[n]);
          out[(int64_t)m * N + n] = f32_to_bf16(y);
        }
      },
      ahead);
}

// ---------------------------------------------------------------------------
// Experts of a small decode step.  Assignment a = t K + k sends token t to
// expert idx[a]; an expert without a token is not read (a batched product over
// all experts reads every one of them).  The row groups of the experts that have
// one, one after the other, are cut evenly for as many workgroups as the chip
// holds: which experts those are stands in the list on the device.  The
// assignments of an expert are found from the list, in passes of as many rows
// as LDS holds (more than one pass only where many tokens meet wide rows).
//
// SWIGLU: out [T K, N] bf16 = silu(x_t Wg^T) * (x_t Wu^T).  Otherwise: in is
// [T K, K] and sums [T K, N] fp32 = weight_a * in_a W^T.
//
// Bound by streaming the chosen experts' weights.  Measured from the hidden
// rows to the combined ones, 8 experts of 14336 x 4096 in bf16, two per token
// (us; batched products over the padded rows of all experts, a fixed number of
// workgroups for each expert, and the even cut): 1 token 588, 120 and 113, 2 of
// four experts 589, 235 and 216, 5 of six or seven 600, 375 / 405 and 324 / 376
// (6.5 TB/s), 8 of eight 612, 470 and 430.  A fixed number leaves compute units idle
// or with one workgroup too many.  Eight loads a row in flight instead of four do
// not fit the registers beside the passes of up to eight rows (141 for the 113).
constexpr int GV_ASSIGN = 64;   // assignments a step may have

template <bool SWIGLU, bool TAIL>
__global__ __launch_bounds__(64 * GV_WAVES, 4) void expert_gemv_kernel(
    uint16_t* __restrict__ out, float* __restrict__ sums,
    const uint16_t* __restrict__ in, const uint16_t* __restrict__ w,
    const int32_t* __restrict__ idx, const float* __restrict__ weight,
    int assigned, int experts, int top_k, int N, int K, int64_t in_rs,
    int max_rows) {
  extern __shared__ __attribute__((aligned(16))) uint16_t xs[];
  __shared__ int list[GV_ASSIGN];
  constexpr int STEP = SWIGLU ? GV_ROWS / 2 : GV_ROWS;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // the experts in the order of their first assignments
  int own = lane < assigned ? idx[lane] : -1;
  if (own >= experts) own = -1;   // nobody's
  uint64_t firsts = 0;
  for (int a = 0; a < assigned; ++a) {
    const int e = __builtin_amdgcn_readlane(own, a);
    if (__builtin_ctzll(__ballot(own == e)) == a && e >= 0) firsts |= 1ull << a;
  }
  // of expert e: its assignments, and the passes over its rows
  auto tokens = [&](int e) { return __ballot(own == e); };
  auto passes = [&](uint64_t all) {
    return (__popcll(all) + max_rows - 1) / max_rows;
  };
  auto expert = [&](uint64_t left) {
    return __builtin_amdgcn_readlane(own, __builtin_ctzll(left));
  };
  const int groups = (N + STEP - 1) / STEP;
  int64_t total = 0;
  for (uint64_t left = firsts; left; left &= left - 1)
    total += (int64_t)passes(tokens(expert(left))) * groups;
  // this workgroup's share of the row groups, each counted once a pass
  int64_t from = total * blockIdx.x / gridDim.x;
  int64_t to = total * (blockIdx.x + 1) / gridDim.x;

  for (uint64_t left = firsts; left && to > 0; left &= left - 1) {
    const int e = expert(left);
    const uint64_t all = tokens(e);
    const int count = __popcll(all), p = passes(all);
    const int first = (int)(min(max(from, (int64_t)0), (int64_t)groups * p) / p);
    const int end = (int)(min(to, (int64_t)groups * p) / p);
    from -= (int64_t)groups * p;
    to -= (int64_t)groups * p;
    if (first >= end) continue;
    const bool mine = own == e;
    if (wave == 0 && mine)
      list[__popcll(all & ((1ull << lane) - 1))] = lane;
    __syncthreads();
    const uint16_t* we = w + (int64_t)e * (SWIGLU ? 2 * N : N) * K;

    for (int at = 0; at < count; at += max_rows) {
      const int rows = min(max_rows, count - at);
      auto pass = [&](auto m_) {
        constexpr int M = decltype(m_)::value;
        gemv_walk<M, GV_ROWS, SWIGLU, TAIL, 4>(
            xs, we, N, K, first + wave, end, GV_WAVES,
            [&] {
              gemv_stage(xs, rows * K, K, [&](int m) {
                const int a = list[at + m];
                return in + (SWIGLU ? a / top_k : a) * in_rs;
              });
            },
            [&](int n, const float* y, const float* up) {
#pragma unroll
              for (int m = 0; m < M; ++m) {
                if (m >= rows) break;
                const int64_t a = list[at + m];
                if (SWIGLU)
                  out[a * N + n] =
                      f32_to_bf16(gate_act<1>(y[m]) * up[m]);
                else
                  sums[a * N + n] = weight[a] * y[m];
              }
            },
            [] {});
      };
      if (rows == 1) pass(std::integral_constant<int, 1>{});
      else if (rows == 2) pass(std::integral_constant<int, 2>{});
      else if (rows <= 4) pass(std::integral_constant<int, 4>{});
      else pass(std::integral_constant<int, 8>{});
      __syncthreads();   // x and the list are replaced by the next pass
    }
  }
}

__global__ void expert_combine_kernel(uint16_t* __restrict__ out,
                                      const float* __restrict__ sums, int N,
                                      int top_k) {
  const int64_t t = blockIdx.y;
  const int n = (blockIdx.x * blockDim.x + threadIdx.x) * 4;
  if (n >= N) return;
  float4 y = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int k = 0; k < top_k; ++k) {
    const float4 v =
        *reinterpret_cast<const float4*>(sums + (t * top_k + k) * N + n);
    y.x += v.x;
    y.y += v.y;
    y.z += v.z;
    y.w += v.w;
  }
  ushort4x o;
  o.v[0] = f32_to_bf16(y.x);
  o.v[1] = f32_to_bf16(y.y);
  o.v[2] = f32_to_bf16(y.z);
  o.v[3] = f32_to_bf16(y.w);
  *reinterpret_cast<ushort4x*>(out + t * N + n) = o;
}

// Most tokens that moe_few takes.  With more of them the experts that many
// tokens share are read once per pass: at 16 tokens 540 us against 594 where
// the router spreads them and 714 where it does not, at 8 it is ahead either
// way (426 to 460 against 612).
constexpr int64_t GV_MOE_TOKENS = 8;

bool moe_few_fits(int64_t T, int64_t top_k, int64_t D, int64_t F) {
  return T >= 1 && T <= GV_MOE_TOKENS && T * top_k <= GV_ASSIGN &&
         D >= 8 && F >= 8 && D % 8 == 0 && F % 8 == 0 && D <= GV_MAX_X &&
         F <= GV_MAX_X;
}

// out [T, D] = sum over a token's experts of weight * down(silu(gate) * up):
// x [T, D], gate_up [E, 2 F, D], down [E, D, F], idx and weight [T, K] (int32,
// fp32).
void moe_few(torch::Tensor out, torch::Tensor x, torch::Tensor gate_up,
             torch::Tensor down, torch::Tensor idx, torch::Tensor weight) {
  TORCH_CHECK(x.is_cuda() && x.dim() == 2 && x.is_contiguous() &&
              gate_up.dim() == 3 && down.dim() == 3 && idx.dim() == 2);
  for (auto* t : {&out, &gate_up, &down, &idx, &weight})
    TORCH_CHECK(t->device() == x.device(), "tensors on different devices");
  for (auto* t : {&out, &x, &gate_up, &down})
    TORCH_CHECK(t->dtype() == torch::kBFloat16 && t->is_contiguous() &&
                (reinterpret_cast<uintptr_t>(t->data_ptr()) & 15) == 0);
  const int64_t T = x.size(0), D = x.size(1), E = gate_up.size(0);
  const int64_t F = down.size(2), top_k = idx.size(1);
  TORCH_CHECK(moe_few_fits(T, top_k, D, F) && out.sizes() == x.sizes() &&
              gate_up.size(1) == 2 * F && gate_up.size(2) == D &&
              down.size(0) == E && down.size(1) == D && idx.size(0) == T);
  TORCH_CHECK(idx.dtype() == torch::kInt32 && idx.is_contiguous() &&
              weight.dtype() == torch::kFloat32 && weight.is_contiguous() &&
              weight.numel() == T * top_k);
  const int64_t n = T * top_k;
  const at::cuda::CUDAGuard guard(x.device());
  auto act = torch::empty({n, F}, x.options());
  auto sums = torch::empty({n, D}, x.options().dtype(torch::kFloat32));
  hipStream_t stream = at::cuda::getCurrentCUDAStream();
  const int64_t cus =
      at::cuda::getCurrentDeviceProperties()->multiProcessorCount;
  auto launch = [&](auto kern, int64_t K, int64_t cols, int64_t group,
                    const torch::Tensor& in, const torch::Tensor& w) {
    // a power of two, as the kernel rounds the rows of a pass up to one
    int64_t rows = 1;
    while (rows < std::min<int64_t>(T, 8) && 2 * rows * K <= GV_MAX_X)
      rows *= 2;
    const size_t shmem = (size_t)(rows * K + 511) / 512 * 1024;
    if (shmem > 64 * 1024)
      TORCH_CHECK(hipFuncSetAttribute(
                      (const void*)kern,
                      hipFuncAttributeMaxDynamicSharedMemorySize,
                      (int)shmem) == hipSuccess);
    // as many as are there at once, no more than there is work for
    const int64_t need =
        (cols / group + GV_WAVES) / GV_WAVES * std::min(E, n);
    const int64_t fit = shmem > 80 * 1024 - 256 ? cus : 2 * cus;
    hipLaunchKernelGGL(kern, dim3(std::min(fit, need)),
                       dim3(64 * GV_WAVES), shmem, stream,
                       (uint16_t*)act.data_ptr(), sums.data_ptr<float>(),
                       (const uint16_t*)in.data_ptr(),
                       (const uint16_t*)w.data_ptr(),
                       (const int32_t*)idx.data_ptr(),
                       (const float*)weight.data_ptr(), (int)n, (int)E, (int)top_k,
                       (int)cols, (int)K, K, (int)rows);
    HIP_CHECK_KERNEL();
  };
  launch(D % 512 ? expert_gemv_kernel<true, true>
                 : expert_gemv_kernel<true, false>,
         D, F, GV_ROWS / 2, x, gate_up);
  launch(F % 512 ? expert_gemv_kernel<false, true>
                 : expert_gemv_kernel<false, false>,
         F, D, GV_ROWS, act, down);
  hipLaunchKernelGGL(expert_combine_kernel, dim3((D / 4 + 255) / 256, T),
                     dim3(256), 0, stream, (uint16_t*)out.data_ptr(),
                     sums.data_ptr<float>(), (int)D, (int)top_k);
  HIP_CHECK_KERNEL();
}

// Whether gemv can take M rows of x with K entries.
bool gemv_fits(int64_t M, int64_t K, bool swiglu) {
  const int64_t mp = M <= 4 ? M : M <= 6 ? 6 : 8;
  return M >= 1 && M <= (swiglu ? 8 : 6) && K >= 8 && K % 8 == 0 &&
         mp * K <= GV_MAX_X;
}

// Whether gemv is ahead of the library for M rows of x and W [N, K] (2 F rows
// with swiglu, where the library has a second launch).
//
// Against it stand three costs that a long stream of W hides: the sums across
// the wave, 6 steps per row of x and row of W, which a short K does not pay
// for; x in LDS, of which the compute unit holds two copies only up to 80 KB;
// and a wave's start, which few rows of W do not share.  All three grow with
// M.  Measured at 893 sizes, 8 to 128256 x 64 to 17920, one to eight rows (us,
// gemv and library): short K, 65536 x 256 one row 15.8 and 10.4, 4 rows 27.2
// and 10.4, 14336 x 1024 6 rows 12.7 and 9.2, 32000 x 1024 8 rows with SwiGLU
// 27.5 and 22.9; much x, 8192 x 8192 6 rows 34.1 and 28.7, 5120 x 5120 16.7 and
// 13.7; few rows of W, 256 x 8192 6 rows 12.4 and 8.7.  The other way, within
// the lines below: 4096 x 4096 6 rows 11.1 and 14.3, 4096 x 14336 4 rows 24.2
// and 26.0, 28672 x 4096 with SwiGLU 8 rows 47 and 68.  On this side gemv is at
// most 4 % behind, but for 10 sizes of 5 to 37 us where it is 7 to 11 % (three
// and four rows).
bool gemv_ahead(int64_t M, int64_t N, int64_t K, bool swiglu) {
  const bool wide = N >= 10240;
  if (swiglu && M <= 2) return true;
  if (swiglu && M <= 4) return K >= 512 || N <= 8192;
  if (swiglu && M <= 6)
    return K <= 5120 ? K >= 1280 || (K >= 384 && N <= 4096) : wide;
  if (M <= 2) return K >= 768 || N <= K * K / (4 * M);
  if (M <= 4) {
    if (K > 5120) return wide || (N >= 1024 && (M == 3 || K > 8192));
    return K >= 1280 || (K >= 128 && N <= 256) ||
           (M == 3 && K >= 512 && N <= 4096);
  }
  return (N >= 22016 && K >= 2048) ||
         (N >= 14336 && K >= 2560 && K <= 6144) ||
         (N >= 512 && N <= 4096 && K >= (swiglu ? 1024 : 1536) && K <= 4096);
}

// Whether eight loads a row are in flight instead of four, for up to three rows of
// x (more of them leave no registers).  Four are up to 8 % ahead at most sizes;
// eight where five to seven make a whole row, and where rows of W lie a multiple of
// 16 KB apart, of which fewer loads reach fewer of the memory channels (us, four and
// eight, one row: 5120 x 5120 12.3 and 12.9, 7680 x 5120 14.4 and 15.2; 2560 wide 2
// to 11 % apart, 8192 x 8192 29.4 and 26.8, 10240 x 8192 35.7 and 32.6, 16384 wide 1
// to 17 %).  At 4096 wide up to 2048 outputs would want eight too (5.9 and 5.5).
static bool gemv_deep(int64_t M, int64_t K) {
  return M <= 3 && (K % 8192 == 0 || (K > 2048 && K <= 3584));
}

// out [M, N] = x [M, K] W^T (+ bias [N]); swiglu: W [2 N, K], out = silu(x
// Wg^T) * (x Wu^T).  Rows of x and W 16-byte aligned.
void gemv(torch::Tensor out, torch::Tensor x, torch::Tensor w,
          c10::optional<torch::Tensor> bias, int64_t gate) {
  const bool swiglu = gate != 0;
  TORCH_CHECK(gate >= 0 && gate <= 2);
  TORCH_CHECK(x.is_cuda() && x.dim() == 2 && x.stride(1) == 1 &&
              x.dtype() == torch::kBFloat16 && w.dtype() == x.dtype() &&
              w.dim() == 2 && w.is_contiguous() && out.is_contiguous() &&
              out.dtype() == x.dtype());
  const int64_t M = x.size(0), K = x.size(1), N = out.size(1);
  TORCH_CHECK(gemv_fits(M, K, swiglu) && out.size(0) == M && w.size(1) == K &&
              w.size(0) == (swiglu ? 2 * N : N) && x.stride(0) % 8 == 0);
  TORCH_CHECK(w.device() == x.device() && out.device() == x.device(),
              "tensors on different devices");
  TORCH_CHECK((reinterpret_cast<uintptr_t>(x.data_ptr()) & 15) == 0 &&
              (reinterpret_cast<uintptr_t>(w.data_ptr()) & 15) == 0);
  const uint16_t* b = nullptr;
  if (bias.has_value()) {
    TORCH_CHECK(!swiglu && bias->dtype() == x.dtype() &&
                bias->device() == x.device() && bias->is_contiguous() &&
                bias->numel() == N);
    b = (const uint16_t*)bias->data_ptr();
  }
  if (N == 0) return;
  const at::cuda::CUDAGuard guard(x.device());
  hipStream_t stream = at::cuda::getCurrentCUDAStream();
  const int64_t mp = M <= 4 ? M : M <= 6 ? 6 : 8;
  const size_t shmem = (size_t)(mp * K + 511) / 512 * 1024;
  const int64_t step = swiglu ? GV_ROWS / 2 : GV_ROWS;
  const int64_t need = ((N + step - 1) / step + GV_WAVES - 1) / GV_WAVES;
  const dim3 grid(std::min<int64_t>(need, 512));
#define GV_KERNEL(MV, TAIL, U)                                                \
  (gate == 2   ? gemv_kernel<MV, GV_ROWS, 2, TAIL, U>                         \
   : gate == 1 ? gemv_kernel<MV, GV_ROWS, 1, TAIL, U>                         \
               : gemv_kernel<MV, GV_ROWS, 0, TAIL, U>)
#define LAUNCH_GV(MV, U)                                                      \
  do {                                                                        \
    auto kern = K % 512 ? GV_KERNEL(MV, true, U) : GV_KERNEL(MV, false, U);   \
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
  const bool deep = gemv_deep(M, K);
  switch (mp) {
    case 1:
      if (deep) LAUNCH_GV(1, 8);
      else LAUNCH_GV(1, 4);
      break;
    case 2:
      if (deep) LAUNCH_GV(2, 8);
      else LAUNCH_GV(2, 4);
      break;
    case 3:
      if (deep) LAUNCH_GV(3, 8);
      else LAUNCH_GV(3, 4);
      break;
    case 4: LAUNCH_GV(4, 4); break;
    case 6: LAUNCH_GV(6, 4); break;
    default: LAUNCH_GV(8, 4); break;
  }
#undef LAUNCH_GV
#undef GV_KERNEL
  HIP_CHECK_KERNEL();
}

// Whether gemv_norm can take M rows of K entries where gemv does.
bool gemv_norm_fits(int64_t M, int64_t K, bool swiglu) {
  return gemv_fits(M, K, swiglu) && K % 512 == 0 && K <= 2 * 64 * GV_WAVES * 8;
}

// out = rmsnorm(residual + delta) W^T (+ bias), or with a gate as gemv; sum takes
// residual + delta (delta undefined: residual alone, and no sum).
void gemv_norm(torch::Tensor out, torch::Tensor sum, torch::Tensor delta,
               torch::Tensor residual, torch::Tensor weight, double eps,
               torch::Tensor w, c10::optional<torch::Tensor> bias,
               int64_t gate) {
  const bool swiglu = gate != 0;
  TORCH_CHECK(gate >= 0 && gate <= 1);
  TORCH_CHECK(residual.is_cuda() && residual.dim() == 2 && w.dim() == 2);
  const int64_t M = residual.size(0), K = residual.size(1);
  const int64_t N = swiglu ? w.size(0) / 2 : w.size(0);
  TORCH_CHECK(gemv_norm_fits(M, K, swiglu) && N >= 1 &&
              delta.defined() == sum.defined());
  auto check = [&](const torch::Tensor& t, int64_t n) {
    TORCH_CHECK(t.device() == residual.device(), "tensors on different devices");
    TORCH_CHECK(t.dtype() == torch::kBFloat16 && t.is_contiguous() &&
                t.numel() == n);
  };
  auto check16 = [&](const torch::Tensor& t, int64_t n) {
    check(t, n);
    TORCH_CHECK((reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0);
  };
  check16(residual, M * K);
  check16(weight, K);
  check16(w, (swiglu ? 2 * N : N) * K);
  check(out, M * N);
  if (delta.defined()) {
    check16(delta, M * K);
    check16(sum, M * K);
  }
  if (bias.has_value()) {
    TORCH_CHECK(!swiglu);
    check(*bias, N);
  }
  const at::cuda::CUDAGuard guard(residual.device());
  hipStream_t stream = at::cuda::getCurrentCUDAStream();
  const int64_t mp = M <= 4 ? M : M <= 6 ? 6 : 8;
  const size_t shmem = (size_t)mp * K * 2;
  const int64_t step = swiglu ? GV_ROWS / 2 : GV_ROWS;
  const int64_t need = ((N + step - 1) / step + GV_WAVES - 1) / GV_WAVES;
  const dim3 grid(std::min<int64_t>(need, 512));
  const GemvNorm g{
      delta.defined() ? (const uint16_t*)delta.data_ptr() : nullptr,
      (const uint16_t*)residual.data_ptr(), (const uint16_t*)weight.data_ptr(),
      sum.defined() ? (uint16_t*)sum.data_ptr() : nullptr, (float)eps};
  const uint16_t* b =
      bias.has_value() ? (const uint16_t*)bias->data_ptr() : nullptr;
  auto launch = [&](auto kern) {
    if (shmem > 64 * 1024)
      TORCH_CHECK(hipFuncSetAttribute(
                      (const void*)kern,
                      hipFuncAttributeMaxDynamicSharedMemorySize,
                      (int)shmem) == hipSuccess);
    hipLaunchKernelGGL(kern, grid, dim3(64 * GV_WAVES), shmem, stream,
                       (uint16_t*)out.data_ptr(), g,
                       (const uint16_t*)w.data_ptr(), b, (int)M, (int)N,
                       (int)K);
    HIP_CHECK_KERNEL();
  };
  const bool deep = gemv_deep(M, K), twice = K > 64 * GV_WAVES * 8;
#define LAUNCH_GVN_G(MV, GATE)                                                \
  do {                                                                        \
    constexpr int DEEP = MV <= 3 ? 8 : 4;                                     \
    if (deep && twice) launch(gemv_norm_kernel<MV, GV_ROWS, GATE, 2, DEEP>);  \
    else if (deep) launch(gemv_norm_kernel<MV, GV_ROWS, GATE, 1, DEEP>);      \
    else if (twice) launch(gemv_norm_kernel<MV, GV_ROWS, GATE, 2, 4>);        \
    else launch(gemv_norm_kernel<MV, GV_ROWS, GATE, 1, 4>);                   \
  } while (0)
#define LAUNCH_GVN(MV)                                                        \
  case MV:                                                                    \
    if (swiglu) LAUNCH_GVN_G(MV, 1);                                          \
    else LAUNCH_GVN_G(MV, 0);                                                 \
    break
  switch (mp) {
    LAUNCH_GVN(1);
    LAUNCH_GVN(2);
    LAUNCH_GVN(3);
    LAUNCH_GVN(4);
    LAUNCH_GVN(6);
    default: LAUNCH_GVN_G(8, 1); break;
  }
#undef LAUNCH_GVN
#undef LAUNCH_GVN_G
}

}  // namespace igw
