// Fused MoE routing kernel for gfx950 (Mixtral).
//
// Replaces the torch glue on the decode hot path (top-k + softmax + one-hot
// + cumsum-rank + index arithmetic was ~5.6 ms/step at batch 256 in
// profiles/r01 — torch's scan_outer_dim alone was 3 ms on a [T*K, E]
// one-hot): one launch computes, per token row,
//
//   * the top-k experts of the router logits (value order, ties by lower
//     expert id — matches torch.topk),
//   * softmax weights over the selected k logits (fp32),
//   * a padded-buffer destination row dst = expert * C + rank, where rank
//     is drawn from a per-expert atomic counter — dispatch order within an
//     expert is NOT semantically meaningful (the gather back uses the same
//     dst), so no stable scan is needed.
//
// One workgroup; per-expert counters live in LDS.  Decode-sized T only
// (the prefill path uses the sorted per-expert torch route).
#include <ATen/cuda/CUDAContext.h>
#include <c10/cuda/CUDAGuard.h>
#include <torch/extension.h>

#include "common.h"

namespace igw {

// The K largest of a row of logits and exp(logit - largest); returns 1 / their sum.
// K is a template constant, so that the arrays stay in registers.
template <int K>
DEVINLINE float top_experts(const float* row, int E, int* sel, float* w) {
  float m = -INFINITY;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    int best = 0;
    float bv = -INFINITY;
    for (int e = 0; e < E; ++e) {
      bool taken = false;
#pragma unroll
      for (int k2 = 0; k2 < K; ++k2) taken |= (k2 < k && sel[k2] == e);
      const float v = row[e];
      if (!taken && v > bv) {
        bv = v;
        best = e;
      }
    }
    sel[k] = best;
    w[k] = bv;
    m = fmaxf(m, bv);
  }
  float z = 0.0f;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    w[k] = __expf(w[k] - m);
    z += w[k];
  }
  return 1.0f / z;
}

template <int BLOCK, int K>
__global__ __launch_bounds__(BLOCK) void moe_route_kernel(
    float* __restrict__ weights,       // [T, K] fp32 softmax weights
    int32_t* __restrict__ dst,         // [T*K] padded-buffer row index
    int32_t* __restrict__ topk_idx,    // [T, K] selected experts
    int32_t* __restrict__ counts,      // [E] per-expert row counts
    const float* __restrict__ logits,  // [T, E] fp32 router logits
    int T, int E, int C) {
  __shared__ uint32_t counters[64];
  for (int e = threadIdx.x; e < 64; e += BLOCK) counters[e] = 0;
  __syncthreads();

  for (int t = threadIdx.x; t < T; t += BLOCK) {
    const float* row = logits + (int64_t)t * E;
    int sel[K];
    float w[K];
    const float inv = top_experts<K>(row, E, sel, w);
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int e = sel[k];
      const uint32_t r = atomicAdd(&counters[e], 1u);
      weights[(int64_t)t * K + k] = w[k] * inv;
      topk_idx[(int64_t)t * K + k] = e;
      dst[(int64_t)t * K + k] = e * C + (int32_t)r;
    }
  }
  __syncthreads();
  for (int e = threadIdx.x; e < E; e += BLOCK)
    counts[e] = (int32_t)counters[e];
}

void moe_route(torch::Tensor weights, torch::Tensor dst,
               torch::Tensor topk_idx, torch::Tensor counts,
               torch::Tensor logits, int64_t C) {
  TORCH_CHECK(logits.is_cuda() && logits.dtype() == torch::kFloat32);
  TORCH_CHECK(logits.is_contiguous());
  TORCH_CHECK(weights.dtype() == torch::kFloat32);
  TORCH_CHECK(dst.dtype() == torch::kInt32 &&
              topk_idx.dtype() == torch::kInt32 &&
              counts.dtype() == torch::kInt32);
  const int T = logits.size(0);
  const int E = logits.size(1);
  const int K = weights.size(1);
  TORCH_CHECK(E <= 64, "moe_route supports up to 64 experts");
  hipStream_t stream = at::cuda::getCurrentCUDAStream();
  constexpr int BLOCK = 256;
#define LAUNCH_ROUTE(KV)                                                     \
  hipLaunchKernelGGL((moe_route_kernel<BLOCK, KV>), dim3(1), dim3(BLOCK), 0, \
                     stream, (float*)weights.data_ptr(),                     \
                     (int32_t*)dst.data_ptr(), (int32_t*)topk_idx.data_ptr(),\
                     (int32_t*)counts.data_ptr(),                            \
                     (const float*)logits.data_ptr(), T, E, (int)C)
  switch (K) {
    case 1: LAUNCH_ROUTE(1); break;
    case 2: LAUNCH_ROUTE(2); break;
    case 4: LAUNCH_ROUTE(4); break;
    case 8: LAUNCH_ROUTE(8); break;
    default: TORCH_CHECK(false, "unsupported top-k for moe_route: ", K);
  }
#undef LAUNCH_ROUTE
  HIP_CHECK_KERNEL();
}

// The router's product of a few tokens with the choice of their experts: a workgroup
// per token, a wave per expert, logits rounded to bf16 like those of a product of its
// own, but summed in another order: a logit, and between near ties the expert, can
// differ.  Bound by latency: 5 tokens of 8 experts x 4096 take 5.8 us; the library's
// product, the conversion and moe_route took 19.7.
template <int K>
__global__ __launch_bounds__(512) void moe_pick_kernel(
    float* __restrict__ weights,       // [T, K] softmax over the chosen
    int32_t* __restrict__ topk_idx,    // [T, K]
    const uint16_t* __restrict__ x,    // [T, D]
    const uint16_t* __restrict__ w,    // [E, D]
    int64_t x_rs, int D, int E) {
  __shared__ float logits[64];
  const int lane = threadIdx.x & 63;
  const uint16_t* row = x + (int64_t)blockIdx.x * x_rs;
  for (int e = threadIdx.x >> 6; e < E; e += 8) {
    const uint16_t* we = w + (int64_t)e * D;
    float sum = 0.0f;
#pragma unroll 8
    for (int d = lane * 8; d < D; d += 512) {
      const ushort8 a = *(const ushort8*)(row + d), b = *(const ushort8*)(we + d);
#pragma unroll
      for (int j = 0; j < 8; ++j)
        sum = fmaf(bf16_to_f32(a.v[j]), bf16_to_f32(b.v[j]), sum);
    }
    sum = wave_reduce_sum(sum);
    if (lane == 0) logits[e] = bf16_to_f32(f32_to_bf16(sum));
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  int sel[K];
  float p[K];
  const float inv = top_experts<K>(logits, E, sel, p);
#pragma unroll
  for (int k = 0; k < K; ++k) {
    weights[(int64_t)blockIdx.x * K + k] = p[k] * inv;
    topk_idx[(int64_t)blockIdx.x * K + k] = sel[k];
  }
}

void moe_pick_rows(torch::Tensor weights, torch::Tensor topk_idx,
                   const torch::Tensor& x, const torch::Tensor& w) {
  const int T = x.size(0), D = x.size(1), E = w.size(0);
  if (T == 0) return;
  hipStream_t stream = at::cuda::getCurrentCUDAStream();
#define LAUNCH_PICK(KV)                                                       \
  case KV:                                                                    \
    hipLaunchKernelGGL((moe_pick_kernel<KV>), dim3(T), dim3(512), 0, stream,  \
                       (float*)weights.data_ptr(),                            \
                       (int32_t*)topk_idx.data_ptr(),                         \
                       (const uint16_t*)x.data_ptr(),                         \
                       (const uint16_t*)w.data_ptr(), x.stride(0), D, E);     \
    break
  switch (weights.size(1)) {
    LAUNCH_PICK(1);
    LAUNCH_PICK(2);
    LAUNCH_PICK(4);
    LAUNCH_PICK(8);
    default: TORCH_CHECK(false, "moe_pick: top_k");
  }
#undef LAUNCH_PICK
  HIP_CHECK_KERNEL();
}

// Routing for the grouped products: as above, but the rows of an expert follow
// those of the one before without gaps (start [E + 1]), for any T.  The row
// within an expert is whatever order the counters give: nothing depends on it.
// One workgroup (1890 tokens of 8 experts: 13 us); every thread keeps its
// assignments in dst between the two passes.
template <typename L, int K>
__global__ __launch_bounds__(1024) void moe_dispatch_kernel(
    float* __restrict__ weights,  // [T, K] softmax over the chosen
    int64_t* __restrict__ dst,    // [T, K] row of the sorted buffer
    int32_t* __restrict__ start,  // [E + 1]
    const L* __restrict__ logits, // [T, E]
    int T, int E) {
  __shared__ uint32_t counters[64];
  __shared__ uint32_t first[64];
  const int tid = threadIdx.x;
  if (tid < 64) counters[tid] = 0;
  __syncthreads();
  for (int t = tid; t < T; t += 1024) {
    const L* row = logits + (int64_t)t * E;
    int sel[K];
    float val[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      int best = -1;
      float bv = 0.0f;
      for (int e = 0; e < E; ++e) {
        bool taken = false;
#pragma unroll
        for (int j = 0; j < k; ++j) taken |= sel[j] == e;
        float v;
        if constexpr (sizeof(L) == 2) v = bf16_to_f32(row[e]);
        else v = row[e];
        if (!taken && (best < 0 || v > bv)) {
          bv = v;
          best = e;
        }
      }
      sel[k] = best;
      val[k] = bv;
    }
    float z = 0.0f, w[K];
#pragma unroll
    for (int k = 0; k < K; ++k) z += w[k] = __expf(val[k] - val[0]);
#pragma unroll
    for (int k = 0; k < K; ++k) {
      weights[(int64_t)t * K + k] = w[k] / z;
      dst[(int64_t)t * K + k] =
          (int64_t)atomicAdd(&counters[sel[k]], 1u) << 6 | sel[k];
    }
  }
  __syncthreads();
  if (tid < 64) {
    uint32_t upto = counters[tid];
    const uint32_t mine = upto;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const uint32_t up = __shfl_up(upto, d, 64);
      if (tid >= d) upto += up;
    }
    first[tid] = upto - mine;
    if (tid < E) start[tid + 1] = (int32_t)upto;
    if (tid == 0) start[0] = 0;
  }
  __syncthreads();
  for (int t = tid; t < T; t += 1024)
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int64_t a = dst[(int64_t)t * K + k];
      dst[(int64_t)t * K + k] = first[a & 63] + (a >> 6);
    }
}

void moe_dispatch(torch::Tensor weights, torch::Tensor dst,
                  torch::Tensor start, torch::Tensor logits) {
  const bool half = logits.dtype() == torch::kBFloat16;
  TORCH_CHECK(logits.is_cuda() && logits.dim() == 2 && logits.is_contiguous() &&
              (half || logits.dtype() == torch::kFloat32));
  const int64_t T = logits.size(0), E = logits.size(1);
  TORCH_CHECK(weights.dim() == 2 && weights.size(0) == T &&
              weights.dtype() == torch::kFloat32 && weights.is_contiguous());
  const int64_t K = weights.size(1);
  TORCH_CHECK(T >= 1 && T < (1 << 25) && E >= K && E <= 64 &&
              dst.dtype() == torch::kInt64 && dst.is_contiguous() &&
              dst.numel() == T * K && start.dtype() == torch::kInt32 &&
              start.is_contiguous() && start.numel() == E + 1);
  for (const auto* t : {&weights, &dst, &start})
    TORCH_CHECK(t->device() == logits.device(), "tensors on different devices");
  const at::cuda::CUDAGuard guard(logits.device());
  hipStream_t stream = at::cuda::getCurrentCUDAStream();
#define LAUNCH_DISPATCH(L, KV)                                                \
  hipLaunchKernelGGL((moe_dispatch_kernel<L, KV>), dim3(1), dim3(1024), 0,    \
                     stream, weights.data_ptr<float>(),                       \
                     dst.data_ptr<int64_t>(), start.data_ptr<int32_t>(),      \
                     (const L*)logits.data_ptr(), (int)T, (int)E)
#define LAUNCH_DISPATCH_K(KV)                                                 \
  case KV:                                                                    \
    if (half) LAUNCH_DISPATCH(uint16_t, KV);                                  \
    else LAUNCH_DISPATCH(float, KV);                                          \
    break
  switch (K) {
    LAUNCH_DISPATCH_K(1);
    LAUNCH_DISPATCH_K(2);
    LAUNCH_DISPATCH_K(4);
    LAUNCH_DISPATCH_K(8);
    default: TORCH_CHECK(false, "unsupported top-k for moe_dispatch: ", K);
  }
#undef LAUNCH_DISPATCH_K
#undef LAUNCH_DISPATCH
  HIP_CHECK_KERNEL();
}

}  // namespace igw
