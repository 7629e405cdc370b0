// Row kernels of a sandwich-norm layer (an RMS norm before AND after every
// sublayer) on an fp32 residual stream (gfx950):
//
//   add_normed_rmsnorm   residual += mult * rmsnorm(delta) * w_post (in place)
//                        out = rmsnorm(residual) * w_pre, or the residual
//                        itself in the activation type when w_pre is absent
//   gelu_mul_rows        gelu_tanh(z) * table[token, col0 : col0 + W]
//
// One block per row (256 threads, of few rows 1024); both statistics are fp32
// block reductions.
//
// add_normed_rmsnorm is bound by one pass over the row: residual read and
// written, delta read, out written.  Rows of up to 8192 entries that allow
// loads of four entries stay in registers between the two statistics, all
// their loads issued before the first is used; longer, odd or misaligned rows
// are read again after each statistic.  Measured, rows read again and kept
// (us): 6000 rows of 4096 71.0 and 47.4 (6.2 TB/s), of 8192 188 and 122; few rows are
// at the launch.  A delta of several parts (a product's sums over parts of its K) is
// added as it is read: a sum of its own takes another 4.5 us of 48 rows (Bivatar's
// decode of 48 sequences, four such sums, 698 and 688).
#include "../csrc_hybrid/act_types.h"

namespace igw {

// PARTS: delta is the sum of `parts` of them, part_stride entries apart.
template <typename TD, typename TO, bool PARTS = false>
__global__ __launch_bounds__(256) void add_normed_rmsnorm_kernel(
    TO* __restrict__ out, float* __restrict__ residual,
    const TD* __restrict__ delta, int64_t delta_rs,
    const float* __restrict__ w_post, const float* __restrict__ w_pre, int D,
    float eps, float mult, int parts, int64_t part_stride) {
  __shared__ float red[8];
  const int t = blockIdx.x, tid = threadIdx.x;
  float* res = residual + (int64_t)t * D;
  TO* o = out + (int64_t)t * D;
  float ss = 0.0f;
  if (delta) {
    const TD* dl = delta + (int64_t)t * delta_rs;
    auto entry = [&](int d) {
      float x = Act<TD>::ld(dl + d);
      if constexpr (PARTS)
        for (int p = 1; p < parts; ++p) x += Act<TD>::ld(dl + p * part_stride + d);
      return x;
    };
    float sd = 0.0f;
    for (int d = tid; d < D; d += 256) {
      const float x = entry(d);
      sd += x * x;
    }
    sd = block_reduce_sum<256>(sd, red);
    const float r1 = mult / sqrtf(sd / (float)D + eps);
    __syncthreads();
    for (int d = tid; d < D; d += 256) {
      const float x = res[d] + entry(d) * r1 * w_post[d];
      res[d] = x;
      ss += x * x;
    }
  } else {
    for (int d = tid; d < D; d += 256) {
      const float x = res[d];
      ss += x * x;
    }
  }
  if (!w_pre) {
    for (int d = tid; d < D; d += 256) Act<TO>::st(o + d, res[d]);
    return;
  }
  ss = block_reduce_sum<256>(ss, red);
  const float r2 = 1.0f / sqrtf(ss / (float)D + eps);
  for (int d = tid; d < D; d += 256)
    Act<TO>::st(o + d, res[d] * r2 * w_pre[d]);
}

// four consecutive entries as fp32
template <typename T>
DEVINLINE float4 load4(const T* p) {
  if constexpr (sizeof(T) == 4) {
    return *reinterpret_cast<const float4*>(p);
  } else {
    const ushort4x v = *reinterpret_cast<const ushort4x*>(p);
    return make_float4(bf16_to_f32(v.v[0]), bf16_to_f32(v.v[1]),
                       bf16_to_f32(v.v[2]), bf16_to_f32(v.v[3]));
  }
}

template <typename T>
DEVINLINE void store4(T* p, float4 v) {
  if constexpr (sizeof(T) == 4) {
    *reinterpret_cast<float4*>(p) = v;
  } else {
    ushort4x o;
    o.v[0] = f32_to_bf16(v.x);
    o.v[1] = f32_to_bf16(v.y);
    o.v[2] = f32_to_bf16(v.z);
    o.v[3] = f32_to_bf16(v.w);
    *reinterpret_cast<ushort4x*>(p) = o;
  }
}

DEVINLINE float square4(float4 v) {
  return v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w;
}

// D <= 4 BLOCK NC, D % 4 == 0, rows and weights aligned to four entries.  PARTS as
// above.
template <typename TD, typename TO, int NC, int BLOCK = 256,
          bool PARTS = false>
__global__ __launch_bounds__(BLOCK) void add_normed_rmsnorm_row_kernel(
    TO* __restrict__ out, float* __restrict__ residual,
    const TD* __restrict__ delta, int64_t delta_rs,
    const float* __restrict__ w_post, const float* __restrict__ w_pre, int D,
    float eps, float mult, int parts, int64_t part_stride) {
  __shared__ float red[BLOCK / WAVE_SIZE];
  const int t = blockIdx.x, tid = threadIdx.x;
  float* res = residual + (int64_t)t * D;
  TO* o = out + (int64_t)t * D;
  const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
  float4 x[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int d = (c * BLOCK + tid) * 4;
    x[c] = d < D ? load4(res + d) : zero;
  }
  if (delta) {
    const TD* dl = delta + (int64_t)t * delta_rs;
    float4 y[NC];
    float sd = 0.0f;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int d = (c * BLOCK + tid) * 4;
      y[c] = d < D ? load4(dl + d) : zero;
    }
    if constexpr (PARTS) {
#pragma unroll 4
      for (int p = 1; p < parts; ++p) {
        dl += part_stride;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          const int d = (c * BLOCK + tid) * 4;
          const float4 v = d < D ? load4(dl + d) : zero;
          y[c].x += v.x;
          y[c].y += v.y;
          y[c].z += v.z;
          y[c].w += v.w;
        }
      }
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) sd += square4(y[c]);
    sd = block_reduce_sum<BLOCK>(sd, red);
    const float r1 = mult / sqrtf(sd / (float)D + eps);
    __syncthreads();
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int d = (c * BLOCK + tid) * 4;
      if (d >= D) break;
      const float4 w = load4(w_post + d);
      x[c].x += y[c].x * r1 * w.x;
      x[c].y += y[c].y * r1 * w.y;
      x[c].z += y[c].z * r1 * w.z;
      x[c].w += y[c].w * r1 * w.w;
      store4(res + d, x[c]);
    }
  }
  float r2 = 1.0f;
  if (w_pre) {
    float ss = 0.0f;
#pragma unroll
    for (int c = 0; c < NC; ++c) ss += square4(x[c]);
    ss = block_reduce_sum<BLOCK>(ss, red);
    r2 = 1.0f / sqrtf(ss / (float)D + eps);
  }
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int d = (c * BLOCK + tid) * 4;
    if (d >= D) break;
    float4 v = x[c];
    if (w_pre) {
      const float4 w = load4(w_pre + d);
      v = make_float4(v.x * r2 * w.x, v.y * r2 * w.y, v.z * r2 * w.z,
                      v.w * r2 * w.w);
    }
    store4(o + d, v);
  }
}

void add_normed_rmsnorm(torch::Tensor out, torch::Tensor residual,
                        c10::optional<torch::Tensor> delta,
                        c10::optional<torch::Tensor> w_post,
                        c10::optional<torch::Tensor> w_pre, double eps,
                        double mult) {
  TORCH_CHECK(residual.is_cuda() && residual.dtype() == torch::kFloat32 &&
              residual.is_contiguous() && residual.dim() == 2);
  const int T = residual.size(0), D = residual.size(1);
  TORCH_CHECK(out.is_contiguous() && out.numel() == residual.numel());
  int parts = 1;
  int64_t part_stride = 0;
  if (delta.has_value() && delta->dim() == 3) {
    TORCH_CHECK(delta->dtype() == torch::kFloat32 && delta->is_contiguous() &&
                delta->size(0) >= 1 && delta->size(0) < (1 << 16));
    parts = (int)delta->size(0);
    part_stride = delta->stride(0);
    delta = delta->select(0, 0);
  }
  if (delta.has_value()) {
    TORCH_CHECK(delta->dim() == 2 && delta->size(0) == T &&
                delta->size(1) == D && delta->stride(1) == 1);
    TORCH_CHECK(w_post.has_value() && w_post->dtype() == torch::kFloat32 &&
                w_post->is_contiguous() && w_post->numel() == D);
  }
  if (w_pre.has_value())
    TORCH_CHECK(w_pre->dtype() == torch::kFloat32 && w_pre->is_contiguous() &&
                w_pre->numel() == D);
  if (T == 0) return;
  hipStream_t stream = at::cuda::getCurrentCUDAStream();
  const float* wp = delta.has_value() ? (const float*)w_post->data_ptr()
                                      : nullptr;
  const float* wn = w_pre.has_value() ? (const float*)w_pre->data_ptr()
                                      : nullptr;
  const int64_t drs = delta.has_value() ? (int64_t)delta->stride(0) : 0;
  const bool d16 = delta.has_value() &&
                   delta->scalar_type() == torch::kBFloat16;
  auto by4 = [](const void* p, int64_t size) {
    return (reinterpret_cast<uintptr_t>(p) & (4 * size - 1)) == 0;
  };
  const bool in_regs =
      D <= 8192 && D % 4 == 0 && drs % 4 == 0 && by4(wp, 4) && by4(wn, 4) &&
      by4(residual.data_ptr(), 4) &&
      by4(out.data_ptr(), out.element_size()) &&
      (!delta.has_value() || by4(delta->data_ptr(), delta->element_size()));
#define LAUNCH_ANR_K(KERN, BLOCK, TD, TO)                                     \
  hipLaunchKernelGGL((KERN), dim3(T), dim3(BLOCK), 0, stream,                 \
                     (TO*)out.data_ptr(), (float*)residual.data_ptr(),        \
                     delta.has_value() ? (const TD*)delta->data_ptr()         \
                                       : nullptr,                             \
                     drs, wp, wn, D, (float)eps, (float)mult, parts,          \
                     part_stride)
// parts come in fp32
#define LAUNCH_ANR_ALL(TD, TO)                                                \
  do {                                                                        \
    if (sizeof(TD) == 4 && parts > 1)                                         \
      LAUNCH_ANR_K((add_normed_rmsnorm_kernel<TD, TO, sizeof(TD) == 4>), 256, \
                   TD, TO);                                                   \
    else                                                                      \
      LAUNCH_ANR_K((add_normed_rmsnorm_kernel<TD, TO>), 256, TD, TO);         \
  } while (0)
#define LAUNCH_ANR_ROW(TD, TO, NC, BLOCK)                                     \
  do {                                                                        \
    if (sizeof(TD) == 4 && parts > 1)                                         \
      LAUNCH_ANR_K((add_normed_rmsnorm_row_kernel<TD, TO, NC, BLOCK,          \
                                                  sizeof(TD) == 4>),          \
                   BLOCK, TD, TO);                                            \
    else                                                                      \
      LAUNCH_ANR_K((add_normed_rmsnorm_row_kernel<TD, TO, NC, BLOCK>), BLOCK, \
                   TD, TO);                                                   \
  } while (0)
  // Few rows wait for their own loads, of which 1024 threads have a quarter each; of
  // many, workgroups wait beside each other (us, bf16 deltas, rows in the caches, 256
  // threads and 1024, 1 / 48 / 256 / 512 rows: 2052 entries, where half the threads
  // have none, 3.3 3.8 4.1 5.3 and 2.7 3.3 3.7 4.9, 3072 3.5 3.7 4.6 6.3 and 2.8 3.1
  // 3.9 5.7, 4096 3.7 4.0 5.7 7.5 and 2.9 3.3 4.8 6.8, 8192 5.2 5.7 9.1 11.9 and 3.6
  // 4.0 7.0 10.4; with a norm behind it 512 rows of 2052 / 4096 / 8192 6.3 8.7 13.7
  // and 6.5 8.4 11.7).
  const bool few = T <= 512;
#define LAUNCH_ANR(TD, TO)                                                    \
  do {                                                                        \
    if (!in_regs) LAUNCH_ANR_ALL(TD, TO);                                     \
    else if (D <= 1024) LAUNCH_ANR_ROW(TD, TO, 1, 256);                       \
    else if (D <= 2048) LAUNCH_ANR_ROW(TD, TO, 2, 256);                       \
    else if (D <= 4096 && few) LAUNCH_ANR_ROW(TD, TO, 1, 1024);               \
    else if (D <= 4096) LAUNCH_ANR_ROW(TD, TO, 4, 256);                       \
    else if (few) LAUNCH_ANR_ROW(TD, TO, 2, 1024);                            \
    else LAUNCH_ANR_ROW(TD, TO, 8, 256);                                      \
  } while (0)
  if (delta.has_value())
    TORCH_CHECK(d16 || delta->scalar_type() == torch::kFloat32,
                "delta must be bfloat16 or float32");
  IGW_DISPATCH_ACT(out, {
    if (d16) LAUNCH_ANR(uint16_t, act_t);
    else LAUNCH_ANR(float, act_t);
  });
#undef LAUNCH_ANR
#undef LAUNCH_ANR_ROW
#undef LAUNCH_ANR_ALL
#undef LAUNCH_ANR_K
  HIP_CHECK_KERNEL();
}

DEVINLINE float gelu_tanh_f32(float z) {
  const float u = 0.7978845608028654f * (z + 0.044715f * z * z * z);
  return 0.5f * z * (1.0f + tanhf(u));
}

template <typename T>
__global__ void gelu_mul_rows_kernel(T* __restrict__ out,
                                     const T* __restrict__ z,
                                     const T* __restrict__ table,
                                     int64_t table_rs,
                                     const int64_t* __restrict__ tokens,
                                     int64_t total, int W, int col0) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= total) return;
  const int64_t t = i / W;
  const int c = (int)(i - t * W);
  const float e = Act<T>::ld(table + tokens[t] * table_rs + col0 + c);
  Act<T>::st(out + i, gelu_tanh_f32(Act<T>::ld(z + i)) * e);
}

void gelu_mul_rows(torch::Tensor out, torch::Tensor z, torch::Tensor table,
                   torch::Tensor tokens, int64_t col0) {
  TORCH_CHECK(z.is_cuda() && z.is_contiguous() && z.dim() == 2 &&
              out.is_contiguous() && out.dtype() == z.dtype() &&
              out.numel() == z.numel());
  const int64_t T = z.size(0);
  const int W = z.size(1);
  TORCH_CHECK(table.dim() == 2 && table.stride(1) == 1 &&
              table.dtype() == z.dtype() && col0 >= 0 &&
              col0 + W <= table.size(1));
  TORCH_CHECK(tokens.dtype() == torch::kInt64 && tokens.is_contiguous() &&
              tokens.numel() == T);
  if (T == 0 || W == 0) return;
  hipStream_t stream = at::cuda::getCurrentCUDAStream();
  const int64_t total = T * W;
  IGW_DISPATCH_ACT(z, {
    hipLaunchKernelGGL((gelu_mul_rows_kernel<act_t>),
                       dim3((unsigned)((total + 255) / 256)), dim3(256), 0,
                       stream, (act_t*)out.data_ptr(),
                       (const act_t*)z.data_ptr(),
                       (const act_t*)table.data_ptr(),
                       (int64_t)table.stride(0),
                       (const int64_t*)tokens.data_ptr(), total, W,
                       (int)col0);
  });
  HIP_CHECK_KERNEL();
}

}  // namespace igw
