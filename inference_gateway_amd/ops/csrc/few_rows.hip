// Host side of ops.linear, ops.linear_silu_mul, ops.linear_gated_act, ops.moe_few
// and ops.moe_rows: which calls the kernels for a few rows of x (gemv.hip), for
// tens of them (rows_gemm and held_gemm in rows_gemm.hip) and for hundreds and
// thousands of them (narrow_gemm.hip, wide_gemm.hip) take.  product_route is the
// rule that the launch goes by.
//
// What they are handed is a pointer, so the tensors have to be what they seem:
// plain dense bf16 on one GPU, in a call that nothing but the product has to
// see.  Everything else (weights elsewhere, autograd in either mode, vmap, a
// trace, a dispatch mode, autocast, other types and layouts) is the library's
// product, with its results and its errors.
#include <ATen/cuda/CUDAContext.h>
#include <c10/cuda/CUDAGuard.h>
#include <torch/extension.h>

#include "plain_call.h"

namespace igw {

bool gemv_fits(int64_t M, int64_t K, bool swiglu);
bool gemv_ahead(int64_t M, int64_t N, int64_t K, bool swiglu);
int64_t rows_gemm_splits(int64_t M, int64_t N, int64_t K, bool swiglu);
bool rows_gemm_ahead(int64_t M, int64_t S, int64_t K, bool swiglu);
bool held_gemm_takes(int64_t M, int64_t N, int64_t K);
int64_t held_splits(int64_t M, int64_t N, int64_t K);
void held_gemm(torch::Tensor out, torch::Tensor x, torch::Tensor w,
               c10::optional<torch::Tensor> bias);
int64_t wide_gemm_tile(int64_t M, int64_t N, int64_t K, bool swiglu);
bool wide_gemm_fits(int64_t x_rs, int64_t N, int64_t K, bool swiglu);
void wide_gemm(torch::Tensor out, torch::Tensor x, torch::Tensor w,
               int64_t gate, int64_t tile);
int64_t narrow_tile(int64_t M, int64_t N, int64_t K, bool gated);
void moe_pick_rows(torch::Tensor weights, torch::Tensor topk_idx,
                   const torch::Tensor& x, const torch::Tensor& w);
void narrow_gemm(torch::Tensor out, torch::Tensor x, torch::Tensor w,
                 int64_t gate, int64_t tile);
int64_t wide_split_ahead(int64_t M, int64_t N, int64_t K, bool norm);
torch::Tensor split_parts(const torch::Tensor& x, const torch::Tensor& w,
                          int64_t tile, int64_t S);
torch::Tensor rows_gemm_parts(const torch::Tensor& out, const torch::Tensor& x,
                              const torch::Tensor& w,
                              const c10::optional<torch::Tensor>& bias,
                              int64_t gate);
torch::Tensor held_gemm_parts(const torch::Tensor& out, const torch::Tensor& x,
                              const torch::Tensor& w,
                              const c10::optional<torch::Tensor>& bias);
void sum_parts(torch::Tensor out, const torch::Tensor& part,
               const c10::optional<torch::Tensor>& bias);
bool sum_add_rmsnorm_fits(int64_t hidden);
void sum_add_rmsnorm(torch::Tensor out, torch::Tensor part,
                     torch::Tensor residual, torch::Tensor weight, double eps);
bool gemv_norm_fits(int64_t M, int64_t K, bool swiglu);
void gemv_norm(torch::Tensor out, torch::Tensor sum, torch::Tensor delta,
               torch::Tensor residual, torch::Tensor weight, double eps,
               torch::Tensor w, c10::optional<torch::Tensor> bias,
               int64_t gate);
bool moe_few_fits(int64_t T, int64_t top_k, int64_t D, int64_t F);
void gemv(torch::Tensor out, torch::Tensor x, torch::Tensor w,
          c10::optional<torch::Tensor> bias, int64_t gate);
void rows_gemm(torch::Tensor out, torch::Tensor x, torch::Tensor w,
               c10::optional<torch::Tensor> bias, int64_t gate);

static bool by16(const torch::Tensor& t) {
  return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0;
}

// Whether the kernels can be handed the call at all.
static bool call_fits(const torch::Tensor& x, const torch::Tensor& w,
                      const c10::optional<torch::Tensor>& bias, bool swiglu,
                      bool anywhere) {
  if (!(anywhere || x.is_cuda()) || x.dim() != 2 || w.dim() != 2 ||
      !call_is_plain() || !plain_bf16(x, x.device()) ||
      !plain_bf16(w, x.device()))
    return false;
  const int64_t K = x.size(1);
  const int64_t N = swiglu ? w.size(0) / 2 : w.size(0);
  if (w.size(1) != K || (swiglu && w.size(0) % 2 != 0) || !w.is_contiguous() ||
      x.stride(1) != 1 || x.stride(0) % 8 != 0 || !by16(x) || !by16(w))
    return false;
  return !bias.has_value() ||
         (!swiglu && plain_bf16(*bias, x.device()) && bias->dim() == 1 &&
          bias->size(0) == N && bias->is_contiguous());
}

// A kernel and what it is launched with: the tile, with K in parts 256 times the
// tile and the parts.
struct Route {
  int64_t kernel = 0, how = 0;
};

// Where GELU inside is ahead of the product (gemv, held_gemm or the library's) and
// gated_act.  SwiGLU's lines are against the library and silu_mul (us, apart and inside:
// gemv, 3 rows 64128 x 512 18.3 and 21.8, 4 rows 68736 x 512 21.8 and 27.5, 7 rows 15360 x
// 2560 17.9 and 23.1, 8 rows 14592 x 3072 19.2 and 24.9, 3712 x 2560 8.6 and 9.9, but
// 28672 x 8192 in 0.77 of the time; tiles that leave a half of the compute units idle, or
// of a long K, 8192 x 3584, 440 rows, 42.0 and 49.6, 4096 x 8192, 1000 rows, 83.4 and 94.6,
// 16384 x 11008, 131 rows, 107 and 181, 32768 x 14336, 288 rows, 279 and 326, but 28672 x
// 4096, 320 to 3000 rows, in 0.86 to 0.96 of the time).
static bool gelu_gemv_ahead(int64_t M, int64_t rows, int64_t K) {
  return M <= 2 || (M <= 6 ? K >= 1024 : rows >= 28672 || K > 4096);
}
static bool gelu_wide_ahead(int64_t M, int64_t N, int64_t K, int64_t tile) {
  const int64_t tm = 32 * (tile >> 4), tn = 16 * (tile & 15);
  return K <= 8192 && (M + tm - 1) / tm * ((N + tn - 1) / tn) >= 192;
}

// The kernel of a call, narrow_gemm aside.  0: none of them, 1: gemv, 2: rows_gemm,
// 3: wide_gemm, 4: held_gemm, 5: wide_gemm with K in parts.  `anywhere`: also off
// the GPU (the rule alone, nothing is launched).  norm: fused_add_rmsnorm follows.
static Route route_of(const torch::Tensor& x, const torch::Tensor& w,
                      const c10::optional<torch::Tensor>& bias, int64_t gate,
                      bool norm) {
  const bool swiglu = gate != 0;
  const int64_t M = x.size(0), K = x.size(1);
  const int64_t N = swiglu ? w.size(0) / 2 : w.size(0);
  if (M > 64) {
    if (!wide_gemm_fits(x.stride(0), N, K, swiglu)) return {};
    const int64_t tile = bias.has_value() ? 0 : wide_gemm_tile(M, N, K, swiglu);
    if (tile > 0)
      return gate != 2 || gelu_wide_ahead(M, N, K, tile) ? Route{3, tile} : Route{};
    const int64_t cut = swiglu ? 0 : wide_split_ahead(M, N, K, norm);
    return cut > 0 ? Route{5, cut} : Route{};
  }
  if (gemv_fits(M, K, swiglu))
    return {gemv_ahead(M, w.size(0), K, swiglu) &&
            (gate != 2 || gelu_gemv_ahead(M, w.size(0), K))};
  if (!swiglu && held_gemm_takes(M, N, K)) return {4};
  const int64_t S = rows_gemm_splits(M, N, K, swiglu);
  return {S > 0 && rows_gemm_ahead(M, S, K, swiglu) ? 2 : 0};
}

// narrow_gemm's tile for a call that it takes before `other`, or 0.  Up to 48 rows
// of fewer than 65536 outputs, and 16 of a K below 4096, the other kernels keep what
// they take, where they are as fast or faster (see narrow_gemm.hip).
static int64_t narrow_before(const Route& other, const torch::Tensor& x,
                             const torch::Tensor& w,
                             const c10::optional<torch::Tensor>& bias,
                             bool swiglu) {
  const int64_t M = x.size(0), K = x.size(1);
  const int64_t N = swiglu ? w.size(0) / 2 : w.size(0);
  if (bias.has_value() || other.kernel == 1 ||
      !wide_gemm_fits(x.stride(0), N, K, swiglu))
    return 0;
  if (other.kernel != 0 && M <= 48 && (N < 65536 || (M <= 16 && K < 4096)))
    return 0;
  return narrow_tile(M, N, K, swiglu);
}

// What runs the call: as above, 6: narrow_gemm.  gate: 0 none, 1 SiLU, 2 GELU.
static Route product_route(const torch::Tensor& x, const torch::Tensor& w,
                           const c10::optional<torch::Tensor>& bias,
                           int64_t gate, bool anywhere) {
  if (!call_fits(x, w, bias, gate != 0, anywhere)) return {};
  const Route other = route_of(x, w, bias, gate, false);
  const int64_t tile = narrow_before(other, x, w, bias, gate != 0);
  return tile > 0 ? Route{6, tile} : other;
}

int64_t product_kernel(const torch::Tensor& x, const torch::Tensor& w,
                       const c10::optional<torch::Tensor>& bias, int64_t gate,
                       bool anywhere) {
  return product_route(x, w, bias, gate, anywhere).kernel;
}

// As product_kernel of gate 0 or 1, were narrow_gemm not there.
int64_t few_rows_takes(const torch::Tensor& x, const torch::Tensor& w,
                       const c10::optional<torch::Tensor>& bias, bool swiglu,
                       bool anywhere) {
  return call_fits(x, w, bias, swiglu, anywhere)
             ? route_of(x, w, bias, swiglu, false).kernel
             : 0;
}

// The tile of narrow_gemm for a call of gate 0 or 1 that it takes, or 0.
int64_t narrow_takes(const torch::Tensor& x, const torch::Tensor& w,
                     const c10::optional<torch::Tensor>& bias, bool swiglu,
                     bool anywhere) {
  const Route r = product_route(x, w, bias, swiglu, anywhere);
  return r.kernel == 6 ? r.how : 0;
}

// The product, or nothing when none of the kernels takes it.  gate: 0 none, else W
// = [gate; up] and the result is SiLU(gate) * up (1) or GELU(gate) * up (2).
c10::optional<torch::Tensor> few_rows(const torch::Tensor& x,
                                      const torch::Tensor& w,
                                      const c10::optional<torch::Tensor>& bias,
                                      int64_t gate) {
  const Route r = product_route(x, w, bias, gate, false);
  if (r.kernel == 0) return c10::nullopt;
  auto out = torch::empty({x.size(0), gate != 0 ? w.size(0) / 2 : w.size(0)},
                          x.options());
  switch (r.kernel) {
    case 1: gemv(out, x, w, bias, gate); break;
    case 2: rows_gemm(out, x, w, bias, gate); break;
    case 3: wide_gemm(out, x, w, gate, r.how); break;
    case 4: held_gemm(out, x, w, bias); break;
    case 5:
      sum_parts(out, split_parts(x, w, r.how >> 8, r.how & 255), bias);
      break;
    default: narrow_gemm(out, x, w, gate, r.how);
  }
  return out;
}

// Which of the kernels takes a product that fused_add_rmsnorm follows, in parts
// that the norm adds; 0: none.
static Route norm_route(const torch::Tensor& x, const torch::Tensor& w,
                        const torch::Tensor& residual,
                        const torch::Tensor& weight, bool anywhere) {
  if (!call_fits(x, w, c10::nullopt, false, anywhere)) return {};
  const Route r = route_of(x, w, c10::nullopt, 0, true);
  if (r.kernel != 2 && r.kernel != 4 && r.kernel != 5) return {};
  const int64_t M = x.size(0), N = w.size(0);
  if (!plain_bf16(residual, x.device()) || !plain_bf16(weight, x.device()) ||
      residual.dim() != 2 || residual.size(0) != M || residual.size(1) != N ||
      !residual.is_contiguous() || weight.dim() != 1 || weight.size(0) != N ||
      !weight.is_contiguous() || !by16(residual) || !by16(weight) ||
      !sum_add_rmsnorm_fits(N))
    return {};
  if (r.kernel == 4 && held_splits(M, N, x.size(1)) < 2) return {};
  if (r.kernel == 2 && rows_gemm_splits(M, N, x.size(1), false) < 2) return {};
  return r;
}

int64_t linear_norm_takes(const torch::Tensor& x, const torch::Tensor& w,
                          const torch::Tensor& residual,
                          const torch::Tensor& weight, bool anywhere) {
  return norm_route(x, w, residual, weight, anywhere).kernel;
}

// residual += x W^T in place and its norm, or nothing (and nothing done) when the
// product does not come in parts.
c10::optional<torch::Tensor> linear_add_rmsnorm(const torch::Tensor& x,
                                                const torch::Tensor& w,
                                                const torch::Tensor& residual,
                                                const torch::Tensor& weight,
                                                double eps) {
  const Route r = norm_route(x, w, residual, weight, false);
  if (r.kernel == 0) return c10::nullopt;
  const torch::Tensor none;
  const auto part =
      r.kernel == 5   ? split_parts(x, w, r.how >> 8, r.how & 255)
      : r.kernel == 4 ? held_gemm_parts(none, x, w, c10::nullopt)
                      : rows_gemm_parts(none, x, w, c10::nullopt, 0);
  auto out = torch::empty_like(residual);
  sum_add_rmsnorm(out, part, residual, weight, eps);
  return out;
}

// The product that few_rows would make of parts of K (gate 0, no bias) as those parts,
// fp32 [S, M, N], for a kernel that adds them as it reads; nothing where it has none.
c10::optional<torch::Tensor> linear_parts(const torch::Tensor& x,
                                          const torch::Tensor& w) {
  const Route r = product_route(x, w, c10::nullopt, 0, false);
  const int64_t M = x.dim() == 2 ? x.size(0) : 0;
  const torch::Tensor none;
  if (r.kernel == 5) return split_parts(x, w, r.how >> 8, r.how & 255);
  if (r.kernel == 4 && held_splits(M, w.size(0), x.size(1)) >= 2)
    return held_gemm_parts(none, x, w, c10::nullopt);
  if (r.kernel == 2 && rows_gemm_splits(M, w.size(0), x.size(1), false) >= 2)
    return rows_gemm_parts(none, x, w, c10::nullopt, 0);
  return c10::nullopt;
}

// Whether gemv takes the product of x = rmsnorm(residual + delta) with the norm in
// it.
bool norm_linear_takes(const c10::optional<torch::Tensor>& delta,
                       const torch::Tensor& residual,
                       const torch::Tensor& weight, const torch::Tensor& w,
                       const c10::optional<torch::Tensor>& bias, bool swiglu,
                       bool anywhere) {
  if (few_rows_takes(residual, w, bias, swiglu, anywhere) != 1) return false;
  const int64_t M = residual.size(0), K = residual.size(1);
  if (!gemv_norm_fits(M, K, swiglu) || !residual.is_contiguous() ||
      !plain_bf16(weight, residual.device()) || weight.dim() != 1 ||
      weight.size(0) != K || !weight.is_contiguous() || !by16(weight))
    return false;
  return !delta.has_value() ||
         (plain_bf16(*delta, residual.device()) && delta->dim() == 2 &&
          delta->size(0) == M && delta->size(1) == K &&
          delta->is_contiguous() && by16(*delta));
}

// The product and residual + delta (in memory of its own; without a delta the
// residual itself), or nothing.
c10::optional<std::tuple<torch::Tensor, torch::Tensor>> norm_linear(
    const c10::optional<torch::Tensor>& delta, const torch::Tensor& residual,
    const torch::Tensor& weight, double eps, const torch::Tensor& w,
    const c10::optional<torch::Tensor>& bias, int64_t gate) {
  if (!norm_linear_takes(delta, residual, weight, w, bias, gate != 0, false))
    return c10::nullopt;
  auto out = torch::empty(
      {residual.size(0), gate != 0 ? w.size(0) / 2 : w.size(0)},
      residual.options());
  torch::Tensor sum, none;
  if (delta.has_value()) sum = torch::empty_like(residual);
  gemv_norm(out, sum, delta.has_value() ? *delta : none, residual, weight, eps,
            w, bias, gate);
  return std::make_tuple(out, delta.has_value() ? sum : residual);
}

// Whether moe_few takes a step: x [T, D], gate_up [E, 2 F, D], down [E, D, F].
bool moe_few_takes(const torch::Tensor& x, const torch::Tensor& gate_up,
                   const torch::Tensor& down, int64_t top_k, bool anywhere) {
  if (!(anywhere || x.is_cuda()) || x.dim() != 2 || gate_up.dim() != 3 ||
      down.dim() != 3 ||
      !(top_k == 1 || top_k == 2 || top_k == 4 || top_k == 8) ||
      !call_is_plain())
    return false;
  for (const auto* t : {&x, &gate_up, &down})
    if (!plain_bf16(*t, x.device()) || !t->is_contiguous() || !by16(*t))
      return false;
  const int64_t D = x.size(1), F = down.size(2), E = gate_up.size(0);
  return gate_up.size(1) == 2 * F && gate_up.size(2) == D &&
         down.size(0) == E && down.size(1) == D &&
         moe_few_fits(x.size(0), top_k, D, F);
}

// Whether moe_pick takes the router's product of these tokens.
bool moe_pick_takes(const torch::Tensor& x, const torch::Tensor& w, int64_t top_k,
                    bool anywhere) {
  return call_fits(x, w, c10::nullopt, false, anywhere) && x.size(0) <= 64 &&
         x.size(1) % 8 == 0 && x.size(1) <= (1 << 20) && w.size(0) <= 64 &&
         top_k <= w.size(0) &&
         (top_k == 1 || top_k == 2 || top_k == 4 || top_k == 8);
}

// Weights and indices of the top_k experts of each token; None where it does not
// take the call.
c10::optional<std::tuple<torch::Tensor, torch::Tensor>> moe_pick(
    torch::Tensor x, torch::Tensor w, int64_t top_k) {
  if (!moe_pick_takes(x, w, top_k, false)) return c10::nullopt;
  const c10::cuda::CUDAGuard guard(x.device());
  auto weights = torch::empty({x.size(0), top_k}, x.options().dtype(torch::kFloat32));
  auto idx = torch::empty({x.size(0), top_k}, x.options().dtype(torch::kInt32));
  moe_pick_rows(weights, idx, x, w);
  return std::make_tuple(weights, idx);
}

// Whether the grouped products take a step of any number of tokens.
bool moe_rows_takes(const torch::Tensor& x, const torch::Tensor& gate_up,
                    const torch::Tensor& down, int64_t top_k, bool anywhere) {
  if (!(anywhere || x.is_cuda()) || x.dim() != 2 || gate_up.dim() != 3 ||
      down.dim() != 3 ||
      !(top_k == 1 || top_k == 2 || top_k == 4 || top_k == 8) ||
      !call_is_plain())
    return false;
  for (const auto* t : {&x, &gate_up, &down})
    if (!plain_bf16(*t, x.device()) || !t->is_contiguous() || !by16(*t))
      return false;
  const int64_t T = x.size(0), D = x.size(1), F = down.size(2),
                E = gate_up.size(0);
  return gate_up.size(1) == 2 * F && gate_up.size(2) == D &&
         down.size(0) == E && down.size(1) == D && E >= top_k && E <= 64 &&
         T >= 1 && T < (1 << 25) && D >= 384 && D % 128 == 0 && F >= 384 &&
         F % 128 == 0 && wide_gemm_fits(D, F, D, true) &&
         wide_gemm_fits(F, D, F, false);
}

}  // namespace igw
