// Python bindings for the MI355X (gfx950) HIP kernel library.
//
// Every op here is a hand-written CDNA4 kernel (see the .hip files); the
// Python side (inference_gateway_amd/ops/__init__.py) requires this
// extension whenever a GPU is present — there is no silent eager fallback
// on the GPU path.

#include <torch/extension.h>

namespace igw {
void rmsnorm(torch::Tensor out, torch::Tensor in, torch::Tensor weight,
             double eps);
void fused_add_rmsnorm(torch::Tensor x, torch::Tensor residual,
                       torch::Tensor weight, double eps);
void rotary_embedding(torch::Tensor positions, torch::Tensor q,
                      torch::Tensor k, int64_t head_dim,
                      torch::Tensor cos_sin_cache);
void rope_append(torch::Tensor positions, torch::Tensor q, torch::Tensor k,
                 torch::Tensor v, torch::Tensor cos_sin_cache,
                 torch::Tensor kcache, torch::Tensor vcache,
                 torch::Tensor slot_mapping);
void append_kv_cache(torch::Tensor k, torch::Tensor v, torch::Tensor kcache,
                     torch::Tensor vcache, torch::Tensor slot_mapping);
void rope_paged_attn_decode(torch::Tensor out, torch::Tensor positions,
                            torch::Tensor q, torch::Tensor k, torch::Tensor v,
                            torch::Tensor cos_sin_cache, torch::Tensor kcache,
                            torch::Tensor vcache, torch::Tensor slot_mapping,
                            torch::Tensor block_table, torch::Tensor ctx_lens,
                            double scale);
void paged_attn_decode(torch::Tensor out, torch::Tensor q,
                       torch::Tensor kcache, torch::Tensor vcache,
                       torch::Tensor block_table, torch::Tensor ctx_lens,
                       double scale);
void flash_prefill(torch::Tensor out, torch::Tensor q, torch::Tensor k,
                   torch::Tensor v, torch::Tensor cu_seqlens,
                   std::vector<int64_t> seq_lens, double scale);
void flash_prefill_paged(torch::Tensor out, torch::Tensor q,
                         torch::Tensor kcache, torch::Tensor vcache,
                         torch::Tensor block_table, torch::Tensor prefix_lens,
                         torch::Tensor cu_seqlens,
                         std::vector<int64_t> seq_lens, double scale);
int64_t rows_gemm_splits(int64_t M, int64_t N, int64_t K, bool swiglu);
void gemv(torch::Tensor out, torch::Tensor x, torch::Tensor w,
          c10::optional<torch::Tensor> bias, int64_t gate);
void rows_gemm(torch::Tensor out, torch::Tensor x, torch::Tensor w,
               c10::optional<torch::Tensor> bias, int64_t gate);
int64_t wide_gemm_tile(int64_t M, int64_t N, int64_t K, bool swiglu);
void wide_gemm(torch::Tensor out, torch::Tensor x, torch::Tensor w,
               int64_t gate, int64_t tile);
bool moe_pick_takes(const torch::Tensor& x, const torch::Tensor& w, int64_t top_k,
                    bool anywhere);
c10::optional<std::tuple<torch::Tensor, torch::Tensor>> moe_pick(
    torch::Tensor x, torch::Tensor w, int64_t top_k);
bool norm_linear_takes(const c10::optional<torch::Tensor>& delta,
                       const torch::Tensor& residual,
                       const torch::Tensor& weight, const torch::Tensor& w,
                       const c10::optional<torch::Tensor>& bias, bool swiglu,
                       bool anywhere);
c10::optional<std::tuple<torch::Tensor, torch::Tensor>> norm_linear(
    const c10::optional<torch::Tensor>& delta, const torch::Tensor& residual,
    const torch::Tensor& weight, double eps, const torch::Tensor& w,
    const c10::optional<torch::Tensor>& bias, int64_t gate);
int64_t narrow_takes(const torch::Tensor& x, const torch::Tensor& w,
                     const c10::optional<torch::Tensor>& bias, bool swiglu,
                     bool anywhere);
void narrow_gemm(torch::Tensor out, torch::Tensor x, torch::Tensor w,
                 int64_t gate, int64_t tile);
int64_t wide_split(int64_t M, int64_t N, int64_t K);
torch::Tensor split_parts(const torch::Tensor& x, const torch::Tensor& w,
                          int64_t tile, int64_t S);
void sum_parts(torch::Tensor out, const torch::Tensor& part,
               const c10::optional<torch::Tensor>& bias);
void sum_add_rmsnorm(torch::Tensor out, torch::Tensor part,
                     torch::Tensor residual, torch::Tensor weight, double eps);
int64_t linear_norm_takes(const torch::Tensor& x, const torch::Tensor& w,
                          const torch::Tensor& residual,
                          const torch::Tensor& weight, bool anywhere);
c10::optional<torch::Tensor> linear_add_rmsnorm(const torch::Tensor& x,
                                                const torch::Tensor& w,
                                                const torch::Tensor& residual,
                                                const torch::Tensor& weight,
                                                double eps);
c10::optional<torch::Tensor> linear_parts(const torch::Tensor& x,
                                          const torch::Tensor& w);
void held_gemm(torch::Tensor out, torch::Tensor x, torch::Tensor w,
               c10::optional<torch::Tensor> bias);
int64_t product_kernel(const torch::Tensor& x, const torch::Tensor& w,
                       const c10::optional<torch::Tensor>& bias, int64_t gate,
                       bool anywhere);
int64_t few_rows_takes(const torch::Tensor& x, const torch::Tensor& w,
                       const c10::optional<torch::Tensor>& bias, bool swiglu,
                       bool anywhere);
c10::optional<torch::Tensor> few_rows(const torch::Tensor& x,
                                      const torch::Tensor& w,
                                      const c10::optional<torch::Tensor>& bias,
                                      int64_t gate);
bool moe_few_takes(const torch::Tensor& x, const torch::Tensor& gate_up,
                   const torch::Tensor& down, int64_t top_k, bool anywhere);
bool moe_rows_takes(const torch::Tensor& x, const torch::Tensor& gate_up,
                    const torch::Tensor& down, int64_t top_k, bool anywhere);
int64_t grouped_tile(int64_t rows, int64_t E, int64_t N, bool swiglu);
void grouped_gemm(torch::Tensor out, torch::Tensor x, torch::Tensor w,
                  torch::Tensor start, bool swiglu, int64_t tile);
void moe_dispatch(torch::Tensor weights, torch::Tensor dst,
                  torch::Tensor start, torch::Tensor logits);
void moe_scatter_rows(torch::Tensor buf, torch::Tensor x, torch::Tensor dst,
                      int64_t K);
void moe_combine(torch::Tensor out, torch::Tensor y, torch::Tensor dst,
                 torch::Tensor w, c10::optional<torch::Tensor> shared,
                 c10::optional<torch::Tensor> g);
void moe_few(torch::Tensor out, torch::Tensor x, torch::Tensor gate_up,
             torch::Tensor down, torch::Tensor idx, torch::Tensor weight);
void sample(torch::Tensor out, torch::Tensor logits, torch::Tensor temperature,
            torch::Tensor top_k, torch::Tensor top_p, torch::Tensor uniforms);
void silu_mul(torch::Tensor out, torch::Tensor gate_up);
void moe_route(torch::Tensor weights, torch::Tensor dst,
               torch::Tensor topk_idx, torch::Tensor counts,
               torch::Tensor logits, int64_t C);
void moe_grouped_gemm(torch::Tensor out, torch::Tensor a, torch::Tensor w,
                      torch::Tensor counts, int64_t capacity);
void silu_mul_grouped(torch::Tensor out, torch::Tensor gate_up,
                      torch::Tensor counts, int64_t capacity);
void fused_gemm_tn(torch::Tensor out, torch::Tensor x, torch::Tensor w,
                   bool swiglu, bool nt_weights);
void fused_gemm_tn2(torch::Tensor out, torch::Tensor x, torch::Tensor w,
                    bool swiglu, bool swz);
void glds_probe(torch::Tensor out, torch::Tensor inp, int64_t swizzle);
int64_t ar_alloc(int64_t bytes, bool finegrained);
void ar_free(int64_t ptr);
py::bytes ar_get_handle(int64_t ptr);
int64_t ar_open_handle(py::bytes handle);
void ar_close_handle(int64_t ptr);
int64_t ar_sig_bytes();
int64_t ar_check_error(int64_t sig_ptr);
py::bytes ar_dump(int64_t ptr, int64_t nbytes);
void oneshot_allreduce(torch::Tensor inout, int64_t rank, int64_t world,
                       std::vector<int64_t> data_ptrs,
                       std::vector<int64_t> sig_ptrs,
                       int64_t buf_stride_elems);
}  // namespace igw

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("rmsnorm", &igw::rmsnorm, "RMSNorm (bf16, gfx950)");
  m.def("fused_add_rmsnorm", &igw::fused_add_rmsnorm,
        "residual += x; x = rmsnorm(residual) (bf16, gfx950)");
  m.def("rotary_embedding", &igw::rotary_embedding,
        "NeoX-style RoPE in-place on q/k (bf16, gfx950)");
  m.def("rope_append", &igw::rope_append,
        "RoPE of q and k, k and v into the paged cache");
  m.def("append_kv_cache", &igw::append_kv_cache,
        "scatter step K/V into the paged cache (bf16, gfx950)");
  m.def("rope_paged_attn_decode", &igw::rope_paged_attn_decode,
        "rope_append and paged_attn_decode in one launch");
  m.def("paged_attn_decode", &igw::paged_attn_decode,
        "GQA paged-attention decode (bf16, gfx950)");
  m.def("flash_prefill", &igw::flash_prefill,
        "varlen causal MFMA flash-attention prefill (bf16, gfx950)");
  m.def("few_rows", &igw::few_rows,
        "x W^T by gemv, rows_gemm, held_gemm or wide_gemm, None: none of them "
        "takes it");
  m.def("gemv", &igw::gemv,
        "x W^T for a few rows of x, optional bias or SwiGLU");
  m.def("rows_gemm", &igw::rows_gemm, "x W^T of tens of rows");
  m.def("held_gemm", &igw::held_gemm,
        "x W^T of tens of rows, x in registers", py::arg("out"), py::arg("x"),
        py::arg("w"), py::arg("bias") = py::none());
  m.def("moe_pick_takes", &igw::moe_pick_takes,
        "whether moe_pick takes the call");
  m.def("moe_pick", &igw::moe_pick,
        "router product and the chosen experts of a few tokens, or None");
  m.def("norm_linear_takes", &igw::norm_linear_takes,
        "whether gemv has the norm before it inside");
  m.def("norm_linear", &igw::norm_linear,
        "rmsnorm(residual + delta) W^T and residual + delta, None: nothing done");
  m.def("narrow_takes", &igw::narrow_takes,
        "narrow_gemm's tile of a call that it takes, 0: it does not");
  m.def("narrow_gemm", &igw::narrow_gemm, "x W^T on tiles of few columns");
  m.def("wide_split", &igw::wide_split,
        "256 x the tile + the parts of K of a product that leaves the chip idle");
  m.def("split_parts", &igw::split_parts, "sums of the parts of K of x W^T");
  m.def("sum_parts", &igw::sum_parts, "out = the parts' sum (+ bias)");
  m.def("sum_add_rmsnorm", &igw::sum_add_rmsnorm,
        "residual += the parts' sum, out = its norm");
  m.def("linear_norm_takes", &igw::linear_norm_takes,
        "as few_rows_takes, of a product in parts that a norm follows");
  m.def("linear_add_rmsnorm", &igw::linear_add_rmsnorm,
        "residual += x W^T and its norm, None: nothing done");
  m.def("linear_parts", &igw::linear_parts,
        "the sums of the parts of K of x W^T, None: not in parts");
  m.def("wide_gemm", &igw::wide_gemm,
        "x W^T of hundreds to thousands of rows on a given tile");
  m.def("wide_gemm_tile", &igw::wide_gemm_tile,
        "its tile (16 MT + NT) for a product; 0: not ahead of the library");
  m.def("product_kernel", &igw::product_kernel,
        "what runs x W^T, plain or gated (gate 1 SiLU, 2 GELU).  0: none of "
        "them, 1: gemv, 2: "
        "rows_gemm, 3: wide_gemm, 4: held_gemm, 5: wide_gemm with K in parts, "
        "6: narrow_gemm");
  m.def("few_rows_takes", &igw::few_rows_takes,
        "as product_kernel of gate 0 or 1, were narrow_gemm not there");
  m.def("moe_few", &igw::moe_few, "SwiGLU experts of a few tokens");
  m.def("moe_rows_takes", &igw::moe_rows_takes,
        "whether the grouped products take a step");
  m.def("grouped_tile", &igw::grouped_tile, "grouped_gemm's tile (16 MT + NT)");
  m.def("grouped_gemm", &igw::grouped_gemm,
        "every expert's rows of x times its weights, optional SwiGLU");
  m.def("moe_dispatch", &igw::moe_dispatch,
        "top-k, softmax weights and rows sorted by expert");
  m.def("moe_scatter_rows", &igw::moe_scatter_rows,
        "buf[dst[t*K + k]] = x[t]");
  m.def("moe_combine", &igw::moe_combine,
        "out[t] = sum_k w[t, k] y[dst[t*K + k]] (+ gated shared rows)");
  m.def("moe_few_takes", &igw::moe_few_takes, "whether moe_few takes a step");
  m.def("rows_gemm_splits", &igw::rows_gemm_splits,
        "parts of K that rows_gemm takes, 0: it does not");
  m.def("flash_prefill_paged", &igw::flash_prefill_paged,
        "paged-extend prefill: chunk queries over cached prefix+chunk K/V "
        "via block table (bf16, gfx950)");
  m.def("sample", &igw::sample,
        "fused temperature/top-k/top-p sampling (fp32 logits, gfx950)");
  m.def("silu_mul", &igw::silu_mul, "fused SwiGLU activation (bf16, gfx950)");
  m.def("moe_route", &igw::moe_route,
        "fused MoE top-k routing + softmax + padded-dispatch ranks (gfx950)");
  m.def("moe_grouped_gemm", &igw::moe_grouped_gemm,
        "grouped per-expert MFMA GEMM over the padded dispatch buffer");
  m.def("silu_mul_grouped", &igw::silu_mul_grouped,
        "SwiGLU over only the real (non-padded) MoE dispatch rows");
  m.def("glds_probe", &igw::glds_probe, "glds round-trip probe (debug)");
  m.def("fused_gemm_tn2", &igw::fused_gemm_tn2,
        "TN bf16 MFMA GEMM v2: block-shared LDS weight tiles "
        "(glds + XOR swizzle), optional fused SwiGLU");
  m.def("fused_gemm_tn", &igw::fused_gemm_tn,
        "TN bf16 MFMA GEMM with optional fused SwiGLU epilogue "
        "(decode weight-streaming shapes, gfx950)");
  m.def("ar_alloc", &igw::ar_alloc,
        "raw device allocation for one-shot all-reduce buffers "
        "(finegrained=true for signal pages)");
  m.def("ar_free", &igw::ar_free, "free an ar_alloc allocation");
  m.def("ar_get_handle", &igw::ar_get_handle,
        "hipIpcMemHandle for a raw allocation (64 bytes)");
  m.def("ar_open_handle", &igw::ar_open_handle,
        "open a peer rank's IPC handle -> device pointer");
  m.def("ar_close_handle", &igw::ar_close_handle,
        "close an opened peer IPC handle");
  m.def("ar_sig_bytes", &igw::ar_sig_bytes,
        "size of the one-shot signal page");
  m.def("ar_check_error", &igw::ar_check_error,
        "read the one-shot spin-timeout error word");
  m.def("ar_dump", &igw::ar_dump, "copy raw device bytes to host (debug)");
  m.def("oneshot_allreduce", &igw::oneshot_allreduce,
        "one-shot bf16 sum all-reduce over xGMI peer buffers "
        "(graph-capturable, device-side epochs)");
}
