// Python bindings for the petals_amd CDNA4 kernel suite.
#include <torch/extension.h>
#include <ATen/cuda/CUDAContext.h>

torch::Tensor rms_norm(torch::Tensor x, torch::Tensor w, double eps);
torch::Tensor rms_norm_f32out(torch::Tensor x, torch::Tensor w, double eps);
torch::Tensor layer_norm(torch::Tensor x, torch::Tensor w, torch::Tensor b, double eps);
torch::Tensor layer_norm_f32out(torch::Tensor x, torch::Tensor w, torch::Tensor b, double eps);
torch::Tensor swiglu(torch::Tensor gate, torch::Tensor up);
void warm_spin(int64_t microseconds);
std::vector<torch::Tensor> apply_rope(
    torch::Tensor q, torch::Tensor k, torch::Tensor cos_t, torch::Tensor sin_t, torch::Tensor pos);
void rope_cache_write(
    torch::Tensor qkv, torch::Tensor cos_t, torch::Tensor sin_t, torch::Tensor pos,
    torch::Tensor k_cache, torch::Tensor v_cache, int64_t qh, int64_t kh);
void kv_cache_write(
    torch::Tensor qkv, torch::Tensor pos,
    torch::Tensor k_cache, torch::Tensor v_cache, int64_t qh, int64_t kh);
torch::Tensor qkv_rope_reduce(
    torch::Tensor partials, c10::optional<torch::Tensor> cos_t, c10::optional<torch::Tensor> sin_t,
    torch::Tensor pos, torch::Tensor k_cache, torch::Tensor v_cache,
    int64_t qh, int64_t kh, bool rope, c10::optional<torch::Tensor> bias);
torch::Tensor gemv_bf16(
    torch::Tensor wt, torch::Tensor x, torch::Tensor workspace,
    c10::optional<torch::Tensor> residual, int64_t epilogue, int64_t splits_override,
    c10::optional<torch::Tensor> bias, c10::optional<torch::Tensor> sumsq_out);
torch::Tensor gemv_bf16_normed(
    torch::Tensor wt, torch::Tensor h, torch::Tensor w, c10::optional<torch::Tensor> sumsq, double eps,
    torch::Tensor workspace, int64_t epilogue);
torch::Tensor attn_decode_fused(
    torch::Tensor q, torch::Tensor k_cache, torch::Tensor v_cache, torch::Tensor kv_len,
    int64_t gq, int64_t n_splits, torch::Tensor part_o, torch::Tensor part_ml, double scale,
    c10::optional<torch::Tensor> alibi_slopes);
torch::Tensor attn_prefill_fused(
    torch::Tensor q, torch::Tensor k, torch::Tensor v,
    int64_t kv_len, int64_t kv_offset, double scale, bool causal,
    c10::optional<torch::Tensor> alibi_slopes);
std::vector<torch::Tensor> attn_prefill_sums(torch::Tensor q, torch::Tensor k, torch::Tensor v, double scale);
torch::Tensor attn_prompt_grad(
    torch::Tensor qkv, torch::Tensor grad_out, torch::Tensor lse, torch::Tensor cos_t,
    torch::Tensor sin_t, int64_t start, int64_t qh, int64_t kh, int64_t hd, double scale);
torch::Tensor rotate_rows(
    torch::Tensor qkv, torch::Tensor cos_t, torch::Tensor sin_t, int64_t start, int64_t qh, int64_t kh, int64_t hd);
torch::Tensor norm_rows_grad(
    torch::Tensor x, torch::Tensor w, torch::Tensor g, c10::optional<torch::Tensor> residual, double eps);
torch::Tensor swiglu_rows_grad(torch::Tensor gu, torch::Tensor g);
torch::Tensor attn_prefill_rows(
    torch::Tensor q, torch::Tensor k, torch::Tensor v, int64_t kv_len, int64_t kv_offset, double scale, bool causal,
    c10::optional<torch::Tensor> alibi_slopes);
void qkv_rows(
    torch::Tensor qkv, c10::optional<torch::Tensor> bias, c10::optional<torch::Tensor> cos_t,
    c10::optional<torch::Tensor> sin_t, c10::optional<torch::Tensor> k_cache, c10::optional<torch::Tensor> v_cache,
    int64_t start, int64_t qh, int64_t kh, int64_t hd);
std::vector<torch::Tensor> add_norm_rows(
    torch::Tensor x, torch::Tensor y, c10::optional<torch::Tensor> y_bias, torch::Tensor w,
    c10::optional<torch::Tensor> b, double eps);
torch::Tensor add_rows(torch::Tensor x, torch::Tensor y, c10::optional<torch::Tensor> z, c10::optional<torch::Tensor> bias);
torch::Tensor swiglu_rows(torch::Tensor gu);
torch::Tensor gemm_rows(torch::Tensor x, torch::Tensor w, bool transposed, int64_t epilogue,
                        c10::optional<torch::Tensor> residual, c10::optional<torch::Tensor> bias, int64_t tile, bool steady);
torch::Tensor gemm_nf4_rows(torch::Tensor x, torch::Tensor tiles, torch::Tensor scales, int64_t epilogue,
                            c10::optional<torch::Tensor> residual, c10::optional<torch::Tensor> bias, int64_t tile);
void bias_gelu_rows(torch::Tensor y, c10::optional<torch::Tensor> bias);
std::vector<torch::Tensor> nf4_quantize(torch::Tensor w);
torch::Tensor gemv_int8(
    torch::Tensor q, torch::Tensor scale, torch::Tensor x, torch::Tensor workspace,
    c10::optional<torch::Tensor> residual, int64_t epilogue, int64_t splits_override,
    c10::optional<torch::Tensor> bias);
torch::Tensor nf4_dequantize(torch::Tensor packed, torch::Tensor absmax);
torch::Tensor gemv_nf4(
    torch::Tensor packed, torch::Tensor absmax, torch::Tensor x, torch::Tensor workspace,
    c10::optional<torch::Tensor> residual, int64_t epilogue, int64_t splits_override,
    c10::optional<torch::Tensor> bias, c10::optional<torch::Tensor> absmax_t,
    c10::optional<torch::Tensor> x_parts, double fold_eps,
    c10::optional<torch::Tensor> sumsq_out);
torch::Tensor sumsq_rows(torch::Tensor x);
torch::Tensor gemv_bf16_moe(
    torch::Tensor wt_all, torch::Tensor x, torch::Tensor sel, int64_t k_per_tok,
    torch::Tensor workspace, int64_t epilogue, int64_t splits_override, double limit, double alpha);
std::vector<torch::Tensor> nf4_tile(torch::Tensor packed, torch::Tensor absmax);
torch::Tensor nf4_untile(torch::Tensor tiles, torch::Tensor scales, int64_t in_dim);
torch::Tensor gemv_nf4_tiles(
    torch::Tensor tiles, torch::Tensor scales, int64_t in_dim, torch::Tensor x, torch::Tensor workspace,
    c10::optional<torch::Tensor> residual, int64_t epilogue, c10::optional<torch::Tensor> bias);
torch::Tensor gemv_nf4_tiles_moe(
    torch::Tensor tiles, torch::Tensor scales, int64_t in_dim, torch::Tensor x, torch::Tensor sel,
    int64_t k_per_tok, torch::Tensor workspace, int64_t epilogue);
std::vector<torch::Tensor> moe_route(torch::Tensor x, torch::Tensor w, int64_t top);
torch::Tensor moe_combine(torch::Tensor rows, torch::Tensor weights, torch::Tensor residual);
std::vector<torch::Tensor> moe_group(torch::Tensor sel, int64_t experts, int64_t mt);
torch::Tensor moe_gemm(
    c10::optional<torch::Tensor> wt_all, c10::optional<torch::Tensor> nf4_all,
    c10::optional<torch::Tensor> scales_all, torch::Tensor x, torch::Tensor sorted_pairs,
    torch::Tensor tile_expert, int64_t k_per_tok, int64_t n_rows, bool general);

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("rms_norm", &rms_norm, "RMSNorm (bf16 -> bf16)");
  m.def("rms_norm_f32out", &rms_norm_f32out, "RMSNorm (bf16 -> f32)");
  m.def("layer_norm", &layer_norm, "LayerNorm with weight+bias (bf16 -> bf16)");
  m.def("layer_norm_f32out", &layer_norm_f32out, "LayerNorm with weight+bias (bf16 -> f32)");
  m.def("swiglu", &swiglu, "silu(gate) * up (bf16)");
  m.def("warm_spin", &warm_spin, "occupy the device queue for ~N us (keep-warm)");
  m.def("apply_rope", &apply_rope, "rotate q,k by positions (bf16)");
  m.def("rope_cache_write", &rope_cache_write, "fused decode rope + kv cache write");
  m.def("kv_cache_write", &kv_cache_write, "decode kv cache write without rope (ALiBi families)");
  m.def("qkv_rope_reduce", &qkv_rope_reduce,
        "fused qkv split-K reduce + rope + kv-cache write (consumes RAW gemv partials)",
        py::arg("partials"), py::arg("cos_t"), py::arg("sin_t"), py::arg("pos"),
        py::arg("k_cache"), py::arg("v_cache"), py::arg("qh"), py::arg("kh"), py::arg("rope") = true,
        py::arg("bias") = py::none());
  m.def("gemv_bf16", &gemv_bf16, "split-K bf16 gemv with fused epilogue",
        py::arg("wt"), py::arg("x"), py::arg("workspace"), py::arg("residual"), py::arg("epilogue"),
        py::arg("splits") = 0, py::arg("bias") = py::none(), py::arg("sumsq_out") = py::none());
  m.def("gemv_bf16_normed", &gemv_bf16_normed, "gemv_bf16 of the RMS norm of bf16 rows",
        py::arg("wt"), py::arg("h"), py::arg("w"), py::arg("sumsq"), py::arg("eps"), py::arg("workspace"),
        py::arg("epilogue"));
  m.def("attn_decode_fused", &attn_decode_fused, "GQA decode attention (flash-decoding)",
        py::arg("q"), py::arg("k_cache"), py::arg("v_cache"), py::arg("kv_len"), py::arg("gq"),
        py::arg("n_splits"), py::arg("part_o"), py::arg("part_ml"), py::arg("scale"),
        py::arg("alibi_slopes") = py::none());
  m.def("attn_prefill_fused", &attn_prefill_fused, "MFMA flash prefill attention (bf16, causal, GQA)",
        py::arg("q"), py::arg("k"), py::arg("v"), py::arg("kv_len"), py::arg("kv_offset"),
        py::arg("scale"), py::arg("causal"), py::arg("alibi_slopes") = py::none());
  m.def("gemv_int8", &gemv_int8, "split-K weight-only int8 gemv (per-column scales) with epilogue",
        py::arg("q"), py::arg("scale"), py::arg("x"), py::arg("workspace"),
        py::arg("residual"), py::arg("epilogue"), py::arg("splits") = 0, py::arg("bias") = py::none());
  m.def("nf4_quantize", &nf4_quantize, "blockwise NF4 quantize [in,out] bf16 -> (packed u8, absmax bf16)");
  m.def("nf4_dequantize", &nf4_dequantize, "NF4 -> bf16");
  m.def("gemv_nf4", &gemv_nf4, "split-K NF4 gemv (dequant fused) with epilogue; "
        "x_parts switches to the folded-RMSNorm mode (bf16 x + sum(h^2) partials)",
        py::arg("packed"), py::arg("absmax"), py::arg("x"), py::arg("workspace"),
        py::arg("residual"), py::arg("epilogue"), py::arg("splits") = 0, py::arg("bias") = py::none(),
        py::arg("absmax_t") = py::none(), py::arg("x_parts") = py::none(),
        py::arg("fold_eps") = 0.0, py::arg("sumsq_out") = py::none());
  m.def("sumsq_rows", &sumsq_rows, "per-row sum(x^2) of a bf16 matrix -> [rows, 1] f32");
  m.def("gemv_bf16_moe", &gemv_bf16_moe,
        "device-routed MoE gemv: stacked bf16 expert weights, expert ids from a device tensor",
        py::arg("wt_all"), py::arg("x"), py::arg("sel"), py::arg("k_per_tok"),
        py::arg("workspace"), py::arg("epilogue"), py::arg("splits") = 0,
        py::arg("limit") = 0.0, py::arg("alpha") = 0.0);
  m.def("attn_prefill_rows", &attn_prefill_rows, "prompt attention on strided heads; results as rows of tokens");
  m.def("attn_prefill_sums", &attn_prefill_sums, "causal prompt attention with log2 of its rows' sums of weights");
  m.def("attn_prompt_grad", &attn_prompt_grad, "gradient of a fused projection through rotation and causal attention");
  m.def("rotate_rows", &rotate_rows, "fused projection with queries and keys rotated");
  m.def("norm_rows_grad", &norm_rows_grad, "gradient of an RMS norm's rows (+ residual)");
  m.def("swiglu_rows_grad", &swiglu_rows_grad, "gradient of [gate | up] rows");
  m.def("qkv_rows", &qkv_rows, "fused projection of a prompt -> rotated queries in place, keys and values to the cache");
  m.def("add_norm_rows", &add_norm_rows, "(x + y + bias, its RMS or layer norm)",
        py::arg("x"), py::arg("y"), py::arg("y_bias"), py::arg("w"), py::arg("b"), py::arg("eps"));
  m.def("add_rows", &add_rows, "x + y (+ z) (+ bias)",
        py::arg("x"), py::arg("y"), py::arg("z") = py::none(), py::arg("bias") = py::none());
  m.def("gemm_rows", &gemm_rows, "a prompt's rows times a bf16 matrix, and what follows", py::arg("x"), py::arg("w"),
        py::arg("transposed") = false, py::arg("epilogue") = 0, py::arg("residual") = py::none(),
        py::arg("bias") = py::none(), py::arg("tile") = -1, py::arg("steady") = false);
  m.def("gemm_nf4_rows", &gemm_nf4_rows, "a prompt's rows times NF4 tiles, and what follows", py::arg("x"), py::arg("tiles"),
        py::arg("scales"), py::arg("epilogue") = 0, py::arg("residual") = py::none(), py::arg("bias") = py::none(),
        py::arg("tile") = -1);
  m.def("swiglu_rows", &swiglu_rows, "[..., gate | up] -> silu(gate) * up");
  m.def("bias_gelu_rows", &bias_gelu_rows, "gelu(y + bias), in place", py::arg("y"), py::arg("bias") = py::none());
  m.def("nf4_tile", &nf4_tile, "NF4 in the order of the matrix cores: (packed, absmax) -> (tiles, scales)");
  m.def("nf4_untile", &nf4_untile, "(tiles, scales) -> bf16 [in, out]");
  m.def("gemv_nf4_tiles", &gemv_nf4_tiles, "few rows times NF4 tiles, with epilogue",
        py::arg("tiles"), py::arg("scales"), py::arg("in_dim"), py::arg("x"), py::arg("workspace"),
        py::arg("residual"), py::arg("epilogue"), py::arg("bias") = py::none());
  m.def("gemv_nf4_tiles_moe", &gemv_nf4_tiles_moe,
        "device-routed MoE gemv: stacked NF4 tiles, expert ids from a device tensor",
        py::arg("tiles"), py::arg("scales"), py::arg("in_dim"), py::arg("x"), py::arg("sel"),
        py::arg("k_per_tok"), py::arg("workspace"), py::arg("epilogue"));
  m.def("moe_route", &moe_route, "router, softmax, top-k, renormalized: (weights, experts)");
  m.def("moe_combine", &moe_combine, "residual + weighted sum of a token's expert rows");
  m.def("moe_group", &moe_group, "expert-sorted, tile-padded pairs");
  m.def("moe_gemm", &moe_gemm,
        "grouped MFMA GEMM over expert-sorted (token, slot) pairs (prefill; NF4 dequant fused "
        "into the LDS B-tile staging)",
        py::arg("wt_all"), py::arg("nf4_all"), py::arg("scales_all"), py::arg("x"),
        py::arg("sorted_pairs"), py::arg("tile_expert"), py::arg("k_per_tok"), py::arg("n_rows"), py::arg("general") = false);
}
