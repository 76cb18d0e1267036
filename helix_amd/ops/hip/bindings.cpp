// Python bindings for the helix_amd CDNA4 kernel library.
#include <torch/extension.h>

void rms_norm(torch::Tensor out, torch::Tensor x, torch::Tensor w, double eps);
void fused_add_rms_norm(torch::Tensor x, torch::Tensor residual,
                        torch::Tensor w, double eps);
bool add_norm(c10::optional<torch::Tensor> sum, torch::Tensor out,
              torch::Tensor x, c10::optional<torch::Tensor> y,
              c10::optional<torch::Tensor> gate, torch::Tensor a,
              torch::Tensor b, int64_t L, double eps,
              c10::optional<torch::Tensor> y_bias);
torch::Tensor gemm_bf16_summand(torch::Tensor x, torch::Tensor w,
                                torch::Tensor bias);
bool text_embed(torch::Tensor out, torch::Tensor ids, torch::Tensor cu,
                torch::Tensor word, torch::Tensor pos, torch::Tensor w,
                torch::Tensor b, double eps);
bool text_pool(torch::Tensor out, torch::Tensor x, torch::Tensor cu);
bool image_rows(torch::Tensor out, torch::Tensor lat, int64_t patch);
bool image_velocity(torch::Tensor out, torch::Tensor rows, int64_t patch,
                    int64_t text);
bool image_tokens(torch::Tensor x, torch::Tensor cond, torch::Tensor cu,
                  torch::Tensor ids, torch::Tensor word, torch::Tensor pos,
                  torch::Tensor image);
bool time_embed(torch::Tensor out, torch::Tensor t);
c10::optional<torch::Tensor> text_block(
    torch::Tensor x, torch::Tensor cu, int64_t max_len, int64_t heads,
    double scale, double eps, std::vector<c10::optional<torch::Tensor>> p);
std::vector<torch::Tensor> text_block_first(
    torch::Tensor x, torch::Tensor cu, int64_t max_len, int64_t heads,
    double scale, double eps, std::vector<c10::optional<torch::Tensor>> p);
std::vector<torch::Tensor> image_block(
    torch::Tensor x, c10::optional<torch::Tensor> y,
    c10::optional<torch::Tensor> gate, c10::optional<torch::Tensor> y_bias,
    torch::Tensor mod, torch::Tensor cu, int64_t L, int64_t heads,
    double scale, double eps, std::vector<c10::optional<torch::Tensor>> p,
    bool stretches);
bool gated_add(torch::Tensor out, torch::Tensor x, torch::Tensor y,
               torch::Tensor gate, int64_t L);
bool norm_in_registers(int64_t rows, int64_t columns);
void add_sums_rms_norm(torch::Tensor h, torch::Tensor x,
                       torch::Tensor residual, torch::Tensor w, double eps);
void add_sums_rms_norm_fp8(torch::Tensor h, torch::Tensor scales,
                           torch::Tensor x, torch::Tensor residual,
                           torch::Tensor w, double eps);
void layer_norm(torch::Tensor out, torch::Tensor x, torch::Tensor w,
                torch::Tensor b, double eps);
void rotary_embedding(torch::Tensor positions, torch::Tensor q,
                      torch::Tensor k, torch::Tensor cos_sin,
                      int64_t head_dim);
void silu_and_mul(torch::Tensor out, torch::Tensor x);
void rope_qkv_cache(torch::Tensor positions, torch::Tensor qkv,
                    torch::Tensor q_out,
                    c10::optional<torch::Tensor> k_cache,
                    c10::optional<torch::Tensor> v_cache,
                    c10::optional<torch::Tensor> slot_mapping,
                    c10::optional<torch::Tensor> k_out,
                    c10::optional<torch::Tensor> v_out,
                    torch::Tensor cos_sin, int64_t num_q_heads,
                    int64_t num_kv_heads, int64_t head_dim);
void gelu_tanh(torch::Tensor out, torch::Tensor x);
void reshape_and_cache(torch::Tensor k, torch::Tensor v,
                       torch::Tensor k_cache, torch::Tensor v_cache,
                       torch::Tensor slot_mapping);
void gather_kv(torch::Tensor k, torch::Tensor v, torch::Tensor k_cache,
               torch::Tensor v_cache, torch::Tensor blk, torch::Tensor off);
void paged_attn_decode(torch::Tensor out, torch::Tensor q,
                       torch::Tensor k_cache, torch::Tensor v_cache,
                       torch::Tensor block_tables, torch::Tensor seq_lens,
                       double scale, torch::Tensor tmp_out,
                       torch::Tensor tmp_ml, int64_t partition_size,
                       int64_t window);
void attn_prefill(torch::Tensor out, torch::Tensor q, torch::Tensor k,
                  torch::Tensor v, torch::Tensor cu_seqlens,
                  torch::Tensor cu_seqlens_k, int64_t max_seqlen,
                  double scale, bool causal, int64_t window);
bool attn_mixed(torch::Tensor out_p, torch::Tensor q_p, torch::Tensor k,
                torch::Tensor v, torch::Tensor cu_seqlens,
                torch::Tensor cu_seqlens_k, int64_t max_seqlen,
                torch::Tensor out_d, torch::Tensor q_d, torch::Tensor k_cache,
                torch::Tensor v_cache, torch::Tensor block_tables,
                torch::Tensor seq_lens, torch::Tensor tmp_out,
                torch::Tensor tmp_ml, int64_t max_len, double scale,
                int64_t window);
void sample_tokens(torch::Tensor out, torch::Tensor logits,
                   torch::Tensor temperatures, torch::Tensor seeds);
void sample_tokens_ext(torch::Tensor out, torch::Tensor logits,
                       torch::Tensor temperatures, torch::Tensor seeds,
                       torch::Tensor top_p, torch::Tensor top_k,
                       torch::Tensor rep_pen, torch::Tensor pres_pen,
                       torch::Tensor freq_pen,
                       c10::optional<torch::Tensor> counts,
                       c10::optional<torch::Tensor> seen,
                       c10::optional<torch::Tensor> row_map);
void gemm_bf16(torch::Tensor out, torch::Tensor x, torch::Tensor w,
               c10::optional<torch::Tensor> bias, int64_t act, int64_t tile);
torch::Tensor gemm_bf16_sums(torch::Tensor x, torch::Tensor w, int64_t tile,
                             int64_t stretches);
std::tuple<int64_t, int64_t, double, int64_t> gemm_bf16_plan(
    int64_t M, int64_t N, int64_t K, bool gelu, bool sums, int64_t cus,
    double below);
std::tuple<bool, int64_t, int64_t, int64_t, double> gemm_bf16_cut(
    int64_t M, int64_t N, int64_t K, bool gelu, int64_t cus);
std::tuple<bool, int64_t, int64_t, int64_t, double> gemm_bf16_glu_cut(
    int64_t M, int64_t N, int64_t K, int64_t cus);
std::tuple<int64_t, int64_t> gemm_bf16_glu_plan(int64_t M, int64_t N, int64_t K,
                                                int64_t cus);
std::vector<int64_t> gemm_ring_places(std::vector<int64_t> k, int64_t steps,
                                      int64_t turn);
void gemm_bf16_glu(torch::Tensor out, torch::Tensor x, torch::Tensor w,
                   int64_t tile);
void gemm_skinny_bf16(torch::Tensor out, torch::Tensor x, torch::Tensor w,
                      c10::optional<torch::Tensor> bias,
                      c10::optional<torch::Tensor> scratch, int64_t split_k,
                      int64_t act, int64_t swizzle);
using OptT = c10::optional<torch::Tensor>;
void gemm_rows(torch::Tensor out, torch::Tensor x, torch::Tensor w, OptT bias,
               OptT x_scale, OptT w_scale, bool gelu);
torch::Tensor gemm_rows_sums(torch::Tensor x, torch::Tensor w, OptT x_scale,
                             OptT w_scale);
std::vector<torch::Tensor> gemm_rows_many(torch::Tensor x,
                                          std::vector<torch::Tensor> ws,
                                          std::vector<OptT> biases);
void gemm_rows_glu(torch::Tensor out, torch::Tensor x, torch::Tensor w,
                   OptT x_scale, OptT w_scale);
std::vector<torch::Tensor> layer_rows_join(torch::Tensor x, torch::Tensor w,
                                           torch::Tensor residual,
                                           torch::Tensor norm);
torch::Tensor layer_rows_glu(torch::Tensor x, torch::Tensor w, OptT squares,
                             double eps);
void layer_rows_qkv(torch::Tensor x, torch::Tensor w, OptT bias, OptT squares,
                    double eps, torch::Tensor positions, torch::Tensor cos_sin,
                    torch::Tensor q, OptT k, OptT v, OptT k_cache,
                    OptT v_cache, OptT slots, int64_t num_q, int64_t num_kv,
                    int64_t head_dim, OptT x_scale, OptT w_scale);
void quantize_rows(torch::Tensor out, torch::Tensor scales, torch::Tensor x);
void gemm_fp8(torch::Tensor out, torch::Tensor x, torch::Tensor w,
              torch::Tensor x_scale, torch::Tensor w_scale,
              c10::optional<torch::Tensor> bias, int64_t act);
void mfma_probe(torch::Tensor d, torch::Tensor a, torch::Tensor b);
torch::Tensor ar_create(int64_t world, int64_t rank, int64_t capacity);
void ar_open(std::vector<torch::Tensor> handles);
int64_t ar_capacity();
void ar_allreduce(torch::Tensor inp, torch::Tensor out);
void ar_destroy();
void mfma_probe_fp8(torch::Tensor d, torch::Tensor a, torch::Tensor b,
                    int64_t scale_a, int64_t scale_b);

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("rms_norm", &rms_norm, "RMSNorm (bf16, CDNA4)");
  m.def("fused_add_rms_norm", &fused_add_rms_norm,
        "Fused residual-add + RMSNorm (in-place)");
  m.def("add_norm", &add_norm,
        "(Gated) add + LayerNorm with weights or an image's modulation",
        py::arg("sum"), py::arg("out"), py::arg("x"), py::arg("y"),
        py::arg("gate"), py::arg("a"), py::arg("b"), py::arg("L"),
        py::arg("eps"), py::arg("y_bias") = py::none());
  m.def("gemm_bf16_summand", &gemm_bf16_summand,
        "x @ w^T + bias as rows, or its stretches for a norm that adds them up");
  m.def("gated_add", &gated_add, "x + gate * y, a gate per image");
  m.def("text_embed", &text_embed,
        "LayerNorm of a text's word and position embeddings");
  m.def("text_pool", &text_pool, "First rows of texts, divided by their length");
  m.def("image_rows", &image_rows, "Patches of latents as rows");
  m.def("image_velocity", &image_velocity, "Rows of image tokens as latents");
  m.def("image_tokens", &image_tokens,
        "Text and image rows with their places, mean of the text");
  m.def("time_embed", &time_embed, "Sinusoidal embedding of times");
  m.def("text_block", &text_block, "A block of the text encoder");
  m.def("text_block_first", &text_block_first,
        "A block of the text encoder, for the first row of each text");
  m.def("image_block", &image_block, "A block of the image model");
  m.def("norm_in_registers", &norm_in_registers,
        "Whether add_sums_rms_norm keeps a row in registers");
  m.def("add_sums_rms_norm", &add_sums_rms_norm,
        "Sum of a product's stretches + residual-add + RMSNorm");
  m.def("add_sums_rms_norm_fp8", &add_sums_rms_norm_fp8,
        "The same, rows as e4m3 bytes and scales (bf16 residual, fp32 in)");
  m.def("layer_norm", &layer_norm, "LayerNorm (bf16)");
  m.def("rotary_embedding", &rotary_embedding,
        "Apply rotary embedding to q,k in-place");
  m.def("silu_and_mul", &silu_and_mul, "Fused SiLU-gated multiply");
  m.def("rope_qkv_cache", &rope_qkv_cache,
        "Fused strided-QKV rope + paged-cache write");
  m.def("gelu_tanh", &gelu_tanh, "GELU (tanh approx)");
  m.def("reshape_and_cache", &reshape_and_cache,
        "Scatter K/V rows into paged cache");
  m.def("gather_kv", &gather_kv, "Gather K/V rows from paged cache");
  m.def("paged_attn_decode", &paged_attn_decode,
        "Paged decode attention (GQA, flash-decoding partitions)");
  m.def("attn_prefill", &attn_prefill,
        "Varlen causal flash prefill attention (MFMA)");
  m.def("attn_mixed", &attn_mixed,
        "Prompt portions' and replies' attention in one launch");
  m.def("sample_tokens", &sample_tokens, "Greedy/Gumbel token sampling");
  m.def("sample_tokens_ext", &sample_tokens_ext,
        "Fused top-k/top-p/penalty Gumbel sampling (histogram threshold)");
  m.def("gemm_bf16", &gemm_bf16, "MFMA bf16 GEMM: x @ w^T (+bias, act)",
        py::arg("out"), py::arg("x"), py::arg("w"), py::arg("bias"),
        py::arg("act"), py::arg("tile") = 0);
  m.def("gemm_bf16_sums", &gemm_bf16_sums,
        "x @ w^T, stretches of the inner dimension apart", py::arg("x"),
        py::arg("w"), py::arg("tile"), py::arg("stretches") = 0);
  m.def("gemm_bf16_plan", &gemm_bf16_plan,
        "Tile, stretches and us of gemm_bf16, or of its sums, as estimated",
        py::arg("M"), py::arg("N"), py::arg("K"), py::arg("gelu"),
        py::arg("sums"), py::arg("cus") = 256, py::arg("below") = 1e30);
  m.def("gemm_bf16_cut", &gemm_bf16_cut,
        "Whether gemm_bf16 cuts a product by rows, behind how many rows or "
        "columns (0: not at all), tiles of both parts, us", py::arg("M"),
        py::arg("N"), py::arg("K"), py::arg("gelu"), py::arg("cus") = 256);
  m.def("gemm_bf16_glu_cut", &gemm_bf16_glu_cut,
        "gemm_bf16_cut of gemm_bf16_glu", py::arg("M"), py::arg("N"),
        py::arg("K"), py::arg("cus") = 256);
  m.def("gemm_bf16_glu_plan", &gemm_bf16_glu_plan,
        "What gemm_bf16_glu does with a product of w [2 N, K], as estimated: "
        "its tile, or tile and stretches of sums", py::arg("M"), py::arg("N"),
        py::arg("K"), py::arg("cus") = 256);
  m.def("gemm_ring_places", &gemm_ring_places,
        "Where a workgroup of gemm_bf16 loads along the inner dimension",
        py::arg("k"), py::arg("steps"), py::arg("turn") = 0);
  m.def("gemm_bf16_glu", &gemm_bf16_glu,
        "silu(x @ w[:N]^T) * (x @ w[N:]^T) of more than a few rows",
        py::arg("out"), py::arg("x"), py::arg("w"), py::arg("tile") = 0);
  m.def("gemm_skinny_bf16", &gemm_skinny_bf16,
        "Skinny-M decode GEMM: split-K + XCD-chunked tile swizzle");
  m.def("gemm_rows", &gemm_rows, "x @ w^T (+bias, GELU) of at most 128 rows",
        py::arg("out"), py::arg("x"), py::arg("w"), py::arg("bias"),
        py::arg("x_scale"), py::arg("w_scale"), py::arg("gelu") = false);
  m.def("gemm_rows_sums", &gemm_rows_sums,
        "x @ w^T of at most 128 rows, stretches of the inner dimension apart");
  m.def("gemm_rows_many", &gemm_rows_many,
        "x @ w^T + bias of at most 64 rows for several w, in one launch");
  m.def("gemm_rows_glu", &gemm_rows_glu,
        "silu(x @ gate^T) * (x @ up^T) of at most 64 rows");
  m.def("layer_rows_join", &layer_rows_join,
        "residual += x @ w^T of at most 16 rows, (rows times norm, squares)");
  m.def("layer_rows_glu", &layer_rows_glu,
        "silu(x @ gate^T f) * (x @ up^T f) of at most 16 rows, f by squares");
  m.def("layer_rows_qkv", &layer_rows_qkv,
        "Heads of x @ w^T f + bias of at most 32 rows, turned and cached");
  m.def("quantize_rows", &quantize_rows,
        "bf16 rows to e4m3 bytes with a scale each");
  m.def("gemm_fp8", &gemm_fp8,
        "MX-fp8 e4m3 MFMA GEMM with epilogue per-row/col dequant");
  m.def("mfma_probe", &mfma_probe, "16x16x32 MFMA layout probe");
  m.def("ar_create", &ar_create,
        "Allocate one-shot allreduce mailbox; returns IPC handle bytes");
  m.def("ar_open", &ar_open, "Map peer mailboxes from IPC handles");
  m.def("ar_capacity", &ar_capacity, "Opened AR data capacity in bytes");
  m.def("ar_allreduce", &ar_allreduce,
        "One-shot bf16 allreduce over xGMI peer mailboxes");
  m.def("ar_destroy", &ar_destroy, "Tear down the allreduce context");
  m.def("mfma_probe_fp8", &mfma_probe_fp8,
        "16x16x128 MX-fp8 MFMA layout probe (unity e8m0 scales)");
}
