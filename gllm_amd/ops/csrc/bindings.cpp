// Python bindings for the gfx950 kernel extension.
#include <torch/extension.h>

void rmsnorm(torch::Tensor out, torch::Tensor in, torch::Tensor weight,
             double eps);
void fused_add_rmsnorm(torch::Tensor x, torch::Tensor residual,
                       torch::Tensor weight, double eps);
void silu_and_mul(torch::Tensor out, torch::Tensor x);
void gelu_and_mul(torch::Tensor out, torch::Tensor x);
void rotary_embedding(torch::Tensor positions, torch::Tensor q,
                      torch::Tensor k, long head_dim,
                      torch::Tensor cos_sin_cache, bool is_neox);
void reshape_and_cache(torch::Tensor k, torch::Tensor v,
                       torch::Tensor k_cache, torch::Tensor v_cache,
                       torch::Tensor slot_mapping);
void paged_attention_decode(torch::Tensor out, torch::Tensor q,
                            torch::Tensor k_cache, torch::Tensor v_cache,
                            torch::Tensor block_table, torch::Tensor seq_lens,
                            double scale, long sliding_window,
                            c10::optional<torch::Tensor> query_start_loc);
bool decode_rows_ok(torch::Tensor k_cache, torch::Tensor v_cache, long Hq);
torch::Tensor resolve_tokens(torch::Tensor tokens, torch::Tensor ring);
torch::Tensor qkv_norm_finish(torch::Tensor src, torch::Tensor q_w,
                              torch::Tensor k_w, double eps,
                              torch::Tensor positions, torch::Tensor cos_sin,
                              torch::Tensor k_cache, torch::Tensor v_cache,
                              torch::Tensor slots, long Hq);
long stream_slice(long M, long N, long K);
torch::Tensor stream_gemm(torch::Tensor x, torch::Tensor w,
                          c10::optional<torch::Tensor> bias);
torch::Tensor stream_gemm_gated(torch::Tensor x, torch::Tensor w);
torch::Tensor tile_gemm(torch::Tensor x, torch::Tensor w,
                        c10::optional<torch::Tensor> bias, bool gated);
double tile_gemm_cost(long M, long N, long K, bool gated);
torch::Tensor stream_parts(torch::Tensor x, torch::Tensor w);
torch::Tensor stream_add_norm(torch::Tensor x, torch::Tensor w,
                              torch::Tensor residual, torch::Tensor norm_w,
                              double eps);
bool qkv_decode_ok(torch::Tensor k_cache, long Hq, long B, bool rounded);
torch::Tensor qkv_decode(torch::Tensor parts,
                         c10::optional<torch::Tensor> bias,
                         torch::Tensor positions, torch::Tensor cos_sin,
                         torch::Tensor k_cache, torch::Tensor v_cache,
                         torch::Tensor slots, torch::Tensor block_table,
                         torch::Tensor seq_lens, torch::Tensor arrived,
                         long Hq, double scale, long sliding_window,
                         bool rounded);
torch::Tensor qkv_finish(torch::Tensor src, c10::optional<torch::Tensor> bias,
                         torch::Tensor positions, torch::Tensor cos_sin,
                         torch::Tensor k_cache, torch::Tensor v_cache,
                         torch::Tensor slots, long Hq, bool rounded);
void paged_attention_prefill(torch::Tensor out, torch::Tensor q,
                             torch::Tensor k_cache, torch::Tensor v_cache,
                             torch::Tensor block_table,
                             torch::Tensor seq_lens,
                             torch::Tensor query_start_loc,
                             long max_query_len, double scale,
                             long sliding_window, bool skip_single);
void window_attention_mfma(torch::Tensor out, torch::Tensor q,
                           c10::optional<torch::Tensor> gate,
                           torch::Tensor k_cache, torch::Tensor v_cache,
                           torch::Tensor block_table, torch::Tensor seq_lens,
                           torch::Tensor query_start_loc, long max_query_len,
                           double scale, long window, long keep_first,
                           bool sink, c10::optional<torch::Tensor> sinks,
                           double softcap,
                           c10::optional<torch::Tensor> bias,
                           double temp_coef, long temp_every);
bool window_attention_decode(torch::Tensor out, torch::Tensor q,
                             c10::optional<torch::Tensor> gate,
                             torch::Tensor k_cache, torch::Tensor v_cache,
                             torch::Tensor block_table,
                             torch::Tensor seq_lens, double scale,
                             long window, long keep_first, bool sink,
                             c10::optional<torch::Tensor> sinks,
                             double softcap,
                             c10::optional<torch::Tensor> bias,
                             double temp_coef, long temp_every);
void mla_paged_attention(torch::Tensor out, torch::Tensor q,
                         torch::Tensor k_cache, torch::Tensor block_table,
                         torch::Tensor seq_lens,
                         torch::Tensor query_start_loc, long max_query_len,
                         double scale);
torch::Tensor mla_queries(torch::Tensor q, torch::Tensor kv,
                          torch::Tensor norm_w, double eps,
                          torch::Tensor positions, torch::Tensor cos_sin,
                          torch::Tensor w_kvb, torch::Tensor k_cache,
                          torch::Tensor slots);
torch::Tensor mla_values(torch::Tensor o_lat, torch::Tensor w_kvb);
std::vector<torch::Tensor> mla_prompt_rows(
    torch::Tensor q, torch::Tensor kv, torch::Tensor norm_w, double eps,
    torch::Tensor positions, torch::Tensor cos_sin, torch::Tensor k_cache,
    torch::Tensor slots);
void mla_prompts(torch::Tensor out, torch::Tensor q, torch::Tensor kv,
                 torch::Tensor pe, torch::Tensor query_start_loc,
                 long max_query_len, double scale);
void cache_latent(torch::Tensor k, torch::Tensor k_cache,
                  torch::Tensor slot_mapping);
void moe_align(torch::Tensor topk_ids, long E_local, long expert_start,
               long block_m, torch::Tensor sorted_ids,
               torch::Tensor expert_blocks, torch::Tensor n_post_pad);
void moe_gemm(torch::Tensor C, torch::Tensor A, torch::Tensor W,
              torch::Tensor sorted_ids, torch::Tensor expert_blocks,
              torch::Tensor n_post_pad,
              c10::optional<torch::Tensor> topk_weights, long n_pairs,
              long topk, long block_m, bool scatter);
torch::Tensor moe_gemm_tiled_shared(
    torch::Tensor C, torch::Tensor A, torch::Tensor W,
    torch::Tensor sorted_ids, torch::Tensor expert_blocks,
    torch::Tensor n_post_pad, c10::optional<torch::Tensor> topk_weights,
    long n_pairs, long topk, long block_m, long act, torch::Tensor rows,
    torch::Tensor w);
void moe_gemm_tiled(torch::Tensor C, torch::Tensor A, torch::Tensor W,
                    torch::Tensor sorted_ids, torch::Tensor expert_blocks,
                    torch::Tensor n_post_pad,
                    c10::optional<torch::Tensor> topk_weights, long n_pairs,
                    long topk, long block_m, long act, double limit,
                    double alpha);
torch::Tensor moe_sum_norm(torch::Tensor pair_out, torch::Tensor ids,
                           long expert_start, long E_local, long topk,
                           c10::optional<torch::Tensor> shared,
                           torch::Tensor residual, torch::Tensor norm_w,
                           double eps);
void moe_sum(torch::Tensor out, torch::Tensor pair_out, torch::Tensor ids,
             long expert_start, long E_local, long topk);
void softmax_topk_rows(torch::Tensor weights, torch::Tensor ids,
                       torch::Tensor logits, bool renorm);
void per_token_group_quant_fp8(torch::Tensor x, torch::Tensor q,
                               torch::Tensor scales,
                               c10::optional<torch::Tensor> scales_t,
                               bool ue8m0);
void moe_gemm_fp8(torch::Tensor C, torch::Tensor A, torch::Tensor As,
                  torch::Tensor W, torch::Tensor Ws,
                  torch::Tensor sorted_ids, torch::Tensor expert_blocks,
                  torch::Tensor n_post_pad,
                  c10::optional<torch::Tensor> topk_weights, long n_pairs,
                  long topk, long block_m, bool scatter);
torch::Tensor quant_gemm(torch::Tensor x, c10::optional<torch::Tensor> xs,
                         torch::Tensor w, torch::Tensor ws,
                         c10::optional<torch::Tensor> bias, long form,
                         long splits);
std::vector<torch::Tensor> quant_gemm_gated_fp8(torch::Tensor x,
                                                torch::Tensor xs,
                                                torch::Tensor w,
                                                torch::Tensor ws);
std::vector<torch::Tensor> parts_add_norm_fp8(torch::Tensor part,
                                              torch::Tensor residual,
                                              torch::Tensor norm_w,
                                              double eps, bool rounded);
std::vector<torch::Tensor> qkv_decode_fp8(
    torch::Tensor parts, c10::optional<torch::Tensor> bias,
    torch::Tensor positions, torch::Tensor cos_sin, torch::Tensor k_cache,
    torch::Tensor v_cache, torch::Tensor slots, torch::Tensor block_table,
    torch::Tensor seq_lens, torch::Tensor arrived, long Hq, double scale,
    long sliding_window, bool rounded);
torch::Tensor parts_add_norm(torch::Tensor part, torch::Tensor residual,
                             torch::Tensor norm_w, double eps,
                             bool rounded);
void moe_gemm_int4(torch::Tensor C, torch::Tensor A, torch::Tensor W,
                   torch::Tensor SB, torch::Tensor sorted_ids,
                   torch::Tensor expert_blocks, torch::Tensor n_post_pad,
                   c10::optional<torch::Tensor> topk_weights, long n_pairs,
                   long topk, long block_m, bool scatter);
void gdn_conv_update(torch::Tensor out, torch::Tensor x,
                     torch::Tensor weight, torch::Tensor conv_state,
                     torch::Tensor slots);
void gdn_chunk_prefill(torch::Tensor o, torch::Tensor q, torch::Tensor k,
                       torch::Tensor v, torch::Tensor g, torch::Tensor beta,
                       torch::Tensor states, double scale);
void gdn_reserve(torch::Tensor like, long T, long B, long Hv);
torch::Tensor gdn_varlen(torch::Tensor conv, torch::Tensor ba,
                         torch::Tensor A_log, torch::Tensor dt_bias,
                         torch::Tensor states, torch::Tensor slots,
                         torch::Tensor has_init, torch::Tensor qsl, long Hk,
                         long max_len, double scale);
torch::Tensor gdn_step(torch::Tensor conv, torch::Tensor ba,
                       torch::Tensor A_log, torch::Tensor dt_bias,
                       torch::Tensor states, torch::Tensor slots, long Hk,
                       double scale);
torch::Tensor gdn_gate(torch::Tensor o, torch::Tensor z, torch::Tensor w,
                       double eps);
void gdn_decode(torch::Tensor o, torch::Tensor qn, torch::Tensor kn,
                torch::Tensor v, torch::Tensor g, torch::Tensor beta,
                torch::Tensor state, torch::Tensor slots);
void rmsnorm_gated(torch::Tensor out, torch::Tensor x, torch::Tensor z,
                   torch::Tensor w, double eps);
void apply_repetition_penalty(torch::Tensor logits, torch::Tensor pool,
                              torch::Tensor slots,
                              torch::Tensor penalties);
torch::Tensor greedy_argmax(torch::Tensor logits);
void topk_topp_filter(torch::Tensor probs, torch::Tensor top_ks,
                      torch::Tensor top_ps,
                      c10::optional<torch::Tensor> min_ps);
std::pair<int64_t, py::bytes> car_alloc(int64_t data_bytes);
std::pair<int64_t, py::bytes> car_alloc_v2(int64_t max_bytes);
void car_all_reduce_v2(torch::Tensor inout, std::vector<int64_t> ptrs,
                       int64_t rank, int64_t world, int64_t max_bytes);
int64_t car_open(py::bytes handle_bytes);
void car_close(int64_t ptr);
void car_free(int64_t ptr);
torch::Tensor car_view_tensor(int64_t ptr, int64_t numel);
void car_all_reduce(torch::Tensor inout, std::vector<int64_t> ptrs,
                    int64_t rank, int64_t world, int64_t epoch);

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("rmsnorm", &rmsnorm, "RMSNorm (gfx950)");
  m.def("fused_add_rmsnorm", &fused_add_rmsnorm,
        "residual += x; x = rmsnorm(residual)");
  m.def("silu_and_mul", &silu_and_mul, "silu(x[:d]) * x[d:]");
  m.def("gelu_and_mul", &gelu_and_mul, "gelu(x[:d]) * x[d:]");
  m.def("rotary_embedding", &rotary_embedding, "in-place RoPE on q,k");
  m.def("reshape_and_cache", &reshape_and_cache,
        "scatter K/V into paged cache");
  m.def("paged_attention_decode", &paged_attention_decode,
        "split-KV paged decode attention");
  m.def("decode_rows_ok", &decode_rows_ok,
        "the decode kernel takes these heads");
  m.def("paged_attention_prefill", &paged_attention_prefill,
        "varlen MFMA paged prefill attention");
  m.def("window_attention_mfma", &window_attention_mfma,
        "prefill MFMA kernel with window + kept first tokens + sink + gate");
  m.def("window_attention_decode", &window_attention_decode,
        "split-KV decode kernels with window + kept first + sink + gate; "
        "false = geometry not instantiated");
  m.def("resolve_tokens", &resolve_tokens,
        "token ids with places in the ring of sampled tokens");
  m.def("stream_slice", &stream_slice,
        "columns of K of one sum of stream_gemm's");
  m.def("stream_gemm", &stream_gemm, "x w^T + bias for at most 256 rows");
  m.def("tile_gemm", &tile_gemm, "x w^T + bias, or its gated form");
  m.def("tile_gemm_cost", &tile_gemm_cost,
        "cost of a tile_gemm in steps of one tile");
  m.def("stream_gemm_gated", &stream_gemm_gated,
        "silu(x w_gate^T) * (x w_up^T) for at most 256 rows");
  m.def("stream_parts", &stream_parts, "fp32 parts of x w^T");
  m.def("stream_add_norm", &stream_add_norm,
        "residual += x w^T; RMS norm of it");
  m.def("qkv_decode_ok", &qkv_decode_ok);
  m.def("qkv_decode", &qkv_decode,
        "bias, rotation, cache and decode attention of projection parts");
  m.def("qkv_norm_finish", &qkv_norm_finish,
        "qkv_finish of bf16 rows with a norm per head");
  m.def("qkv_finish", &qkv_finish,
        "bias, rotation, keys and values to the cache; queries");
  m.def("mla_paged_attention", &mla_paged_attention,
        "absorbed-MLA varlen attention over the 576-dim latent cache");
  m.def("mla_queries", &mla_queries,
        "latent cache rows and absorbed, rotated query rows");
  m.def("mla_prompt_rows", &mla_prompt_rows,
        "normed and rotated latent rows of prompts, queries in place");
  m.def("mla_prompts", &mla_prompts, "per-head attention of whole prompts");
  m.def("mla_values", &mla_values, "per-head values of the weighted latent");
  m.def("cache_latent", &cache_latent,
        "scatter the per-token latent row into the paged cache");
  m.def("moe_align", &moe_align,
        "device-side moe_align_block_size (graph-safe)");
  m.def("moe_gemm", &moe_gemm,
        "grouped MFMA GEMM over sorted (token, expert) pairs");
  m.def("moe_gemm_tiled_shared", &moe_gemm_tiled_shared,
        "moe_gemm_tiled with a shared expert's product beside it");
  m.def("moe_gemm_tiled", &moe_gemm_tiled,
        "grouped MFMA GEMM of wide tiles, activation in the epilogue");
  m.def("softmax_topk_rows", &softmax_topk_rows,
        "softmax over all experts, then top-k");
  m.def("moe_sum_norm", &moe_sum_norm,
        "pair outputs over topk (+ shared), residual and RMS norm");
  m.def("moe_sum", &moe_sum, "sum pair outputs over topk");
  m.def("per_token_group_quant_fp8", &per_token_group_quant_fp8,
        "per (token, 128-group) e4m3 quant + fp32 scales");
  m.def("moe_gemm_fp8", &moe_gemm_fp8,
        "block-scale fp8 grouped MoE GEMM");
  m.def("quant_gemm", &quant_gemm,
        "few-row product with int4 or block-scale fp8 weights");
  m.def("quant_gemm_gated_fp8", &quant_gemm_gated_fp8,
        "gated fp8 product with its e4m3 rows");
  m.def("parts_add_norm_fp8", &parts_add_norm_fp8,
        "parts_add_norm with its e4m3 rows");
  m.def("qkv_decode_fp8", &qkv_decode_fp8,
        "qkv_decode with its e4m3 rows");
  m.def("parts_add_norm", &parts_add_norm,
        "residual += sum of fp32 parts, RMS norm of it");
  m.def("moe_gemm_int4", &moe_gemm_int4,
        "fused-dequant int4 grouped MoE GEMM (w4a16)");
  m.def("gdn_conv_update", &gdn_conv_update,
        "batched causal-conv1d decode step w/ state roll");
  m.def("gdn_chunk_prefill", &gdn_chunk_prefill,
        "fused WY chunk-parallel gated delta rule prefill");
  m.def("gdn_reserve", &gdn_reserve,
        "takes and gives back the memory of a gdn_varlen call");
  m.def("gdn_varlen", &gdn_varlen,
        "ragged chunk-parallel gated delta rule");
  m.def("gdn_step", &gdn_step,
        "one token per sequence from the convolved projection");
  m.def("gdn_gate", &gdn_gate, "rmsnorm(o) * w * silu(z) per head");
  m.def("gdn_decode", &gdn_decode,
        "batched fused recurrent gated-delta-rule decode step");
  m.def("rmsnorm_gated", &rmsnorm_gated, "rmsnorm(x)*w*silu(z)");
  m.def("apply_repetition_penalty", &apply_repetition_penalty,
        "scaling penalty vs persistent seen-token mask pool");
  m.def("greedy_argmax", &greedy_argmax, "first largest value of each row");
  m.def("topk_topp_filter", &topk_topp_filter,
        "fused sorting-free top-k/top-p/min-p filter + renormalize");
  m.def("car_alloc", &car_alloc, "alloc hipIpc-shared AR buffer");
  m.def("car_alloc_v2", &car_alloc_v2,
        "alloc v2 AR buffer (device epoch + out slices)");
  m.def("car_all_reduce_v2", &car_all_reduce_v2,
        "two-shot/one-shot xGMI AR, device-epoch (graph-capturable)");
  m.def("car_open", &car_open, "map a peer's AR buffer");
  m.def("car_close", &car_close);
  m.def("car_free", &car_free);
  m.def("car_view_tensor", &car_view_tensor,
        "non-owning bf16 view over raw device memory");
  m.def("car_all_reduce", &car_all_reduce,
        "one-shot xGMI custom all-reduce (epoch advances by 2/call)");
}
