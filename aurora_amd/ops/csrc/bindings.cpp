// Python bindings of the decoder kernels (gfx950).
#include <torch/extension.h>

torch::Tensor rmsnorm(torch::Tensor x, torch::Tensor weight, double eps);
std::vector<torch::Tensor> rmsnorm_residual(torch::Tensor x, torch::Tensor res,
                                            torch::Tensor weight, double eps);
torch::Tensor silu_mul(torch::Tensor gu);
void rope_apply_(torch::Tensor q, torch::Tensor k, torch::Tensor positions,
                 torch::Tensor cos_sin);
void kv_cache_write(torch::Tensor k, torch::Tensor v, torch::Tensor kc,
                    torch::Tensor vc, torch::Tensor slots);
torch::Tensor paged_attention_decode(torch::Tensor q, torch::Tensor kc,
                                     torch::Tensor vc, torch::Tensor bt,
                                     torch::Tensor ctx, double scale,
                                     c10::optional<torch::Tensor> into,
                                     c10::optional<torch::Tensor> marks);
long decode_marks(long B, long Hq, long Hkv, long longest, long window, long chunk);
torch::Tensor attention_prefill_paged(torch::Tensor q, torch::Tensor kc,
                                      torch::Tensor vc, torch::Tensor bt,
                                      torch::Tensor cu_q, torch::Tensor ctx,
                                      double scale, c10::optional<torch::Tensor> into);
torch::Tensor skinny_gemm(torch::Tensor x, torch::Tensor w);
torch::Tensor fused_rope_kv_write(torch::Tensor qkv, torch::Tensor positions,
                                  torch::Tensor slots, torch::Tensor cos_sin,
                                  torch::Tensor kc, torch::Tensor vc,
                                  long Hq, long Hkv,
                                  c10::optional<torch::Tensor> bias);
c10::optional<torch::Tensor> own_product(const torch::Tensor& x, const torch::Tensor& w,
                                         long form);
torch::Tensor many_rows(torch::Tensor x, torch::Tensor w, bool silu);
torch::Tensor few_rows(torch::Tensor x, torch::Tensor w, bool raw, long parts, long width,
                       long rows);
torch::Tensor linear_few_rows(torch::Tensor x, torch::Tensor w, bool raw, bool steady);
torch::Tensor silu_few_rows(torch::Tensor x, torch::Tensor w);
torch::Tensor one_row_product(torch::Tensor x, torch::Tensor res, torch::Tensor weight, double eps,
                              torch::Tensor res_out, torch::Tensor w, bool silu, bool steady);
bool norms_row(const torch::Tensor& x, const torch::Tensor& res, const torch::Tensor& weight,
               const torch::Tensor& w, bool silu, bool steady);
torch::Tensor skinny_gemm2_ex(torch::Tensor x, torch::Tensor w, long s_target);
torch::Tensor skinny_gemm3_ex(torch::Tensor x, torch::Tensor w, long s_target);
torch::Tensor moe_grouped_gemm(torch::Tensor xp, torch::Tensor w,
                               torch::Tensor starts, torch::Tensor counts);
// ---- layer-listed decoders
using OptT = c10::optional<torch::Tensor>;
std::vector<torch::Tensor> residual_rmsnorm(torch::Tensor x, torch::Tensor weight, OptT delta,
                                            OptT gate_pre, OptT gate_bias, OptT y, OptT place,
                                            OptT gate, OptT post, OptT step, OptT conv_w, OptT ring,
                                            OptT pos, OptT slots, double eps, double offset,
                                            bool to_bf16);
void embed_pairs(torch::Tensor ids, torch::Tensor table, double scale, torch::Tensor pairs,
                 long mul_prev, long mul_cur, torch::Tensor weight, double eps,
                 torch::Tensor prev, OptT cu, torch::Tensor starts, torch::Tensor slots,
                 torch::Tensor out);
long short_conv_rows();
void short_conv_add(torch::Tensor h, torch::Tensor w, torch::Tensor ring, OptT cu, OptT bseq,
                    OptT boff, torch::Tensor starts, torch::Tensor slots, torch::Tensor out);
torch::Tensor xielu(torch::Tensor z, torch::Tensor act);
void latent_front(torch::Tensor proj, long c0, long rank, OptT weight, double eps, long k0,
                  long key_at, OptT cos_sin, OptT pos, torch::Tensor slots,
                  torch::Tensor cache, long q0, OptT q_weight, OptT cq);
torch::Tensor gather_latents(torch::Tensor cache, torch::Tensor rows);
std::vector<torch::Tensor> latent_places(torch::Tensor block_tables, torch::Tensor cu,
                                         torch::Tensor ctx, long page, long window, long longest,
                                         long total);
void rotate_heads(torch::Tensor x, torch::Tensor pos, torch::Tensor cos_sin,
                  torch::Tensor out);
void head_linear(torch::Tensor x, torch::Tensor w, OptT gate, torch::Tensor out, OptT turn_x,
                 OptT turn_pos, OptT turn_cs, OptT turn_out);
torch::Tensor latent_attention(torch::Tensor q, torch::Tensor cache, torch::Tensor bt, OptT cu,
                               torch::Tensor ctx, OptT bseq, OptT boff, long rows,
                               double scale, OptT sink, long VR, long window);
void latent_attention_rows(torch::Tensor q, torch::Tensor cache, torch::Tensor bt, OptT cu,
                           torch::Tensor ctx, OptT row_seq, OptT row_off, double scale,
                           OptT sink, long window, torch::Tensor out);
void tailed_attention_prefill(torch::Tensor q, torch::Tensor kc, torch::Tensor vc,
                              torch::Tensor tail, torch::Tensor bt, torch::Tensor cu_q,
                              torch::Tensor ctx, torch::Tensor bseq, torch::Tensor boff,
                              double scale, long window, torch::Tensor out);
long conv_qkv_rows();
void conv_qkv(torch::Tensor proj, long q0, long k0, long v0, torch::Tensor w,
              torch::Tensor turn, OptT value_turn, torch::Tensor ring, torch::Tensor kv_slots,
              OptT cu, OptT bseq, OptT boff, torch::Tensor starts, torch::Tensor slots,
              torch::Tensor kc, torch::Tensor vc, torch::Tensor q, long d, long dv);
void sink_attention_prefill(torch::Tensor q, torch::Tensor kc, torch::Tensor vc,
                            torch::Tensor bt, torch::Tensor cu_q, torch::Tensor ctx,
                            torch::Tensor bseq, torch::Tensor boff, double scale,
                            torch::Tensor sink, torch::Tensor gate, torch::Tensor out);
torch::Tensor bias_kv_write(torch::Tensor proj, long q0, long k0, long v0,
                            torch::Tensor bias, torch::Tensor slots, torch::Tensor kc,
                            torch::Tensor vc, long Hq, long Hkv, long d, long dv);
long biased_prefill_rows(long G);
void biased_attention_prefill(torch::Tensor q, torch::Tensor kc, torch::Tensor vc,
                              torch::Tensor bt, torch::Tensor cu_q, torch::Tensor ctx,
                              torch::Tensor bseq, torch::Tensor boff, double scale,
                              long window, long chunk, OptT slopes, OptT rates, OptT sink,
                              OptT turn, OptT gate, torch::Tensor out, long col, long dv,
                              double oscale);
c10::optional<torch::Tensor> fresh_attention_decode(
    torch::Tensor qkv, c10::optional<torch::Tensor> bias, torch::Tensor cos_sin, torch::Tensor kc,
    torch::Tensor vc, torch::Tensor bt, torch::Tensor ctx, long Hq, double scale,
    c10::optional<torch::Tensor> marks);
void biased_attention_decode(torch::Tensor q, torch::Tensor kc, torch::Tensor vc,
                             torch::Tensor bt, torch::Tensor ctx, double scale, long window,
                             long chunk, OptT slopes, OptT rates, OptT sink, OptT turn,
                             OptT gate, torch::Tensor out, long col, long dv, double oscale,
                             OptT marks);
void biased_attention_rows(torch::Tensor q, torch::Tensor kc, torch::Tensor vc,
                           torch::Tensor bt, OptT cu, torch::Tensor ctx, OptT row_seq,
                           OptT row_off, double scale, long window, long chunk, OptT slopes,
                           OptT rates, OptT sink, OptT turn, OptT gate, torch::Tensor out,
                           long col, long dv, double oscale);
void delta_prefill(torch::Tensor proj, torch::Tensor z, torch::Tensor conv_w,
                   torch::Tensor a_log, torch::Tensor dt_bias, torch::Tensor norm, long H,
                   long G, long d, long e, long taps, long q0, long k0, long v0, long b0,
                   double eps, torch::Tensor state, torch::Tensor ring, torch::Tensor cu,
                   torch::Tensor cseq, torch::Tensor coff, torch::Tensor cfirst,
                   torch::Tensor starts, torch::Tensor slots, torch::Tensor out, long col,
                   double oscale);
void delta_decode(torch::Tensor proj, torch::Tensor z, torch::Tensor conv_w,
                  torch::Tensor a_log, torch::Tensor dt_bias, torch::Tensor norm, long H,
                  long G, long d, long e, long taps, long q0, long k0, long v0, long b0,
                  double eps, torch::Tensor state, torch::Tensor ring, torch::Tensor starts,
                  torch::Tensor slots, torch::Tensor out, long col, double oscale);
void retention_prefill(torch::Tensor proj, torch::Tensor decay, torch::Tensor cos_sin,
                       long H, long d, long e, long rot, long q0, long k0, long v0, long g0,
                       double eps, torch::Tensor state, torch::Tensor cu, torch::Tensor cseq,
                       torch::Tensor coff, torch::Tensor cfirst, torch::Tensor starts,
                       torch::Tensor slots, torch::Tensor out);
void retention_decode(torch::Tensor proj, torch::Tensor decay, torch::Tensor cos_sin, long H,
                      long d, long e, long rot, long q0, long k0, long v0, long g0,
                      double eps, torch::Tensor state, torch::Tensor starts,
                      torch::Tensor slots, torch::Tensor out);
std::vector<torch::Tensor> moe_route(torch::Tensor h, torch::Tensor router,
                                     c10::optional<torch::Tensor> bias, long top);
torch::Tensor moe_combine(torch::Tensor y, torch::Tensor place, torch::Tensor gate);
std::vector<torch::Tensor> moe_silu_glu(torch::Tensor h, torch::Tensor sel, torch::Tensor w_gu,
                                        torch::Tensor w_dn);
std::vector<torch::Tensor> moe_clamped_glu(torch::Tensor h, torch::Tensor sel,
                                           torch::Tensor w_gu, torch::Tensor w_dn,
                                           double limit, double alpha, double shift);
std::vector<torch::Tensor> moe_route_grouped(torch::Tensor h, torch::Tensor router,
                                             OptT correction, long top, long groups,
                                             long keep, double scale);
std::vector<torch::Tensor> moe_relu2(torch::Tensor h, torch::Tensor sel, torch::Tensor w_up,
                                     torch::Tensor w_dn);
torch::Tensor gelu(torch::Tensor z);
torch::Tensor relu2(torch::Tensor z);
torch::Tensor silu_glu(torch::Tensor z, long F);
torch::Tensor output_norm(torch::Tensor src, torch::Tensor x, torch::Tensor weight,
                          torch::Tensor bias, OptT delta, OptT gate, OptT y, OptT place,
                          OptT share, OptT kept, OptT coefs, OptT fw, OptT fb, double eps,
                          bool to_bf16);
torch::Tensor normed_qkv(torch::Tensor proj, long q0, long k0, long v0, torch::Tensor qw,
                         torch::Tensor kw, bool whole, double eps, OptT cos_sin, double coef,
                         long every, torch::Tensor pos, torch::Tensor slots, torch::Tensor kc,
                         torch::Tensor vc, long Hq, long Hkv, long d, long dv);
void head_delta_prefill(torch::Tensor proj, torch::Tensor conv_w, torch::Tensor a_log,
                        torch::Tensor dt_bias, torch::Tensor norm, long H, long G, long d,
                        long e, long taps, long q0, long k0, long v0, long b0, long a0,
                        long g0, double eps, torch::Tensor state, torch::Tensor ring,
                        torch::Tensor cu, torch::Tensor cseq, torch::Tensor coff,
                        torch::Tensor cfirst, torch::Tensor starts, torch::Tensor slots,
                        torch::Tensor out, long col, double oscale);
void head_delta_decode(torch::Tensor proj, torch::Tensor conv_w, torch::Tensor a_log,
                       torch::Tensor dt_bias, torch::Tensor norm, long H, long G, long d,
                       long e, long taps, long q0, long k0, long v0, long b0, long a0,
                       long g0, double eps, torch::Tensor state, torch::Tensor ring,
                       torch::Tensor starts, torch::Tensor slots, torch::Tensor out,
                       long col, double oscale);
void memory_prefill(torch::Tensor proj, torch::Tensor i_bias, torch::Tensor f_bias,
                    torch::Tensor norm, long H, long d, long e, long q0, long k0, long v0,
                    long i0, long f0, long g0, double cap, double eps, torch::Tensor state,
                    torch::Tensor nstate, torch::Tensor mstate, torch::Tensor cu,
                    torch::Tensor cseq, torch::Tensor coff, torch::Tensor cfirst,
                    torch::Tensor starts, torch::Tensor slots, torch::Tensor out, long col,
                    double oscale);
void memory_decode(torch::Tensor proj, torch::Tensor i_bias, torch::Tensor f_bias,
                   torch::Tensor norm, long H, long d, long e, long q0, long k0, long v0,
                   long i0, long f0, long g0, double cap, double eps, torch::Tensor state,
                   torch::Tensor nstate, torch::Tensor mstate, torch::Tensor starts,
                   torch::Tensor slots, torch::Tensor out, long col, double oscale);

py::object pack_batch(py::list ids, std::vector<long> first, std::vector<long> end,
                      py::list pages, std::vector<long> states, long prompts, long page,
                      torch::Device device);
py::object pack_texts(py::list texts, long most, torch::Device device);
py::object pack_rows(py::list rows, torch::Device device);
bool stage_decode(py::list seqs, torch::Tensor ids, torch::Tensor host, torch::Tensor keys,
                  torch::Tensor inputs, long width, long page, long scratch_page,
                  long scratch_slot);

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("rmsnorm", &rmsnorm, "fused RMSNorm (bf16, gfx950)");
  m.def("rmsnorm_residual", &rmsnorm_residual, "fused residual-add + RMSNorm");
  m.def("silu_mul", &silu_mul, "fused SiLU(gate)*up");
  m.def("rope_apply_", &rope_apply_, "in-place RoPE on q/k");
  m.def("kv_cache_write", &kv_cache_write, "scatter K/V into paged cache");
  m.def("paged_attention_decode", &paged_attention_decode, "paged GQA decode attention",
        py::arg("q"), py::arg("kc"), py::arg("vc"), py::arg("bt"), py::arg("ctx"),
        py::arg("scale"), py::arg("into") = py::none(), py::arg("marks") = py::none());
  m.def("decode_marks", &decode_marks,
        "zeros that decode attention wants to merge stretches of contexts, 0 for none");
  m.def("attention_prefill_paged", &attention_prefill_paged,
        "MFMA flash prefill over paged KV");
  m.def("skinny_gemm", &skinny_gemm, "decode-path skinny GEMM (M<=64)");
  m.def("fused_rope_kv_write", &fused_rope_kv_write,
        "fused qkv split + RoPE + paged KV scatter");
  m.def("own_product", &own_product, "a product by the own kernels where they win");
  m.def("many_rows", &many_rows, "products of many rows, with silu(gate) * up");
  m.def("few_rows", &few_rows, "products of at most 128 rows, K in parts", py::arg("x"),
        py::arg("w"), py::arg("raw"), py::arg("parts"), py::arg("width") = 64,
        py::arg("rows") = 0);
  m.def("linear_few_rows", &linear_few_rows, "linear of at most 128 rows", py::arg("x"),
        py::arg("w"), py::arg("raw"), py::arg("steady") = false);
  m.def("one_row_product", &one_row_product, "a norm and the product of its one row",
        py::arg("x"), py::arg("res"), py::arg("weight"), py::arg("eps"), py::arg("res_out"),
        py::arg("w"), py::arg("silu"), py::arg("steady") = false);
  m.def("norms_row", &norms_row, "whether one_row_product serves", py::arg("x"), py::arg("res"),
        py::arg("weight"), py::arg("w"), py::arg("silu"), py::arg("steady") = false);
  m.def("silu_few_rows", &silu_few_rows, "gate and up of at most 128 rows, silu(gate) * up");
  m.def("skinny_gemm2_ex", &skinny_gemm2_ex, "products of at most 256 rows");
  m.def("skinny_gemm3_ex", &skinny_gemm3_ex, "glds double-buffered projection GEMM (M<=256)");
  m.def("moe_grouped_gemm", &moe_grouped_gemm,
        "packed per-expert grouped GEMM (skips unrouted experts)");
  m.def("residual_rmsnorm", &residual_rmsnorm,
        "fp32 residual add (dense, gated or routed rows, normed or not, pass vector) + RMSNorm, "
        "+ input convolution of single tokens");
  m.def("embed_pairs", &embed_pairs, "token + token-pair embedding, normed");
  m.def("short_conv_rows", &short_conv_rows);
  m.def("short_conv_add", &short_conv_add, "input plus its causal convolution");
  m.def("xielu", &xielu, "xIELU activation");
  m.def("latent_front", &latent_front,
        "latent norm + rotated key part + paged scatter, norm of the queries' latent");
  m.def("latent_places", &latent_places, "where the visible context of portions lies");
  m.def("gather_latents", &gather_latents, "cached latent rows, packed");
  m.def("rotate_heads", &rotate_heads, "rotary positions of neighbouring pairs");
  m.def("head_linear", &head_linear,
        "per-head product with an optional gate, or beside rotated dimensions");
  m.def("latent_attention", &latent_attention,
        "MFMA attention in the latents' space over the paged cache, with sink and window");
  m.def("latent_attention_rows", &latent_attention_rows,
        "any latent width / float32 latent attention with sink and window");
  m.def("sink_attention_prefill", &sink_attention_prefill,
        "MFMA flash prefill with a sink and a gate per head");
  m.def("tailed_attention_prefill", &tailed_attention_prefill,
        "MFMA flash prefill whose heads share their keys' last dimensions, with a window");
  m.def("conv_qkv_rows", &conv_qkv_rows);
  m.def("conv_qkv", &conv_qkv,
        "causal convolution + rotation of heads and values + paged KV scatter");
  m.def("bias_kv_write", &bias_kv_write, "bias + head split + paged KV scatter");
  m.def("biased_prefill_rows", &biased_prefill_rows);
  m.def("biased_attention_prefill", &biased_attention_prefill,
        "MFMA flash prefill with distance bias, window or chunks, sink, turn and gate");
  m.def("fresh_attention_decode", &fresh_attention_decode,
        "rotation, cache write and decode attention of rows of different sequences");
  m.def("biased_attention_decode", &biased_attention_decode,
        "paged decode with distance bias, window or chunks, sink, turn and gate",
        py::arg("q"), py::arg("kc"), py::arg("vc"), py::arg("bt"), py::arg("ctx"),
        py::arg("scale"), py::arg("window"), py::arg("chunk"), py::arg("slopes"),
        py::arg("rates"), py::arg("sink"), py::arg("turn"), py::arg("gate"), py::arg("out"),
        py::arg("col"), py::arg("dv"), py::arg("oscale"), py::arg("marks") = py::none());
  m.def("biased_attention_rows", &biased_attention_rows,
        "any head width / float32 attention with distance bias, window or chunks, sink, "
        "turn and gate");
  m.def("delta_prefill", &delta_prefill, "gated delta rule, chunked");
  m.def("delta_decode", &delta_decode, "gated delta rule, one token per sequence");
  m.def("retention_prefill", &retention_prefill, "retention, chunked");
  m.def("retention_decode", &retention_decode, "retention, one token per sequence");
  m.def("moe_route", &moe_route, "fp32 router, top choice, softmax over the chosen");
  m.def("moe_silu_glu", &moe_silu_glu, "sorted grouped silu GLU experts");
  m.def("moe_combine", &moe_combine, "weighted sum of every token's expert rows");
  m.def("moe_route_grouped", &moe_route_grouped,
        "fp32 sigmoid or softmax router, top choice among the best groups");
  m.def("moe_relu2", &moe_relu2, "sorted grouped squared-relu experts");
  m.def("moe_clamped_glu", &moe_clamped_glu, "sorted grouped clamped-GLU experts");
  m.def("head_delta_prefill", &head_delta_prefill,
        "gated delta rule with a decay per head, chunked");
  m.def("head_delta_decode", &head_delta_decode,
        "gated delta rule with a decay per head, one token per sequence");
  m.def("memory_prefill", &memory_prefill, "matrix memory (mLSTM), chunked");
  m.def("memory_decode", &memory_decode, "matrix memory (mLSTM), one token per sequence");
  m.def("output_norm", &output_norm,
        "sub-layer result put together, layer norm, fp32 residual, depth average, "
        "final norm");
  m.def("normed_qkv", &normed_qkv,
        "head norms + rotation + temperature + paged KV scatter");
  m.def("pack_batch", &pack_batch, "a step's batch from lists, in one copy");
  m.def("pack_texts", &pack_texts, "texts to embed from lists, in one copy");
  m.def("pack_rows", &pack_rows, "integers to the device without waiting");
  m.def("stage_decode", &stage_decode, "the inputs of a captured decode step, in one copy");
  m.def("gelu", &gelu, "exact gelu");
  m.def("relu2", &relu2, "squared relu");
  m.def("silu_glu", &silu_glu, "silu(gate) * up");
}
