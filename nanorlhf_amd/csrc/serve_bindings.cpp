// Python bindings of the serving kernels: paged cache, attention over it,
// linear attention with its state slots, mixture of experts, residual-stream
// operations.
#include <torch/extension.h>

using OptTensor = c10::optional<torch::Tensor>;

// kvcache.hip
void kv_append(torch::Tensor k, torch::Tensor v, torch::Tensor slots,
               torch::Tensor k_cache, torch::Tensor v_cache);
std::vector<torch::Tensor> qkv_rope_append(torch::Tensor qkv, torch::Tensor table,
                                           torch::Tensor positions, torch::Tensor slots,
                                           torch::Tensor k_cache, torch::Tensor v_cache, long Hq,
                                           bool want_kv, OptTensor bias);
void copy_pages(std::vector<torch::Tensor> pools, torch::Tensor src, torch::Tensor dst);
torch::Tensor paged_attn_decode_new(torch::Tensor qkv, torch::Tensor table, torch::Tensor positions,
                                    torch::Tensor slots, torch::Tensor k_cache,
                                    torch::Tensor v_cache, torch::Tensor block_tables,
                                    torch::Tensor seq_lens, long Hq, OptTensor bias, double scale);
torch::Tensor paged_attn_decode(torch::Tensor q, torch::Tensor k_cache,
                                torch::Tensor v_cache, torch::Tensor block_tables,
                                torch::Tensor seq_lens, double scale);
void paged_attn_decode_window(torch::Tensor q, torch::Tensor k_cache, torch::Tensor v_cache,
                              torch::Tensor block_tables, torch::Tensor seq_lens,
                              torch::Tensor out, double scale, long size, long keep,
                              OptTensor uncs);
// paged_attention.hip
void paged_attn_varlen(torch::Tensor q, torch::Tensor kc, torch::Tensor vc, torch::Tensor cu,
                       torch::Tensor seq_lens, torch::Tensor bt, torch::Tensor out, long max_q,
                       double scale, long size, long keep, OptTensor uncs);
void paged_attn_plain(torch::Tensor q, torch::Tensor kc, torch::Tensor vc, torch::Tensor row_seq,
                      torch::Tensor positions, torch::Tensor bt, torch::Tensor out, double scale,
                      long size, long keep, OptTensor uncs);
// linear_attn.hip
long linear_attn_segment(long n, long B, long H, long D, long V);
void linear_attn_chunked(torch::Tensor q, torch::Tensor k, torch::Tensor v, torch::Tensor pw,
                         OptTensor cs, bool interleaved, bool silu, double kscale,
                         torch::Tensor chunks, torch::Tensor first, torch::Tensor slots,
                         torch::Tensor fresh, torch::Tensor state, OptTensor gate, double eps,
                         torch::Tensor o);
void linear_attn_decode(torch::Tensor q, torch::Tensor k, torch::Tensor v, torch::Tensor pw,
                        OptTensor cs, bool interleaved, bool silu, double kscale,
                        torch::Tensor slots, torch::Tensor seq_lens, torch::Tensor state,
                        OptTensor gate, double eps, torch::Tensor o);
// stream.hip
torch::Tensor residual_group_norm(torch::Tensor x, OptTensor delta, OptTensor embed,
                                  OptTensor ids, OptTensor add, OptTensor bias, OptTensor w,
                                  long groups, double mult, double eps, double offset,
                                  double gain);
void relu_squared_(torch::Tensor x);
void gated_norm(torch::Tensor in, OptTensor w, torch::Tensor gate, torch::Tensor out,
                long groups, long act, double eps);
void gelu_glu(torch::Tensor gate, torch::Tensor up, torch::Tensor out, long pad, long tail);
torch::Tensor rope_angles(torch::Tensor positions, torch::Tensor freqs);
torch::Tensor rotary_qkv(torch::Tensor proj, long qoff, long koff, long voff, OptTensor qw,
                         OptTensor kw, OptTensor csk, OptTensor csv, torch::Tensor slots,
                         torch::Tensor kc, torch::Tensor vc, long H, long G, long D, long V,
                         bool interleaved, double eps);

// glu.hip
torch::Tensor linear_mid(torch::Tensor x, torch::Tensor w, OptTensor u,
                         OptTensor b, OptTensor bias);
torch::Tensor linear_big(torch::Tensor x, torch::Tensor w, OptTensor bias);
std::vector<torch::Tensor> linear_big_rope(torch::Tensor x, torch::Tensor w, OptTensor bias,
                                           torch::Tensor table, torch::Tensor positions, long Hq,
                                           long Hkv);
void glu_linear(torch::Tensor x, torch::Tensor gate, torch::Tensor up, torch::Tensor out,
                long act);
// linear_rows.hip
torch::Tensor linear_rows(torch::Tensor x, torch::Tensor w, OptTensor bias);
torch::Tensor linear_rows_parts(torch::Tensor x, torch::Tensor w, OptTensor bias);
torch::Tensor linear_blocks(torch::Tensor x, torch::Tensor w, OptTensor bias);
torch::Tensor glu_rows(torch::Tensor x, torch::Tensor gate, torch::Tensor up);
// wkv.hip
void token_shift(torch::Tensor h, torch::Tensor mu, OptTensor seq_lens, torch::Tensor slots,
                 OptTensor cu, OptTensor row_seq, OptTensor fresh, torch::Tensor last,
                 torch::Tensor out, long row0, long rows);
torch::Tensor wkv_decay(torch::Tensor low, torch::Tensor w2, torch::Tensor w0);
void wkv_step(torch::Tensor r, torch::Tensor k, torch::Tensor v, torch::Tensor w, torch::Tensor u,
              torch::Tensor gate, torch::Tensor norm, double eps, torch::Tensor state,
              torch::Tensor slots, OptTensor seq_lens, OptTensor fresh, OptTensor cu,
              torch::Tensor out);
void wkv_chunked(torch::Tensor r, torch::Tensor k, torch::Tensor v, torch::Tensor w,
                 torch::Tensor u, torch::Tensor gate, torch::Tensor norm, double eps,
                 torch::Tensor state, torch::Tensor slots, torch::Tensor fresh,
                 torch::Tensor chunks, torch::Tensor first, torch::Tensor out);
// latent_attn.hip
void latent_append(torch::Tensor c, torch::Tensor w, torch::Tensor slots, torch::Tensor cache,
                   double eps);
torch::Tensor latent_gather(torch::Tensor cache, torch::Tensor bt, torch::Tensor seq_lens,
                            torch::Tensor first, long rows);
torch::Tensor latent_attn(torch::Tensor qa, torch::Tensor cache, OptTensor cu,
                          torch::Tensor seq_lens, torch::Tensor bt, long max_q, double scale);
torch::Tensor latent_attn_plain(torch::Tensor qa, torch::Tensor cache, torch::Tensor row_seq,
                                torch::Tensor positions, torch::Tensor bt, double scale);
// paged_attention.hip
void expanded_attn_varlen(torch::Tensor q, torch::Tensor k, torch::Tensor vt, torch::Tensor cu,
                          torch::Tensor seq_lens, torch::Tensor first, torch::Tensor out,
                          long heads, long max_q, double scale);
// moe.hip
void group_linear(torch::Tensor x, torch::Tensor w, torch::Tensor out);
bool group_linear_fills(long T, long G, long N, long K);
std::vector<torch::Tensor> moe_route(torch::Tensor h, torch::Tensor router, torch::Tensor bias,
                                     long top);
torch::Tensor moe_gate_up(torch::Tensor h, torch::Tensor gate_up, torch::Tensor lists,
                          torch::Tensor counts, long top);
torch::Tensor moe_down(torch::Tensor act, torch::Tensor down, torch::Tensor lists,
                       torch::Tensor counts, torch::Tensor weights);

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("kv_append", &kv_append);
  m.def("copy_pages", &copy_pages);
  m.def("qkv_rope_append", &qkv_rope_append, py::arg("qkv"), py::arg("table"),
        py::arg("positions"), py::arg("slots"), py::arg("k_cache"), py::arg("v_cache"),
        py::arg("heads"), py::arg("want_kv"), py::arg("bias") = py::none());
  m.def("paged_attn_decode", &paged_attn_decode);
  m.def("paged_attn_decode_new", &paged_attn_decode_new);
  m.def("paged_attn_decode_window", &paged_attn_decode_window);
  m.def("paged_attn_varlen", &paged_attn_varlen);
  m.def("paged_attn_plain", &paged_attn_plain);
  m.def("linear_attn_chunked", &linear_attn_chunked);
  m.def("linear_attn_segment", &linear_attn_segment);
  m.def("linear_attn_decode", &linear_attn_decode);
  m.def("residual_group_norm", &residual_group_norm);
  m.def("gated_norm", &gated_norm);
  m.def("gelu_glu", &gelu_glu);
  m.def("linear_big", &linear_big);
  m.def("linear_big_rope", &linear_big_rope);
  m.def("linear_mid", &linear_mid);
  m.def("glu_linear", &glu_linear);
  m.def("linear_rows", &linear_rows);
  m.def("linear_rows_parts", &linear_rows_parts);
  m.def("linear_blocks", &linear_blocks);
  m.def("glu_rows", &glu_rows);
  m.def("relu_squared_", &relu_squared_);
  m.def("token_shift", &token_shift);
  m.def("wkv_decay", &wkv_decay);
  m.def("wkv_step", &wkv_step);
  m.def("wkv_chunked", &wkv_chunked);
  m.def("latent_append", &latent_append);
  m.def("latent_gather", &latent_gather);
  m.def("latent_attn", &latent_attn);
  m.def("latent_attn_plain", &latent_attn_plain);
  m.def("expanded_attn_varlen", &expanded_attn_varlen);
  m.def("group_linear", &group_linear);
  m.def("group_linear_fills", &group_linear_fills);
  m.def("moe_route", &moe_route);
  m.def("moe_gate_up", &moe_gate_up);
  m.def("moe_down", &moe_down);
  m.def("rope_angles", &rope_angles);
  m.def("rotary_qkv", &rotary_qkv);
}
