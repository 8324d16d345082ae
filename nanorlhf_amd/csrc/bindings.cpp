// Python bindings for the nanorlhf_amd gfx950 HIP kernel library.
#include <torch/extension.h>

// elementwise.hip
std::vector<torch::Tensor> rmsnorm_fwd(torch::Tensor x, torch::Tensor w, double eps);
std::vector<torch::Tensor> rmsnorm_bwd(torch::Tensor dy, torch::Tensor x,
                                       torch::Tensor w, torch::Tensor invrms,
                                       c10::optional<torch::Tensor> extra, bool want_dw);
std::vector<torch::Tensor> rmsnorm_parts_fwd(torch::Tensor parts, torch::Tensor res,
                                             torch::Tensor w, double eps);
std::vector<torch::Tensor> rmsnorm_addres_fwd(torch::Tensor x, torch::Tensor res,
                                              torch::Tensor w, double eps);
torch::Tensor rope_fwd(torch::Tensor x, torch::Tensor table, torch::Tensor positions, double sign);
std::vector<torch::Tensor> qkv_rope_fwd(torch::Tensor qkv, torch::Tensor table,
                                        torch::Tensor positions, long Hq, long Hkv);
torch::Tensor qkv_rope_bwd(c10::optional<torch::Tensor> dq, c10::optional<torch::Tensor> dk,
                           c10::optional<torch::Tensor> dv, torch::Tensor table,
                           torch::Tensor positions, long Hq, long Hkv);
torch::Tensor swiglu_fwd(torch::Tensor gu);
torch::Tensor swiglu_bwd(torch::Tensor dy, torch::Tensor gu);
torch::Tensor embedding_grad(torch::Tensor ids, torch::Tensor dy, long V);
// logprob.hip
void ce_rowstats(torch::Tensor logits, torch::Tensor labels, double inv_temp,
                 torch::Tensor lp, torch::Tensor ent, torch::Tensor lse);
void ce_backward_dlogits(torch::Tensor logits, torch::Tensor labels,
                         torch::Tensor lse, torch::Tensor g, double inv_temp);
// adamw.hip
void adamw_step(torch::Tensor p, torch::Tensor g, torch::Tensor m, torch::Tensor v,
                double lr, double b1, double b2, double eps, double wd, long step);
void adamw_step_many(std::vector<torch::Tensor> p, std::vector<torch::Tensor> g,
                     std::vector<torch::Tensor> m, std::vector<torch::Tensor> v, double lr,
                     double b1, double b2, double eps, double wd, long step);
// sampling.hip
std::vector<torch::Tensor> decode_inputs(torch::Tensor lens, torch::Tensor bt, long page_size);
std::vector<torch::Tensor> embed_rms_norm(torch::Tensor ids, torch::Tensor table, torch::Tensor w,
                                          double eps, c10::optional<torch::Tensor> lens,
                                          c10::optional<torch::Tensor> bt, long page_size);
void decode_commit(torch::Tensor tokens, c10::optional<torch::Tensor> lps, torch::Tensor out,
                   torch::Tensor lp, torch::Tensor count, torch::Tensor lens, torch::Tensor last,
                   torch::Tensor finished, c10::optional<long> stop,
                   c10::optional<torch::Tensor> step);
torch::Tensor sample_topp(torch::Tensor logits, double temperature, double top_p,
                          long seed, long step);
std::vector<torch::Tensor> sample_topp_dev(torch::Tensor logits, double temperature,
                                           double top_p, long seed, torch::Tensor step,
                                           long ahead);
// masked.hip
std::vector<torch::Tensor> masked_moments(torch::Tensor v, torch::Tensor mask);
torch::Tensor whiten_apply(torch::Tensor v, double mean, double invstd, double shift);
// lora.hip
bool lora_gemm_big(long M, long N, long K);
long lora_gemm_tiles(long M, long K);
long lora_gemm_round(long M, long N, long K);
torch::Tensor lora_gemm(torch::Tensor x, torch::Tensor w,
                        c10::optional<torch::Tensor> u,
                        c10::optional<torch::Tensor> b,
                        c10::optional<torch::Tensor> bias);
std::vector<torch::Tensor> lora_glu(torch::Tensor x, torch::Tensor w, torch::Tensor u,
                                    torch::Tensor b);
void lora_add_(torch::Tensor y, torch::Tensor u, torch::Tensor b);
// attention.hip
std::vector<torch::Tensor> fa_fwd_varlen(torch::Tensor q, torch::Tensor k,
                                         torch::Tensor v, torch::Tensor cu_seqlens,
                                         long max_seqlen, double scale, bool causal);
long fa_head_window(long heads, long tiles, long rounds, bool causal);
long fa_bwd_parts(long T, long B, long Hq, long Hkv, long D, long max_seqlen);
std::vector<torch::Tensor> fa_bwd_varlen(torch::Tensor dout, torch::Tensor q,
                                         torch::Tensor k, torch::Tensor v,
                                         torch::Tensor o, torch::Tensor lse,
                                         torch::Tensor cu_seqlens, long max_seqlen,
                                         double scale, bool causal);

// lora_grad.hip
std::vector<torch::Tensor> lora_grads(c10::optional<torch::Tensor> x,
                                      c10::optional<torch::Tensor> du,
                                      c10::optional<torch::Tensor> dy,
                                      c10::optional<torch::Tensor> u);
torch::Tensor lora_down(torch::Tensor z, torch::Tensor p, double scale, bool flat);
std::vector<torch::Tensor> lora_forward(torch::Tensor x, torch::Tensor w,
                                        c10::optional<torch::Tensor> bias, torch::Tensor A,
                                        torch::Tensor B, double scale, bool fused);
std::vector<torch::Tensor> lora_backward(torch::Tensor dy, torch::Tensor x, torch::Tensor u,
                                         torch::Tensor A, torch::Tensor B, torch::Tensor w_t,
                                         double scale, bool fused, bool want_x, bool want_A,
                                         bool want_B);

// glu.hip
torch::Tensor linear_mid(torch::Tensor x, torch::Tensor w, c10::optional<torch::Tensor> u,
                         c10::optional<torch::Tensor> b, c10::optional<torch::Tensor> bias);
torch::Tensor linear_big(torch::Tensor x, torch::Tensor w, c10::optional<torch::Tensor> bias);
std::vector<torch::Tensor> linear_big_rope(torch::Tensor x, torch::Tensor w,
                                           c10::optional<torch::Tensor> bias, torch::Tensor table,
                                           torch::Tensor positions, long Hq, long Hkv);
void glu_linear(torch::Tensor x, torch::Tensor gate, torch::Tensor up, torch::Tensor out,
                long act);
// linear_rows.hip
torch::Tensor linear_rows(torch::Tensor x, torch::Tensor w, c10::optional<torch::Tensor> bias);
torch::Tensor linear_blocks(torch::Tensor x, torch::Tensor w, c10::optional<torch::Tensor> bias);
torch::Tensor linear_rows_parts(torch::Tensor x, torch::Tensor w,
                                c10::optional<torch::Tensor> bias);
torch::Tensor glu_rows(torch::Tensor x, torch::Tensor gate, torch::Tensor up);

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("rmsnorm_fwd", &rmsnorm_fwd);
  m.def("rmsnorm_bwd", &rmsnorm_bwd, py::arg("dy"), py::arg("x"), py::arg("w"),
        py::arg("invrms"), py::arg("extra") = py::none(), py::arg("want_dw") = true);
  m.def("rmsnorm_addres_fwd", &rmsnorm_addres_fwd);
  m.def("rmsnorm_parts_fwd", &rmsnorm_parts_fwd);
  m.def("rope_fwd", &rope_fwd);
  m.def("qkv_rope_fwd", &qkv_rope_fwd);
  m.def("qkv_rope_bwd", &qkv_rope_bwd);
  m.def("swiglu_fwd", &swiglu_fwd);
  m.def("swiglu_bwd", &swiglu_bwd);
  m.def("ce_rowstats", &ce_rowstats);
  m.def("ce_backward_dlogits", &ce_backward_dlogits);
  m.def("linear_big", &linear_big);
  m.def("linear_big_rope", &linear_big_rope);
  m.def("embedding_grad", &embedding_grad);
  m.def("linear_mid", &linear_mid);
  m.def("glu_linear", &glu_linear);
  m.def("linear_rows", &linear_rows);
  m.def("linear_rows_parts", &linear_rows_parts);
  m.def("linear_blocks", &linear_blocks);
  m.def("glu_rows", &glu_rows);
  m.def("lora_grads", &lora_grads);
  m.def("lora_glu", &lora_glu);
  m.def("lora_forward", &lora_forward);
  m.def("lora_backward", &lora_backward);
  m.def("lora_down", &lora_down);
  m.def("adamw_step", &adamw_step);
  m.def("adamw_step_many", &adamw_step_many);
  m.def("decode_inputs", &decode_inputs);
  m.def("embed_rms_norm", &embed_rms_norm, py::arg("ids"), py::arg("table"), py::arg("w"),
        py::arg("eps"), py::arg("lens") = py::none(), py::arg("bt") = py::none(),
        py::arg("page_size") = 0);
  m.def("decode_commit", &decode_commit, py::arg("tokens"), py::arg("lps"), py::arg("out"),
        py::arg("lp"), py::arg("count"), py::arg("lens"), py::arg("last"), py::arg("finished"),
        py::arg("stop"), py::arg("step") = py::none());
  m.def("sample_topp", &sample_topp);
  m.def("sample_topp_dev", &sample_topp_dev, py::arg("logits"), py::arg("temperature"),
        py::arg("top_p"), py::arg("seed"), py::arg("step"), py::arg("ahead") = 0);
  m.def("masked_moments", &masked_moments);
  m.def("whiten_apply", &whiten_apply);
  m.def("lora_gemm_big", &lora_gemm_big);
  m.def("lora_gemm_tiles", &lora_gemm_tiles);
  m.def("lora_gemm_round", &lora_gemm_round);
  m.def("lora_gemm", &lora_gemm, py::arg("x"), py::arg("w"),
        py::arg("u") = py::none(), py::arg("b") = py::none(),
        py::arg("bias") = py::none());
  m.def("lora_add_", &lora_add_);
  m.def("fa_fwd_varlen", &fa_fwd_varlen);
  m.def("fa_bwd_varlen", &fa_bwd_varlen);
  m.def("fa_bwd_parts", &fa_bwd_parts);
  m.def("fa_head_window", &fa_head_window);
}
