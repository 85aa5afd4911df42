// Python bindings of ``penroz_serve``: the decode-shaped GEMMs and the kernels of the packed decoder
// step (latent attention, causal convolution, grouped norms, experts). A module of its own, so a
// process that only steps such a model compiles and loads nothing else.
#include <torch/extension.h>
#include <hip/hip_runtime.h>
#include <vector>

// skinny_gemm.hip, decode_linear.hip
int64_t skinny_gemm(torch::Tensor x, torch::Tensor w, c10::optional<torch::Tensor> bias, torch::Tensor out,
                    torch::Tensor ws, torch::Tensor cnt, int64_t splitk);
void skinny_gated(torch::Tensor x, torch::Tensor gu, torch::Tensor out, int64_t kind);
std::vector<int64_t> skinny_qkv_rope_plan(int64_t M, int64_t N, int64_t K);
int64_t skinny_qkv_rope(torch::Tensor x, torch::Tensor w, torch::Tensor cosv, torch::Tensor sinv, int64_t D,
                        int64_t nrot, torch::Tensor out, torch::Tensor ws, torch::Tensor cnt, int64_t splitk);
void decode_ln_linear(torch::Tensor rin, c10::optional<torch::Tensor> delta, c10::optional<torch::Tensor> dbias,
                      c10::optional<torch::Tensor> rout, torch::Tensor gamma, torch::Tensor beta, double eps,
                      torch::Tensor w, c10::optional<torch::Tensor> bias, torch::Tensor out, int64_t act);
void decode_ln_gemm(torch::Tensor resid, torch::Tensor gamma, torch::Tensor beta, double eps, torch::Tensor w,
                    c10::optional<torch::Tensor> bias, torch::Tensor out, int64_t act);
void decode_gemv(c10::optional<torch::Tensor> x, c10::optional<torch::Tensor> rin, c10::optional<torch::Tensor> delta,
                 c10::optional<torch::Tensor> dbias, c10::optional<torch::Tensor> rout,
                 c10::optional<torch::Tensor> gamma, c10::optional<torch::Tensor> beta, double eps, torch::Tensor w,
                 c10::optional<torch::Tensor> bias, torch::Tensor out, int64_t act, int64_t rows_per_wave,
                 c10::optional<torch::Tensor> emb_idx, c10::optional<torch::Tensor> emb_wte,
                 c10::optional<torch::Tensor> emb_wpe, c10::optional<torch::Tensor> emb_pos, bool past);
void decode_gemv_pair(torch::Tensor x, torch::Tensor w, torch::Tensor out, int64_t mode, int64_t kind, int64_t D,
                      int64_t nrot, c10::optional<torch::Tensor> cosv, c10::optional<torch::Tensor> sinv,
                      int64_t pairs_per_wave, bool past);
void decode_norm_pair(c10::optional<torch::Tensor> x, c10::optional<torch::Tensor> a, c10::optional<torch::Tensor> w1, torch::Tensor w2,
                      int64_t step, double eps1, double eps2, c10::optional<torch::Tensor> h, torch::Tensor w, torch::Tensor out,
                      int64_t mode, int64_t kind, int64_t D, int64_t nrot, c10::optional<torch::Tensor> cosv,
                      c10::optional<torch::Tensor> sinv, c10::optional<torch::Tensor> tok, c10::optional<torch::Tensor> table,
                      double scale, bool past);
void decode_gemm_acc(torch::Tensor x, torch::Tensor w, c10::optional<torch::Tensor> bias, torch::Tensor resid, bool past);
void decode_gemm(torch::Tensor x, torch::Tensor w, torch::Tensor out, int64_t kind);
// rows_gemm.hip
c10::optional<torch::Tensor> rows_gemm(torch::Tensor x, torch::Tensor w, c10::optional<torch::Tensor> bias,
                                       c10::optional<torch::Tensor> out, bool fp32, bool in_order, bool gelu, bool past);
int64_t rows_gemm_tile(int64_t M, int64_t N, int64_t K, bool in_order);
// packed_rows.hip
void row_norm_add(c10::optional<torch::Tensor> tok, c10::optional<torch::Tensor> table,
                  c10::optional<torch::Tensor> x_in, c10::optional<torch::Tensor> x_out,
                  c10::optional<torch::Tensor> y, c10::optional<torch::Tensor> pw, c10::optional<torch::Tensor> nw,
                  int64_t groups, double eps, c10::optional<torch::Tensor> cw, c10::optional<torch::Tensor> state,
                  c10::optional<torch::Tensor> slot, c10::optional<torch::Tensor> pos, bool advance,
                  c10::optional<torch::Tensor> h);
void row_norm(torch::Tensor x, c10::optional<torch::Tensor> rows, torch::Tensor w, int64_t groups, double eps,
              torch::Tensor out);
void residual_norm(c10::optional<torch::Tensor> tok, c10::optional<torch::Tensor> table,
                   c10::optional<torch::Tensor> ptable, c10::optional<torch::Tensor> x_in,
                   c10::optional<torch::Tensor> x_out, c10::optional<torch::Tensor> ya, c10::optional<torch::Tensor> wa,
                   c10::optional<torch::Tensor> yb, c10::optional<torch::Tensor> wb, double coef, double yeps,
                   c10::optional<torch::Tensor> pw, c10::optional<torch::Tensor> ys, c10::optional<torch::Tensor> nw,
                   double eps, c10::optional<torch::Tensor> pos, bool advance, c10::optional<torch::Tensor> h);
void norm_conv_rows(torch::Tensor x, torch::Tensor x_out, torch::Tensor y, torch::Tensor nw, int64_t groups,
                    double eps, torch::Tensor cw, torch::Tensor state, torch::Tensor slot, torch::Tensor pos,
                    torch::Tensor first, torch::Tensor cu, torch::Tensor seq_slot, torch::Tensor h);
void conv_rows(torch::Tensor x, torch::Tensor cw, torch::Tensor state, torch::Tensor slot, torch::Tensor pos,
               torch::Tensor first, torch::Tensor cu, torch::Tensor seq_slot, torch::Tensor h);
// latent_attn.hip
void latent_store(torch::Tensor z, int64_t H, int64_t d8, int64_t r8, int64_t rot, int64_t R, int64_t R8,
                  c10::optional<torch::Tensor> nw, double eps, torch::Tensor tab, c10::optional<torch::Tensor> cache,
                  torch::Tensor slot, torch::Tensor pos, c10::optional<torch::Tensor> c_out,
                  c10::optional<torch::Tensor> kr_out, bool rotate_q);
void latent_gather(torch::Tensor cache, torch::Tensor kcu, torch::Tensor seq_slot, int64_t R8, int64_t r8,
                   torch::Tensor c_out, torch::Tensor kr_out);
void latent_absorb(torch::Tensor z, int64_t H, int64_t d8, int64_t r8, int64_t rot, int64_t R, torch::Tensor wuk,
                   torch::Tensor tab, torch::Tensor slot, torch::Tensor pos, torch::Tensor qa,
                   c10::optional<torch::Tensor> nw, double eps, c10::optional<torch::Tensor> cache);
void latent_attn_row(torch::Tensor qa, torch::Tensor cache, torch::Tensor slot, torch::Tensor pos, int64_t R8,
                     double scale, torch::Tensor ol);
// latent_mfma.hip
bool latent_decode_ok(int64_t R8, int64_t r8);
void latent_decode(torch::Tensor qa, torch::Tensor cache, torch::Tensor slot, torch::Tensor pos, int64_t R8,
                   double scale, torch::Tensor ol, torch::Tensor ml);
bool latent_flash_ok(int64_t Dk, int64_t v8);
void latent_flash(torch::Tensor z, torch::Tensor kv, torch::Tensor kr, torch::Tensor blocks, torch::Tensor cu,
                  torch::Tensor kcu, int64_t H, int64_t d8, int64_t r8, int64_t v8, double scale, torch::Tensor out);
void latent_uv(torch::Tensor ol, c10::optional<torch::Tensor> ml, torch::Tensor wuv, torch::Tensor out);
// experts.hip
void router_topk(c10::optional<torch::Tensor> logits, c10::optional<torch::Tensor> h, c10::optional<torch::Tensor> wr,
                 bool sigmoid, c10::optional<torch::Tensor> correction, double scale, bool renorm, torch::Tensor ids,
                 torch::Tensor wts);
void experts_plain(torch::Tensor h, torch::Tensor ids, torch::Tensor wgu, torch::Tensor wd, int64_t kind, double limit,
                   torch::Tensor act, torch::Tensor y);
void experts_rows(torch::Tensor h, torch::Tensor ids, torch::Tensor wgu, torch::Tensor wd, int64_t kind, double limit,
                  torch::Tensor act, torch::Tensor y, bool past);
c10::optional<std::tuple<torch::Tensor, torch::Tensor>> experts_rows_shared(torch::Tensor h, torch::Tensor ids, torch::Tensor wgu,
                                                                            torch::Tensor wd, double limit, torch::Tensor up,
                                                                            torch::Tensor down, bool past);
void experts_grouped(torch::Tensor h, torch::Tensor ids, torch::Tensor wgu, torch::Tensor wd, int64_t kind, double limit,
                     torch::Tensor act, torch::Tensor y, torch::Tensor perm, torch::Tensor tiles);
void gelu_rows(torch::Tensor u);
void gated_rows(torch::Tensor gu, int64_t kind, double limit, torch::Tensor out);
// window_attn.hip
void window_store(torch::Tensor z, std::vector<int64_t> sizes, torch::Tensor ktab, torch::Tensor vtab,
                  torch::Tensor cache, torch::Tensor pooled, torch::Tensor slot, torch::Tensor pos, bool one);
bool window_rows_ok(int64_t d8, int64_t v8);
void window_rows(torch::Tensor z, std::vector<int64_t> sizes, double scale, double cap, torch::Tensor cache,
                 torch::Tensor pooled, torch::Tensor pb, torch::Tensor vtab, torch::Tensor slot, torch::Tensor pos,
                 int64_t ranges, c10::optional<torch::Tensor> ol, torch::Tensor out);
// window_mfma.hip
bool window_flash_ok(int64_t d8, int64_t v8);
void window_flash(torch::Tensor z, std::vector<int64_t> sizes, double scale, double cap, torch::Tensor cache,
                  torch::Tensor pooled, torch::Tensor pb, torch::Tensor vtab, torch::Tensor blocks, torch::Tensor cu,
                  torch::Tensor seq_slot, torch::Tensor slot, torch::Tensor pos, torch::Tensor out);
// linear_attn.hip
void linear_step(torch::Tensor z, std::vector<int64_t> sizes, double scale, double eps, double tau,
                 c10::optional<torch::Tensor> decay, c10::optional<torch::Tensor> wa, c10::optional<torch::Tensor> ba,
                 torch::Tensor state, c10::optional<torch::Tensor> nw, torch::Tensor cu, torch::Tensor seq_slot,
                 torch::Tensor pos, torch::Tensor out);
void linear_decode(torch::Tensor z, std::vector<int64_t> sizes, double scale, double eps, double tau,
                   c10::optional<torch::Tensor> decay, c10::optional<torch::Tensor> wa, c10::optional<torch::Tensor> ba,
                   torch::Tensor state, c10::optional<torch::Tensor> nw, torch::Tensor cu, torch::Tensor seq_slot,
                   torch::Tensor pos, torch::Tensor out);
// linear_mfma.hip
bool linear_chunk_ok(int64_t d8, int64_t v8);
void linear_chunk(torch::Tensor z, std::vector<int64_t> sizes, double scale, double eps, double tau,
                  c10::optional<torch::Tensor> decay, c10::optional<torch::Tensor> wa, c10::optional<torch::Tensor> ba,
                  torch::Tensor state, c10::optional<torch::Tensor> nw, torch::Tensor cu, torch::Tensor seq_slot,
                  torch::Tensor pos, c10::optional<torch::Tensor> zdec, torch::Tensor spans, torch::Tensor cs, int64_t span,
                  c10::optional<torch::Tensor> ws, c10::optional<torch::Tensor> wdec, torch::Tensor out);

PYBIND11_MODULE(penroz_serve, m) {
  m.doc() = "penroz HIP kernels of the serving step for MI355X (gfx950)";
  m.def("skinny_gemm", &skinny_gemm, pybind11::arg("x"), pybind11::arg("w"), pybind11::arg("bias"),
        pybind11::arg("out"), pybind11::arg("ws"), pybind11::arg("cnt"), pybind11::arg("splitk") = 0,
        "decode-shaped out[M<=64, N] = x·wᵀ (+bias), bf16; returns the split-K factor used");
  m.def("skinny_gated", &skinny_gated, pybind11::arg("x"), pybind11::arg("gu"), pybind11::arg("out"),
        pybind11::arg("kind"),
        "decode gated MLP projection: out[M<=64, I] = act(x·gu[:I]ᵀ)·(x·gu[I:]ᵀ), bf16, one launch");
  m.def("skinny_qkv_rope_plan", &skinny_qkv_rope_plan, pybind11::arg("M"), pybind11::arg("N"), pybind11::arg("K"),
        "(split-K, fp32 workspace floats, counters) skinny_qkv_rope uses at this shape (host only)");
  m.def("skinny_qkv_rope", &skinny_qkv_rope, pybind11::arg("x"), pybind11::arg("w"), pybind11::arg("cos"),
        pybind11::arg("sin"), pybind11::arg("D"), pybind11::arg("nrot"), pybind11::arg("out"), pybind11::arg("ws"),
        pybind11::arg("cnt"), pybind11::arg("splitk") = 0,
        "decode QKV projection with RoPE on the first nrot heads in the epilogue, M <= 64; returns the split");
  m.def("decode_ln_linear", &decode_ln_linear, pybind11::arg("resid_in"), pybind11::arg("delta"),
        pybind11::arg("dbias"), pybind11::arg("resid_out"), pybind11::arg("gamma"), pybind11::arg("beta"),
        pybind11::arg("eps"), pybind11::arg("w"), pybind11::arg("bias"), pybind11::arg("out"), pybind11::arg("act") = 0,
        "decode step: out = act(LN(resid_in + delta + dbias)·wᵀ + bias) for M <= 64 rows, K <= 1024; "
        "resid_out receives the residual sum");
  m.def("decode_ln_gemm", &decode_ln_gemm, pybind11::arg("resid"), pybind11::arg("gamma"), pybind11::arg("beta"),
        pybind11::arg("eps"), pybind11::arg("w"), pybind11::arg("bias"), pybind11::arg("out"), pybind11::arg("act") = 0,
        "batched decode: out = act(LayerNorm(resid)·wᵀ + bias), fp32 resid [M, K <= 1024]");
  m.def("decode_gemv", &decode_gemv, pybind11::arg("x"), pybind11::arg("resid_in"), pybind11::arg("delta"),
        pybind11::arg("dbias"), pybind11::arg("resid_out"), pybind11::arg("gamma"), pybind11::arg("beta"),
        pybind11::arg("eps"), pybind11::arg("w"), pybind11::arg("bias"), pybind11::arg("out"), pybind11::arg("act") = 0,
        pybind11::arg("rows_per_wave") = 0, pybind11::arg("emb_idx") = pybind11::none(),
        pybind11::arg("emb_wte") = pybind11::none(), pybind11::arg("emb_wpe") = pybind11::none(),
        pybind11::arg("emb_pos") = pybind11::none(), pybind11::arg("past") = false,
        "decode GEMV for 1..4 rows: act(x · Wᵀ + bias), or act(LN(resid_in + delta + dbias) · Wᵀ + bias), or "
        "act(LN(wte[idx] + wpe[pos]) · Wᵀ + bias) with the embedding rows written to resid_out");
  m.def("decode_gemv_pair", &decode_gemv_pair, pybind11::arg("x"), pybind11::arg("w"), pybind11::arg("out"),
        pybind11::arg("mode"), pybind11::arg("kind") = 0, pybind11::arg("D") = 0, pybind11::arg("nrot") = 0,
        pybind11::arg("cos") = pybind11::none(), pybind11::arg("sin") = pybind11::none(),
        pybind11::arg("pairs_per_wave") = 0, pybind11::arg("past") = false,
        "paired-row decode GEMV for 1..4 rows: gated MLP (mode 1) or RoPE QKV (mode 2) epilogue");
  m.def("decode_norm_pair", &decode_norm_pair, pybind11::arg("x"), pybind11::arg("a"), pybind11::arg("w1"), pybind11::arg("w2"),
        pybind11::arg("step"), pybind11::arg("eps1"), pybind11::arg("eps2"), pybind11::arg("h"), pybind11::arg("w"),
        pybind11::arg("out"), pybind11::arg("mode"), pybind11::arg("kind") = 0, pybind11::arg("D") = 0, pybind11::arg("nrot") = 0,
        pybind11::arg("cos") = pybind11::none(), pybind11::arg("sin") = pybind11::none(), pybind11::arg("tok") = pybind11::none(),
        pybind11::arg("table") = pybind11::none(), pybind11::arg("scale") = 1.0, pybind11::arg("past") = false,
        "decode_gemv_pair behind the residual add and norms of a Gemma block (rms_residual), for 1..4 rows");
  m.def("rows_gemm", &rows_gemm, pybind11::arg("x"), pybind11::arg("w"), pybind11::arg("bias"), pybind11::arg("out"),
        pybind11::arg("fp32") = false, pybind11::arg("in_order") = false, pybind11::arg("gelu") = false, pybind11::arg("past") = false);
  m.def("rows_gemm_tile", &rows_gemm_tile, pybind11::arg("M"), pybind11::arg("N"), pybind11::arg("K"),
        pybind11::arg("in_order") = false);
  m.def("decode_gemm_acc", &decode_gemm_acc, pybind11::arg("x"), pybind11::arg("w"), pybind11::arg("bias"),
        pybind11::arg("resid"), pybind11::arg("past") = false,
        "batched decode: resid += x·wᵀ + bias (fp32 residual, in place)");
  m.def("decode_gemm", &decode_gemm, pybind11::arg("x"), pybind11::arg("w"), pybind11::arg("out"),
        pybind11::arg("kind") = -1,
        "batched decode (16-64 rows): out = x·wᵀ, or the gated MLP act(x·Wgᵀ)·(x·Wuᵀ) of a packed [gate; up] weight");
  m.def("row_norm_add", &row_norm_add, pybind11::arg("tok"), pybind11::arg("table"), pybind11::arg("x_in"),
        pybind11::arg("x_out"), pybind11::arg("y"), pybind11::arg("pw"), pybind11::arg("nw"), pybind11::arg("groups"),
        pybind11::arg("eps"), pybind11::arg("cw"), pybind11::arg("state"), pybind11::arg("slot"), pybind11::arg("pos"),
        pybind11::arg("advance"), pybind11::arg("h"),
        "x += grouped RMS norm(y)·nw; h = x + causal conv(x) (one new token per sequence)");
  m.def("row_norm", &row_norm, "grouped RMS norm of selected fp32 rows");
  m.def("norm_conv_rows", &norm_conv_rows, "x_out = x + grouped norm(y) and h = x_out + causal conv(x_out), in one pass");
  m.def("conv_rows", &conv_rows, "h = x + causal conv(x) over packed sequences; moves their states on");
  m.def("latent_store", &latent_store, "norm, rotate and cache the latent rows of a projection; rotate its queries");
  m.def("latent_gather", &latent_gather, "cached latent rows of sequences, packed");
  m.def("latent_absorb", &latent_absorb, "queries in latent space (+ the step's latent rows into the cache)");
  m.def("latent_attn_row", &latent_attn_row, "latent attention, one wave per (token, head)");
  m.def("latent_uv", &latent_uv, "merge key ranges and apply the value up-projection per head");
  m.def("router_topk", &router_topk, "softmax or sigmoid router: chosen experts and their weights");
  m.def("experts_plain", &experts_plain, "gated experts, one wave per output value");
  m.def("latent_decode_ok", &latent_decode_ok, "latent_decode takes these sizes");
  m.def("latent_decode", &latent_decode, "latent attention of single rows over the cache, split over key ranges (MFMA)");
  m.def("latent_flash_ok", &latent_flash_ok, "latent_flash takes these sizes");
  m.def("latent_flash", &latent_flash, "causal attention of packed prompts / portions over expanded keys (MFMA)");
  m.def("experts_rows", &experts_rows, pybind11::arg("h"), pybind11::arg("ids"), pybind11::arg("wgu"), pybind11::arg("wd"),
        pybind11::arg("kind"), pybind11::arg("limit"), pybind11::arg("act"), pybind11::arg("y"), pybind11::arg("past") = false,
        "gated experts of few (token, expert) pairs (MFMA)");
  m.def("experts_rows_shared", &experts_rows_shared, pybind11::arg("h"), pybind11::arg("ids"), pybind11::arg("wgu"),
        pybind11::arg("wd"), pybind11::arg("limit"), pybind11::arg("up"), pybind11::arg("down"), pybind11::arg("past") = false,
        "experts_rows of ungated experts and a shared expert of twice their width in the same launches, or None");
  m.def("experts_grouped", &experts_grouped, "gated experts of pairs grouped by expert (MFMA tiles)");
  m.def("gated_rows", &gated_rows, "act(g)·u of packed [g | u] rows");
  m.def("gelu_rows", &gelu_rows, "gelu (erf form) in place");
  m.def("residual_norm", &residual_norm, "x += a sublayer's output (or embedding rows); h = rms_norm(x)·w");
  m.def("window_store", &window_store, "rotate queries, keys and values of a projection; cache rows and pooled blocks");
  m.def("window_rows_ok", &window_rows_ok, "window_rows takes these sizes");
  m.def("window_rows", &window_rows, "sigmoid attention of single rows over a window and pooled blocks");
  m.def("window_flash_ok", &window_flash_ok, "window_flash takes these sizes");
  m.def("window_flash", &window_flash, "sigmoid attention of prompts / portions over window tiles and pooled tiles (MFMA)");
  m.def("linear_step", &linear_step, "linear attention, token by token (short portions)");
  m.def("linear_decode", &linear_decode, "linear attention of one token per sequence");
  m.def("linear_chunk_ok", &linear_chunk_ok, "linear_chunk takes these sizes");
  m.def("linear_chunk", &linear_chunk, "linear attention of prompts / portions in chunks (MFMA)");
}
