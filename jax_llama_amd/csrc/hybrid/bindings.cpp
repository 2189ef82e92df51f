// Python bindings of the hybrid-mixer kernels (module jax_llama_amd._C_hybrid). Thin: validate dtypes, shapes and
// contiguity on the host (a wrong shape must never reach a kernel), take raw pointers and launch on torch's current HIP
// stream, so hipGraph capture through torch.cuda.graph records these launches.
#include <torch/extension.h>
#include <c10/hip/HIPStream.h>

#include "hybrid.h"

namespace {

using torch::Tensor;
using OptT = c10::optional<Tensor>;

hipStream_t stream() { return c10::hip::getCurrentHIPStream().stream(); }

void check(bool cond, const char* msg) { TORCH_CHECK(cond, "jax_llama_amd._C_hybrid: ", msg); }

void rc(int r, const char* what) { TORCH_CHECK(r == 0, "jax_llama_amd._C_hybrid: ", what, " failed (code ", r, ")"); }

void gpu(const Tensor& t, const char* name) {
  TORCH_CHECK(t.is_cuda(), "jax_llama_amd._C_hybrid: ", name, " must be a GPU tensor");
  TORCH_CHECK(t.is_contiguous(), "jax_llama_amd._C_hybrid: ", name, " must be contiguous");
}

const float* f32(const Tensor& t, const char* name) {
  gpu(t, name);
  TORCH_CHECK(t.scalar_type() == torch::kFloat32, "jax_llama_amd._C_hybrid: ", name, " must be float32");
  return reinterpret_cast<const float*>(t.data_ptr());
}
float* f32w(const Tensor& t, const char* name) { return const_cast<float*>(f32(t, name)); }

const int32_t* i32(const Tensor& t, const char* name, int64_t min_numel) {
  gpu(t, name);
  TORCH_CHECK(t.scalar_type() == torch::kInt32 && t.numel() >= min_numel, "jax_llama_amd._C_hybrid: ", name,
              " must be int32 with at least ", min_numel, " elements");
  return reinterpret_cast<const int32_t*>(t.data_ptr());
}
int32_t* i32w(const Tensor& t, const char* name, int64_t n) { return const_cast<int32_t*>(i32(t, name, n)); }

// weight / cache element type: 1 = bf16, 0 = fp32
int wtype(const Tensor& t, const char* name) {
  gpu(t, name);
  TORCH_CHECK(t.scalar_type() == torch::kBFloat16 || t.scalar_type() == torch::kFloat32, "jax_llama_amd._C_hybrid: ",
              name, " must be bfloat16 or float32");
  return t.scalar_type() == torch::kBFloat16;
}

// a 2-d fp32 or bf16 view with unit inner stride (rows may be strided); *bf = 1 for bf16
void* rows2d_any(const Tensor& t, const char* name, int64_t cols, int* ld, int* bf) {
  TORCH_CHECK(t.is_cuda() && (t.scalar_type() == torch::kFloat32 || t.scalar_type() == torch::kBFloat16) &&
                  t.dim() == 2 && t.stride(1) == 1 && t.size(1) == cols && t.stride(0) >= cols,
              "jax_llama_amd._C_hybrid: ", name, " must be a float32 / bfloat16 [rows, ", cols,
              "] GPU view with unit inner stride");
  *ld = (int)t.stride(0);
  *bf = t.scalar_type() == torch::kBFloat16;
  return t.data_ptr();
}

// a 2-d fp32 view with unit inner stride (rows may be strided)
const float* rows2d(const Tensor& t, const char* name, int64_t cols, int* ld) {
  TORCH_CHECK(t.is_cuda() && t.scalar_type() == torch::kFloat32 && t.dim() == 2 && t.stride(1) == 1 &&
                  t.size(1) == cols && t.stride(0) >= cols,
              "jax_llama_amd._C_hybrid: ", name, " must be a float32 [rows, ", cols, "] GPU view with unit inner stride");
  *ld = (int)t.stride(0);
  return reinterpret_cast<const float*>(t.data_ptr());
}

void embed_rows(Tensor ids, Tensor table, int64_t col0, Tensor out, double scale, int64_t copies, OptT norm, double eps) {
  const int wb = wtype(table, "table");
  check(table.dim() == 2 && out.dim() == 2 && copies >= 1 && out.size(0) % copies == 0,
        "embed_rows: 2-d table, out is [copies * M, D]");
  const int M = out.size(0) / copies, D = out.size(1);
  check(!norm.has_value() || norm->numel() == D, "embed_rows: norm is [D]");
  rc(jla::hy_embed_rows(i32(ids, "ids", M), table.data_ptr(), wb, table.size(0), table.size(1), col0,
                        (float)scale, f32w(out, "out"), M, D, copies, norm.has_value() ? f32(*norm, "norm") : nullptr, eps, stream()),
     "embed_rows");
}

jla::RowLinear row_linear_any(Tensor a, OptT a_idx, Tensor w, Tensor out, OptT dst_idx, OptT offs, OptT row_expert, int64_t R,
                          int64_t act, double act_limit, double act_alpha, OptT a_scale, OptT a_norm_w, double a_norm_eps,
                          int64_t even_rows, bool add_out, bool tabled) {
  jla::RowLinear p{};
  p.even_rows = even_rows;
  p.add_out = add_out;
  p.wbf16 = wtype(w, "w");
  check(w.dim() == 2 || w.dim() == 3, "linear_rows: w is [Nw, K] or [E, Nw, K]");
  p.E = w.dim() == 3 ? w.size(0) : 1;
  const int64_t Nw = w.size(-2);
  p.K = w.size(-1);
  check(act >= jla::HY_ACT_NONE && act <= jla::HY_ACT_GELU_GLU, "linear_rows: unknown activation");
  const bool gated = jla::hy_act_gated(act);
  check(!gated || Nw % 2 == 0, "linear_rows: a gated activation needs gate and up rows");
  p.N = gated ? Nw / 2 : Nw;
  p.w = w.data_ptr();
  p.w_stride = Nw * (int64_t)p.K;
  p.a = rows2d_any(a, "a", p.K, &p.lda, &p.a_bf16);
  p.out = rows2d_any(out, "out", p.N, &p.ldo, &p.out_bf16);
  p.R = R;
  p.act = act;
  p.act_limit = act_limit;
  p.act_alpha = act_alpha;
  check(R >= 0, "linear_rows: R");
  if (a_idx.has_value()) p.a_idx = i32(*a_idx, "a_idx", R);
  else check(a.size(0) >= R, "linear_rows: a has fewer rows than R");
  if (dst_idx.has_value()) p.dst_idx = i32(*dst_idx, "dst_idx", R);
  else check(out.size(0) >= R, "linear_rows: out has fewer rows than R");
  if (offs.has_value()) p.offs = i32(*offs, "offs", p.E + 1);
  if (row_expert.has_value()) p.row_expert = i32(*row_expert, "row_expert", R);
  if (a_scale.has_value()) {
    check(a_scale->numel() >= R && !p.a_bf16, "linear_rows: a_scale is [R] and needs float32 activations");
    p.a_scale = f32(*a_scale, "a_scale");
  }
  if (a_norm_w.has_value()) {
    check(a_norm_w->numel() == p.K && !p.a_bf16, "linear_rows: a_norm_w is [K] and needs float32 activations");
    p.a_norm_w = f32(*a_norm_w, "a_norm_w");
    p.a_norm_eps = a_norm_eps;
  }
  check(p.E == 1 || p.offs || p.row_expert || tabled, "linear_rows: stacked experts need offs or row_expert");
  return p;
}

jla::RowLinear row_linear(Tensor a, OptT a_idx, Tensor w, Tensor out, OptT dst_idx, OptT offs, OptT row_expert, int64_t R,
                          int64_t act, double act_limit, double act_alpha, OptT a_scale, OptT a_norm_w, double a_norm_eps,
                          int64_t even_rows, bool add_out) {
  return row_linear_any(a, a_idx, w, out, dst_idx, offs, row_expert, R, act, act_limit, act_alpha, a_scale, a_norm_w, a_norm_eps,
                        even_rows, add_out, false);
}

// scratch of a call, from the allocator of the stream that uses it
Tensor row_scratch(long long floats, const Tensor& like) {
  return floats > 0 ? torch::empty({floats}, like.options().dtype(torch::kFloat32)) : Tensor();
}
float* scratch_ptr(const Tensor& t) { return t.defined() ? reinterpret_cast<float*>(t.data_ptr()) : nullptr; }

void linear_rows(Tensor a, OptT a_idx, Tensor w, Tensor out, OptT dst_idx, OptT offs, OptT row_expert, int64_t R,
                 int64_t act, double act_limit, double act_alpha, OptT a_scale, OptT a_norm_w, double a_norm_eps,
                 int64_t even_rows, bool add_out) {
  const jla::RowLinear p = row_linear(a, a_idx, w, out, dst_idx, offs, row_expert, R, act, act_limit, act_alpha, a_scale,
                                      a_norm_w, a_norm_eps, even_rows, add_out);
  const Tensor ws = row_scratch(jla::hy_linear_rows_floats(p), out);
  rc(jla::hy_linear_rows(p, scratch_ptr(ws), stream()), "linear_rows");
}

// A pending residual add (res_y .. res_out) onto the activations of p: [rows, K], rows of y res_nsum per activation row
void set_residual(jla::RowLinear& p, const Tensor& a, const OptT& y, int64_t nsum, double ysc, const OptT& w, double eps,
                  const OptT& x_out) {
  if (!y.has_value()) return;
  check(w.has_value() && x_out.has_value() && (w->numel() == 1 || w->numel() == p.K) && nsum >= 1,
        "residual: one gain or one per column, nsum >= 1");
  check(a.is_contiguous() && y->numel() == a.numel() * nsum && x_out->sizes() == a.sizes() &&
            x_out->data_ptr() != a.data_ptr(), "residual: y is [rows * nsum, K], x_out another [rows, K]");
  p.res_y = f32(*y, "y");
  p.res_nsum = nsum;
  p.res_ysc = ysc;
  p.res_w = f32(*w, "w");
  p.res_w_vec = w->numel() != 1;
  p.res_eps = eps;
  p.res_out = f32w(*x_out, "x_out");
}

// out = f(a' @ w^T) for a few rows in one launch: a' = a + rms_norm(ysc * sum of nsum rows of y) * res_w with y (written to x_out
// too), then normed with gain a_norm_w where that is given; f = act, then with ids gelu_tanh * table[ids, col0 ..]. False: not a call of that kernel, nothing was launched.
bool rows_fused(Tensor a, Tensor w, Tensor out, OptT y, int64_t nsum, double ysc, OptT res_w, double eps, OptT x_out, OptT ids,
                OptT table, int64_t col0, OptT a_norm_w, double a_norm_eps, int64_t act, double act_limit) {
  const bool one = a_norm_w.has_value() && a_norm_w->numel() == 1 && w.size(-1) != 1;
  jla::RowLinear p = row_linear(a, c10::nullopt, w, out, c10::nullopt, c10::nullopt, c10::nullopt, a.size(0), act, act_limit, 1.0,
                                c10::nullopt, one ? OptT() : a_norm_w, a_norm_eps, 0, false);
  if (one) {
    check(!p.a_bf16, "rows_fused: a normed row is float32");
    p.a_norm_w = f32(*a_norm_w, "a_norm_w");
    p.a_norm_eps = a_norm_eps;
    p.a_norm_one = 1;
  }
  check(act != jla::HY_ACT_SOFTCAP || act_limit > 0, "rows_fused: softcap");
  set_residual(p, a, y, nsum, ysc, res_w, eps, x_out);
  if (ids.has_value()) {
    check(table.has_value() && table->dim() == 2 && col0 >= 0 && col0 + p.N <= table->size(1), "rows_fused: table columns");
    p.mul_ids = i32(*ids, "ids", p.R);
    p.mul_bf16 = wtype(*table, "table");
    p.mul_table = table->data_ptr();
    p.mul_V = table->size(0); p.mul_ld = table->size(1); p.mul_col0 = col0;
    check(p.mul_V >= 1, "rows_fused: empty table");
  }
  if (p.R == 0 || p.N < 1 || !(p.res_y || one ? jla::hy_rows_gemv_takes_residual(p) : jla::hy_rows_gemv_takes(p))) return false;
  rc(jla::hy_rows_gemv(p, stream()), "rows_fused");
  return true;
}

// The largest of the (softcapped) products of one or two normed rows, the pending residual add included, per workgroup: [R, n, 2] (value,
// column bits). None: not a call of that kernel, nothing was launched.
OptT rows_best(Tensor a, Tensor w, OptT y, int64_t nsum, double ysc, OptT res_w, double eps, OptT x_out, Tensor a_norm_w,
               double a_norm_eps, double cap) {
  const bool one = a_norm_w.numel() == 1 && w.size(-1) != 1;
  jla::RowLinear p{};
  check(a.dim() == 2 && w.dim() == 2 && w.size(1) == a.size(1), "rows_best: a [R, K], w [N, K]");
  p.wbf16 = wtype(w, "w");
  p.E = 1; p.K = a.size(1); p.N = w.size(0); p.R = a.size(0);
  p.w = w.data_ptr();
  p.w_stride = (long long)p.N * p.K;
  p.a = rows2d(a, "a", p.K, &p.lda);
  p.act = cap > 0 ? jla::HY_ACT_SOFTCAP : jla::HY_ACT_NONE;
  p.act_limit = cap;
  p.a_norm_w = f32(a_norm_w, "a_norm_w");
  check(one || a_norm_w.numel() == p.K, "rows_best: norm gain");
  p.a_norm_one = one;
  p.a_norm_eps = a_norm_eps;
  set_residual(p, a, y, nsum, ysc, res_w, eps, x_out);
  if (p.R == 0 || p.N < 1 || !(p.res_y || one ? jla::hy_rows_gemv_takes_residual(p) : jla::hy_rows_gemv_takes(p))) return c10::nullopt;
  const int groups = jla::hy_rows_walk_groups(p);
  if (groups < 1) return c10::nullopt;
  Tensor best = torch::empty({(int64_t)p.R, (int64_t)groups, 2}, a.options());
  p.best = reinterpret_cast<float2*>(best.data_ptr());
  rc(jla::hy_rows_gemv(p, stream()), "rows_best");
  return best;
}

// Several matrices on one or two normed rows, blended or not, in one launch: out[i] = ws[i] v_i, v = rms_norm(x) gain, blended v + (prev -
// v) mu[mix[i]] for mix[i] >= 0, capped (cap[i] > 0); row <- v. False: not a call of that kernel, nothing was launched.
bool rows_parts(Tensor x, Tensor gain, double eps, Tensor prev, Tensor mu, std::vector<Tensor> ws, std::vector<int64_t> mix,
                std::vector<double> cap, std::vector<Tensor> outs, Tensor row) {
  const int64_t R = x.size(0), K = x.size(1);
  check(x.dim() == 2 && mu.dim() == 2 && mu.size(1) == K && gain.numel() == K && prev.numel() == R * K && row.numel() == R * K,
        "rows_parts: rows of x, prev, row; mu and gain of its width");
  check(ws.size() == mix.size() && ws.size() == cap.size() && ws.size() == outs.size(), "rows_parts: parts");
  if (ws.empty() || ws.size() > (size_t)jla::RV_MAX_PARTS) return false;
  jla::RowLinear p{};
  p.a = rows2d(x, "x", K, &p.lda);
  p.K = K; p.R = R; p.E = 1;
  p.wbf16 = wtype(ws[0], "w");
  p.a_norm_w = f32(gain, "gain");
  p.a_norm_eps = eps;
  jla::RowParts t{};
  t.n = ws.size();
  t.prev = f32(prev, "prev");
  t.mu = f32(mu, "mu");
  t.row = f32w(row, "row");
  for (int i = 0; i < t.n; ++i) {
    if (wtype(ws[i], "w") != p.wbf16) return false;
    check(ws[i].dim() == 2 && ws[i].size(1) == K && mix[i] < mu.size(0), "rows_parts: w is [N, K], mix a row of mu");
    t.w[i] = ws[i].data_ptr();
    t.N[i] = ws[i].size(0);
    t.out[i] = const_cast<float*>(rows2d(outs[i], "out", t.N[i], &t.ldo[i]));
    check(outs[i].size(0) == R, "rows_parts: out rows");
    t.mix[i] = std::max<int64_t>(mix[i], -1);
    t.cap[i] = cap[i];
  }
  if (!jla::hy_rows_parts_takes(p, t)) return false;
  rc(jla::hy_rows_parts(p, t, stream()), "rows_parts");
  return true;
}

// Both products of a few tokens' table-chosen SwiGLU experts, the table read by the products: h [M * top, F], out [M * top, D] in
// (token, choice) order. False: not a call of that kernel, nothing was launched.
bool table_rows(Tensor a, Tensor ids, Tensor table, Tensor w_gu, Tensor w_down, Tensor h, Tensor out, OptT y, int64_t nsum,
                double ysc, OptT res_w, double eps, OptT x_out) {
  check(table.dim() == 2 && w_gu.dim() == 3 && w_down.dim() == 3 && w_gu.size(0) == w_down.size(0), "table_rows: shapes");
  const int64_t M = a.size(0), top = table.size(1), R = M * top;
  check(top >= 1 && R <= 0x7fffffff && h.size(0) == R && out.size(0) == R, "table_rows: rows");
  if (R == 0 || R > jla::HY_GEMV_MAX_R) return false;
  // (checked as M rows: linear row r of the first product reads activation row r / top)
  jla::RowLinear p = row_linear_any(a, c10::nullopt, w_gu, h, c10::nullopt, c10::nullopt, c10::nullopt, M, jla::HY_ACT_SWIGLU, 0.0,
                                1.0, c10::nullopt, c10::nullopt, 0.0, 0, false, true);
  jla::RowLinear q = row_linear_any(h, c10::nullopt, w_down, out, c10::nullopt, c10::nullopt, c10::nullopt, R, 0, 0.0, 1.0,
                                c10::nullopt, c10::nullopt, 0.0, 0, false, true);
  p.R = R;
  p.a_div = top;
  for (jla::RowLinear* l : {&p, &q}) {
    l->tab = i32(table, "table", table.numel());
    l->tab_ids = i32(ids, "ids", M);
    l->tab_V = table.size(0);
    l->tab_top = top;
  }
  check(p.tab_V >= 1 && q.K == p.N, "table_rows: shapes");
  set_residual(p, a, y, nsum, ysc, res_w, eps, x_out);
  if (!(p.res_y ? jla::hy_rows_gemv_takes_residual(p) : jla::hy_rows_gemv_takes(p)) || !jla::hy_rows_gemv_takes(q)) return false;
  rc(jla::hy_rows_gemv(p, stream()), "table_rows");
  rc(jla::hy_rows_gemv(q, stream()), "table_rows");
  return true;
}

// p and q from row_linear: the tensors they were made from must be alive
void linear_rows_pair(const jla::RowLinear& p, const jla::RowLinear& q) {
  const long long a = jla::hy_linear_rows_floats(p), b = jla::hy_linear_rows_floats(q);
  Tensor ws;
  if (a > 0 || b > 0) ws = torch::empty({a > b ? a : b}, torch::TensorOptions().dtype(torch::kFloat32).device(torch::kCUDA));
  rc(jla::hy_linear_rows_pair(p, q, scratch_ptr(ws), stream()), "linear_rows_pair");
}

// whether a dense linear of `rows` rows with `n` output columns runs the GEMV (where an input norm can be fused)
bool dense_is_gemv(int64_t rows, int64_t n) {
  jla::RowLinear p{};
  p.R = rows; p.N = n; p.E = 1;
  return jla::hy_linear_rows_is_gemv(p);
}

// a dense linear of `rows` contiguous bf16 rows on `w`, for the questions below; false: there is none
static bool bf16_rows_linear(int64_t rows, const Tensor& w, int64_t act, jla::RowLinear& p) {
  if (w.dim() != 2 || !w.is_contiguous() || w.scalar_type() != at::kBFloat16) return false;
  if (act < jla::HY_ACT_NONE || act > jla::HY_ACT_GELU_GLU || rows < 0 || rows > 0x7fffffff) return false;
  const bool gated = jla::hy_act_gated(act);
  if (gated && w.size(0) % 2) return false;
  p.R = rows; p.N = gated ? w.size(0) / 2 : w.size(0); p.K = w.size(1); p.E = 1;
  p.lda = p.K; p.ldo = p.N; p.a_bf16 = p.wbf16 = 1; p.act = act;
  p.w = w.data_ptr(); p.w_stride = w.numel();
  return true;
}

// whether it is best rounded to bf16 for the large tiles (rows_gemm.hip)
bool rows_gemm_pays(int64_t rows, const Tensor& w, int64_t act) {
  jla::RowLinear p{};
  return bf16_rows_linear(rows, w, act, p) && jla::hy_rows_gemm_pays(p);
}

// whether it runs on the tiles for some ten to a few hundred rows (rows_mid.hip)
bool rows_mid_takes(int64_t rows, const Tensor& w, int64_t act) {
  jla::RowLinear p{};
  return bf16_rows_linear(rows, w, act, p) && jla::hy_rows_mid_takes(p);
}

// whether it runs on one of the kernels for few rows; w [E, N, K]: E of them, `rows` rows each, in one launch
bool rows_bf16_takes(int64_t rows, const Tensor& w, int64_t act) {
  jla::RowLinear p{};
  if (w.dim() == 3 && w.is_contiguous() && w.size(0) >= 1 && rows <= 0x7fffffff / w.size(0)) {
    if (!bf16_rows_linear(rows, w.select(0, 0), act, p)) return false;
    static const int32_t any = 0;
    p.offs = &any;  // (asked of, not read)
    p.E = w.size(0);
    p.even_rows = rows;
    p.R = rows * p.E;
    return jla::hy_rows_bf16_takes(p);
  }
  return bf16_rows_linear(rows, w, act, p) && jla::hy_rows_bf16_takes(p);
}

void route_table(Tensor ids, Tensor table, int64_t E, Tensor row_expert, Tensor row_tok, Tensor sort_tok, Tensor sort_dst,
                 Tensor offs) {
  check(table.dim() == 2, "route_table: table is [vocab, top]");
  const int M = ids.numel(), top = table.size(1);
  const int64_t R = (int64_t)M * top;
  rc(jla::hy_route_table(i32(ids, "ids", M), i32(table, "table", table.numel()), table.size(0), M, top, E,
                         i32w(row_expert, "row_expert", R), i32w(row_tok, "row_tok", R), i32w(sort_tok, "sort_tok", R),
                         i32w(sort_dst, "sort_dst", R), i32w(offs, "offs", E + 1), stream()),
     "route_table");
}

void route_topk(Tensor z, int64_t E, int64_t top, Tensor row_expert, Tensor row_tok, Tensor row_w, OptT sort_tok,
                OptT sort_dst, OptT sort_w, OptT offs) {
  check(z.dim() == 2 && z.size(1) >= E && top >= 1 && top <= E, "route_topk: z is [M, >= E], 1 <= top <= E");
  int ldz = 0;
  const float* zp = rows2d(z, "z", z.size(1), &ldz);
  const int M = z.size(0);
  const int64_t R = (int64_t)M * top;
  check(row_w.numel() >= R, "route_topk: weight outputs hold R numbers");
  const bool sorted = sort_tok.has_value();
  check(sorted == sort_dst.has_value() && sorted == sort_w.has_value() && sorted == offs.has_value(),
        "route_topk: the sorted outputs come together");
  check(!sorted || sort_w->numel() >= R, "route_topk: weight outputs hold R numbers");
  rc(jla::hy_route_topk(zp, ldz, M, top, E, i32w(row_expert, "row_expert", R), i32w(row_tok, "row_tok", R),
                        f32w(row_w, "row_w"), sorted ? i32w(*sort_tok, "sort_tok", R) : nullptr,
                        sorted ? i32w(*sort_dst, "sort_dst", R) : nullptr,
                        sorted ? f32w(*sort_w, "sort_w") : nullptr, sorted ? i32w(*offs, "offs", E + 1) : nullptr,
                        stream()),
     "route_topk");
}

void route_grouped(Tensor z, OptT correction, int64_t E, int64_t top, int64_t groups, int64_t keep, Tensor row_expert,
                   Tensor row_tok, Tensor row_w, OptT sort_tok, OptT sort_dst, OptT sort_w, OptT offs, bool sigmoid,
                   int64_t group_top, bool normalise, double w_scale, OptT z_bias) {
  check(z.dim() == 2 && z.size(1) >= E && top >= 1 && top <= E, "route_grouped: z is [M, >= E], 1 <= top <= E");
  int ldz = 0;
  const float* zp = rows2d(z, "z", z.size(1), &ldz);
  const int M = z.size(0);
  const int64_t R = (int64_t)M * top;
  check(row_w.numel() >= R, "route_grouped: weight outputs hold R numbers");
  check(!correction.has_value() || correction->numel() == E, "route_grouped: correction is [E]");
  check(!z_bias.has_value() || z_bias->numel() == E, "route_grouped: z_bias is [E]");
  const bool sorted = sort_tok.has_value();
  check(sorted == sort_dst.has_value() && sorted == sort_w.has_value() && sorted == offs.has_value(),
        "route_grouped: the sorted outputs come together");
  check(!sorted || sort_w->numel() >= R, "route_grouped: weight outputs hold R numbers");
  rc(jla::hy_route_grouped(zp, ldz, correction.has_value() ? f32(*correction, "correction") : nullptr, M, top, E,
                           jla::RouteRule{(int)groups, (int)keep, (int)group_top, sigmoid, normalise, (float)w_scale,
                                          z_bias.has_value() ? f32(*z_bias, "z_bias") : nullptr},
                           i32w(row_expert, "row_expert", R), i32w(row_tok, "row_tok", R), f32w(row_w, "row_w"),
                           sorted ? i32w(*sort_tok, "sort_tok", R) : nullptr,
                           sorted ? i32w(*sort_dst, "sort_dst", R) : nullptr, sorted ? f32w(*sort_w, "sort_w") : nullptr,
                           sorted ? i32w(*offs, "offs", E + 1) : nullptr, stream()),
     "route_grouped");
}

void hc_update(Tensor xs, OptT mix, OptT out_w, OptT y, int64_t nsum, OptT row_w, OptT row_expert, int64_t n_real,
               OptT ident, OptT extra, OptT next_in, OptT u) {
  jla::HyperUpdate p{};
  check(xs.dim() == 3, "hc_update: xs is [S, M, D]");
  p.S = xs.size(0); p.M = xs.size(1); p.D = xs.size(2);
  p.xs = f32w(xs, "xs");
  const int64_t md = (int64_t)p.M * p.D;
  check(mix.has_value() == out_w.has_value() && mix.has_value() == y.has_value(), "hc_update: mix, out_w and y together");
  if (mix.has_value()) {
    check(mix->numel() == (int64_t)p.S * p.S && out_w->numel() == p.S, "hc_update: mix is [S, S], out_w [S]");
    p.mix = f32(*mix, "mix");
    p.out_w = f32(*out_w, "out_w");
    check(nsum >= 1 && y->numel() == md * nsum, "hc_update: y is [M * nsum, D]");
    p.y = f32(*y, "y");
    p.nsum = nsum;
    const int64_t R = (int64_t)p.M * nsum;
    if (row_w.has_value()) {
      check(row_w->numel() >= R, "hc_update: row_w is [M * nsum]");
      p.row_w = f32(*row_w, "row_w");
    }
    if (row_expert.has_value()) {
      check(row_w.has_value() && ident.has_value() && ident->numel() == md, "hc_update: row_expert needs row_w and ident [M, D]");
      p.row_expert = i32(*row_expert, "row_expert", R);
      p.ident = f32(*ident, "ident");
      p.n_real = n_real;
    }
    if (extra.has_value()) {
      check(extra->numel() == md, "hc_update: extra is [M, D]");
      p.extra = f32(*extra, "extra");
    }
  }
  check(next_in.has_value() == u.has_value(), "hc_update: next_in and u together");
  if (next_in.has_value()) {
    check(next_in->numel() == p.S && u->numel() == md, "hc_update: next_in is [S], u [M, D]");
    p.next_in = f32(*next_in, "next_in");
    p.u = f32w(*u, "u");
  }
  rc(jla::hy_hc_update(p, stream()), "hc_update");
}

void norm_residual(Tensor y, int64_t nsum, double ysc, Tensor w, double eps, OptT x, OptT out, OptT extra,
                   OptT extra_gate, OptT rounded) {
  check(y.dim() == 2 && nsum >= 1 && y.size(0) % nsum == 0, "norm_residual: y is [M * nsum, D]");
  const int M = y.size(0) / nsum, D = y.size(1);
  check(w.numel() == 1 || w.numel() == D, "norm_residual: w has 1 or D elements");
  float* xp = nullptr;
  float* op = nullptr;
  if (x.has_value()) {
    check(x->numel() == (int64_t)M * D, "norm_residual: x shape");
    xp = f32w(*x, "x");
  }
  if (out.has_value()) {
    check(out->numel() == (int64_t)M * D, "norm_residual: out shape");
    op = f32w(*out, "out");
  }
  check(xp || op, "norm_residual: x or out");
  const float* ep = nullptr;
  const float* gp = nullptr;
  int ldg = 0;
  if (extra.has_value()) {
    check(extra->numel() == (int64_t)M * D, "norm_residual: extra shape");
    ep = f32(*extra, "extra");
  }
  if (extra_gate.has_value()) {
    check(ep && extra_gate->dim() == 2 && extra_gate->size(0) == M, "norm_residual: extra_gate is [M, 1] beside extra");
    gp = rows2d(*extra_gate, "extra_gate", 1, &ldg);
  }
  jla::bf16_t* rp = nullptr;
  if (rounded.has_value()) {
    gpu(*rounded, "rounded");
    check(rounded->scalar_type() == torch::kBFloat16 && rounded->is_contiguous() && rounded->numel() == (int64_t)M * D && D % 8 == 0,
          "norm_residual: rounded is bf16 [M, D], D a multiple of 8");
    rp = reinterpret_cast<jla::bf16_t*>(rounded->data_ptr());
  }
  rc(jla::hy_norm_residual(f32(y, "y"), nsum, (float)ysc, f32(w, "w"), w.numel() > 1 || D == 1, (float)eps, xp, op, M,
                           D, ep, gp, ldg, rp, stream()),
     "norm_residual");
}

void cast_bf16(Tensor x, Tensor y, int64_t act) {
  gpu(y, "y");
  check(y.scalar_type() == torch::kBFloat16 && y.numel() == x.numel() && x.numel() % 8 == 0, "cast_bf16 shapes");
  rc(jla::hy_cast_bf16(f32(x, "x"), reinterpret_cast<jla::bf16_t*>(y.data_ptr()), x.numel(), act, stream()), "cast_bf16");
}

void softcap(Tensor x, double cap) {
  rc(jla::hy_softcap(f32w(x, "x"), x.numel(), (float)cap, stream()), "softcap");
}

void gelu_gate_rows(Tensor gp, Tensor ids, Tensor table, int64_t col0, Tensor g) {
  const int wb = wtype(table, "table");
  check(gp.dim() == 2 && table.dim() == 2 && g.sizes() == gp.sizes(), "gelu_gate_rows shapes");
  const int M = gp.size(0), D = gp.size(1);
  rc(jla::hy_gelu_gate_rows(f32(gp, "gp"), i32(ids, "ids", M), table.data_ptr(), wb, table.size(0), table.size(1), col0,
                            f32w(g, "g"), M, D, stream()),
     "gelu_gate_rows");
}

void* slice2d_any(const Tensor& t, const char* name, int64_t rows, int64_t cols, int* ld, int* bf);
float* slice2d(const Tensor& t, const char* name, int64_t rows, int64_t cols, int* ld);

void glu_rows(Tensor gu, Tensor out, int64_t act, double limit, double alpha) {
  check(gu.dim() == 2 && out.dim() == 2 && gu.size(1) >= 2 * out.size(1) && jla::hy_act_gated(act),
        "glu_rows: gu is [M, >= 2F], out [M, F], a gated activation");
  int ldg = 0, ldo = 0, bf = 0;
  const float* gp = rows2d(gu, "gu", gu.size(1), &ldg);
  void* op = slice2d_any(out, "out", gu.size(0), out.size(1), &ldo, &bf);
  rc(jla::hy_glu_rows(gp, ldg, gu.size(0), out.size(1), act, limit, alpha, op, bf, ldo, stream()), "glu_rows");
}

// fp32 or bf16 dense [M, D] output
void* rows_out(const Tensor& h, const char* name, int64_t n, int* bf) {
  *bf = wtype(h, name);
  check(h.numel() == n, "an output row tensor has the wrong size");
  return h.data_ptr();
}

void squash_rows(Tensor x, Tensor alpha, Tensor w, Tensor b, Tensor h) {
  check(x.dim() == 2, "squash_rows: x is [M, D]");
  const int64_t M = x.size(0), D = x.size(1);
  check(alpha.numel() == 1 && w.numel() == D && b.numel() == D, "squash_rows: alpha is one number, w and b are [D]");
  int bf = 0;
  void* hp = rows_out(h, "h", M * D, &bf);
  rc(jla::hy_squash_rows(f32(x, "x"), M, D, f32(alpha, "alpha"), f32(w, "w"), f32(b, "b"), hp, bf, stream()),
     "squash_rows");
}

void depth_update(Tensor hist, int64_t i, bool store, Tensor x, Tensor x_out, double mult, Tensor y, OptT bias, OptT ye,
                  int64_t nsum, OptT row_w, Tensor coef, OptT alpha, OptT w, OptT b, OptT h) {
  jla::DepthUpdate p{};
  check(hist.dim() == 3 && i >= 0 && i + (store ? 1 : 0) < hist.size(0), "depth_update: hist is [planes, M, D], planes past i");
  p.M = hist.size(1); p.D = hist.size(2);
  const int64_t md = (int64_t)p.M * p.D;
  p.hist = f32w(hist, "hist");
  p.i = i; p.store = store;
  check(x.numel() == md && x_out.numel() == md && y.numel() == md, "depth_update: x, x_out and y are [M, D]");
  p.x = f32(x, "x");
  p.x_out = f32w(x_out, "x_out");
  p.mult = mult;
  p.y = f32(y, "y");
  if (bias.has_value()) {
    check(bias->numel() == p.D, "depth_update: bias is [D]");
    p.bias = f32(*bias, "bias");
  }
  if (ye.has_value()) {
    check(row_w.has_value() && nsum >= 1 && ye->numel() == md * nsum && row_w->numel() >= p.M * nsum,
          "depth_update: ye is [M * nsum, D], row_w [M * nsum]");
    p.ye = f32(*ye, "ye");
    p.row_w = f32(*row_w, "row_w");
    p.nsum = nsum;
  }
  check(coef.numel() == i + 2, "depth_update: coef is [i + 2]");
  p.coef = f32(coef, "coef");
  if (h.has_value()) {
    check(alpha.has_value() && w.has_value() && b.has_value() && alpha->numel() == 1 && w->numel() == p.D &&
              b->numel() == p.D,
          "depth_update: the norm's alpha is one number, w and b are [D]");
    p.alpha = f32(*alpha, "alpha");
    p.w = f32(*w, "w");
    p.b = f32(*b, "b");
    p.h = rows_out(*h, "h", md, &p.h_bf16);
  }
  rc(jla::hy_depth_update(p, stream()), "depth_update");
}

void sandwich_update(Tensor x, OptT y, int64_t nsum, OptT row_w, OptT bias, OptT extra, OptT post, double eps, OptT pre,
                     OptT h) {
  jla::SandwichUpdate p{};
  check(x.dim() == 2, "sandwich_update: x is [M, D]");
  p.M = x.size(0); p.D = x.size(1);
  const int64_t md = (int64_t)p.M * p.D;
  p.x = f32w(x, "x");
  p.eps = eps;
  p.nsum = nsum;
  if (y.has_value()) {
    check(nsum >= 1 && y->numel() == md * nsum, "sandwich_update: y is [M * nsum, D]");
    check(post.has_value() && post->numel() == p.D, "sandwich_update: post is [D]");
    p.y = f32(*y, "y");
    p.post = f32(*post, "post");
    if (row_w.has_value()) {
      check(row_w->numel() >= (int64_t)p.M * nsum, "sandwich_update: row_w is [M * nsum]");
      p.row_w = f32(*row_w, "row_w");
    }
    if (bias.has_value()) {
      check(bias->numel() == p.D, "sandwich_update: bias is [D]");
      p.bias = f32(*bias, "bias");
    }
    if (extra.has_value()) {
      check(extra->numel() == md, "sandwich_update: extra is [M, D]");
      p.extra = f32(*extra, "extra");
    }
  }
  check(pre.has_value() == h.has_value(), "sandwich_update: pre and h together");
  if (h.has_value()) {
    check(pre->numel() == p.D, "sandwich_update: pre is [D]");
    p.pre = f32(*pre, "pre");
    p.h = rows_out(*h, "h", md, &p.h_bf16);
  }
  rc(jla::hy_sandwich_update(p, stream()), "sandwich_update");
}

void attn_prep(Tensor proj, Tensor positions, Tensor slot, int64_t B, int64_t S, int64_t H, int64_t G, int64_t dim,
               int64_t vdim, OptT kc, OptT vc, Tensor q, double eps, double temp_coef, int64_t temp_every, OptT q_w, OptT k_w,
               bool norm_v) {
  jla::AttnPrep p{};
  p.norm_v = norm_v;
  if (q_w.has_value()) {
    check(q_w->numel() == dim, "attn_prep: q_w is [dim]");
    p.q_w = f32(*q_w, "q_w");
  }
  if (k_w.has_value()) {
    check(k_w->numel() == dim, "attn_prep: k_w is [dim]");
    p.k_w = f32(*k_w, "k_w");
  }
  p.has_kv = kc.has_value();
  check(kc.has_value() == vc.has_value(), "attn_prep: k and v caches together");
  const int64_t cols = H * dim + (p.has_kv ? G * (dim + vdim) : 0);
  check(proj.dim() == 2 && proj.size(0) == B * S, "attn_prep: proj rows");
  p.proj = rows2d(proj, "proj", cols, &p.ld);
  p.positions = i32(positions, "positions", B * S);
  p.slot = i32(slot, "slot", 1);
  p.B = B; p.S = S; p.H = H; p.G = G; p.dim = dim; p.vdim = vdim;
  p.T = 1;
  if (p.has_kv) {
    p.cbf16 = wtype(*kc, "k cache");
    check(wtype(*vc, "v cache") == p.cbf16, "attn_prep: cache dtypes differ");
    check(kc->dim() == 4 && kc->size(0) == B && kc->size(1) == G && kc->size(3) == dim, "attn_prep: k cache shape");
    p.T = kc->size(2);
    check(vc->dim() == 4 && vc->size(0) == B && vc->size(1) == G && vc->size(2) == p.T && vc->size(3) == vdim,
          "attn_prep: v cache shape");
    p.kc = kc->data_ptr();
    p.vc = vc->data_ptr();
  }
  check(q.numel() == B * S * H * dim, "attn_prep: q shape");
  p.q = f32w(q, "q");
  p.eps = eps;
  p.temp_coef = temp_coef;
  p.temp_every = temp_every;
  rc(jla::hy_attn_prep(p, stream()), "attn_prep");
}

const double* f64(const Tensor& t, const char* name);

void latent_prep(Tensor proj, int64_t col0, Tensor w, Tensor slot, int64_t B, int64_t S, Tensor cache, double eps,
                 OptT q, int64_t q_col0, OptT q_norm_w, OptT rot_freq, OptT positions, bool rot_halves) {
  jla::LatentPrep p{};
  p.rot_halves = rot_halves;
  check(proj.dim() == 2 && proj.size(0) == B * S && proj.scalar_type() == torch::kFloat32 && proj.is_cuda() &&
            proj.stride(1) == 1,
        "latent_prep: proj is a float32 [B * S, cols] GPU view with unit inner stride");
  p.proj = reinterpret_cast<const float*>(proj.data_ptr());
  p.ld = proj.stride(0);
  p.col0 = col0;
  p.cbf16 = wtype(cache, "latent cache");
  check(cache.dim() == 4 && cache.size(0) == B && cache.size(1) == 1, "latent_prep: cache is [B, 1, T, row]");
  p.T = cache.size(2);
  p.row = cache.size(3);
  p.rank = w.numel();
  check(col0 >= 0 && p.rank >= 1 && p.rank <= p.row && col0 + p.row <= proj.size(1), "latent_prep: latent columns / gain");
  if (rot_freq.has_value() && rot_freq->numel() > 0) {
    p.rot_half = rot_freq->numel();
    check(2 * p.rot_half <= p.row - p.rank && positions.has_value(), "latent_prep: rotated numbers / positions");
    p.rot_freq = f64(*rot_freq, "rot_freq");
    p.positions = i32(*positions, "positions", B * S);
  }
  p.w = f32(w, "w");
  p.slot = i32(slot, "slot", 1);
  p.B = B; p.S = S;
  p.cache = cache.data_ptr();
  p.eps = eps;
  if (q.has_value()) {
    check(q->dim() == 2 && q->size(0) == B * S && q_col0 >= 0 && q_col0 + q->size(1) <= proj.size(1),
          "latent_prep: q is [B * S, q_cols]");
    p.q = rows_out(*q, "q", q->numel(), &p.q_bf16);
    p.q_cols = q->size(1);
    p.q_col0 = q_col0;
    if (q_norm_w.has_value()) {
      check(q_norm_w->numel() == p.q_cols, "latent_prep: q_norm_w is [q_cols]");
      p.q_norm_w = f32(*q_norm_w, "q_norm_w");
    }
  }
  rc(jla::hy_latent_prep(p, stream()), "latent_prep");
}

int64_t attn_decode_splits(int64_t B, int64_t H, int64_t t_cap) { return jla::hy_attn_decode_splits(B, H, t_cap); }

int64_t attn_prefill_ws_bytes(int64_t B, int64_t S, int64_t G, int64_t dim, int64_t vdim, int64_t T, bool cbf16) {
  return jla::hy_attn_prefill_ws_bytes(B, S, G, dim, vdim, T, cbf16);
}

void attn_bias(Tensor q, Tensor kc, Tensor vc, Tensor slot, double scale, double softcap, OptT bias, Tensor out,
               int64_t t_cap, OptT ws, int64_t splits, OptT vt_ws, OptT sink, int64_t chunk, OptT head_scale, int64_t window,
               int64_t keep_first, OptT gate, c10::optional<int64_t> vdim, bool gate_cols, int64_t maps, double diff_lambda,
               double diff_eps, double diff_gain, OptT turn_pos, OptT turn_freq, double turn_sign, double turn_gain) {
  jla::AttnBias p{};
  check(maps == 1 || maps == 2, "attn_bias: one or two maps per head");
  check(q.dim() == 4 && q.size(2) % maps == 0, "attn_bias: q is [B, S, H * maps, dim]");
  p.B = q.size(0); p.S = q.size(1); p.H = q.size(2) / maps; p.dim = q.size(3);
  const int64_t qheads = q.size(2);
  p.maps = maps;
  p.ldk = maps * p.dim;
  p.diff_lambda = diff_lambda; p.diff_eps = diff_eps; p.diff_gain = diff_gain;
  p.q = f32(q, "q");
  p.cbf16 = wtype(kc, "k cache");
  check(wtype(vc, "v cache") == p.cbf16, "attn_bias: cache dtypes differ");
  check(kc.dim() == 4 && vc.dim() == 4 && kc.size(0) == p.B && vc.size(0) == p.B && kc.size(3) == p.ldk &&
            kc.size(1) == vc.size(1) && kc.size(2) == vc.size(2),
        "attn_bias: cache shapes");
  p.G = kc.size(1); p.T = kc.size(2);
  p.ldv = vc.size(3);
  p.vdim = vdim.has_value() ? *vdim : vc.size(3);
  check(p.vdim >= 1 && p.vdim <= p.ldv, "attn_bias: vdim is at most the width of a value row");
  check(window >= 0 && window <= INT32_MAX && keep_first >= 0 && keep_first <= INT32_MAX, "attn_bias: window / keep_first");
  p.window = window;
  p.keep_first = keep_first;
  if (gate.has_value()) {
    p.gate_cols = gate_cols;
    check(gate->dim() == 2 && gate->size(0) == (int64_t)p.B * p.S &&
              gate->size(1) >= (gate_cols ? (int64_t)p.H * p.vdim : (int64_t)p.H),
          "attn_bias: gate is [B * S, >= H], with gate_cols [B * S, >= H * vdim]");
    p.gate = rows2d(*gate, "gate", gate->size(1), &p.ldg);
  }
  p.kc = kc.data_ptr();
  p.vc = vc.data_ptr();
  p.slot = i32(slot, "slot", 1);
  p.scale = scale;
  p.softcap = softcap;
  if (bias.has_value()) {
    check(bias->dim() == 2 && bias->size(1) == qheads, "attn_bias: bias is [distances, query heads]");
    p.bias = f32(*bias, "bias");
    p.nbias = bias->size(0);
  }
  if (sink.has_value()) {
    check(sink->numel() == qheads, "attn_bias: one sink per query head");
    p.sink = f32(*sink, "sink");
  }
  check(chunk >= 0 && chunk <= INT32_MAX, "attn_bias: chunk");
  p.chunk = chunk;
  if (head_scale.has_value()) {
    check(head_scale->numel() == qheads, "attn_bias: one factor per query head");
    p.head_scale = f32(*head_scale, "head_scale");
  }
  p.out = slice2d_any(out, "out", (int64_t)p.B * p.S, (int64_t)p.H * p.vdim, &p.ldo, &p.out_bf16);
  p.t_cap = std::min<int64_t>(t_cap, p.T);
  p.splits = splits;
  if (p.S == 1) {
    check(ws.has_value() && splits >= 1 && ws->numel() >= (int64_t)p.B * qheads * splits * (p.vdim + 2),
          "attn_bias: decode workspace");
    p.ws = f32w(*ws, "ws");
  }
  if (vt_ws.has_value()) {
    gpu(*vt_ws, "vt_ws");
    check((int64_t)(vt_ws->numel() * vt_ws->element_size()) >=
              jla::hy_attn_prefill_ws_bytes(p.B, p.S, p.G, p.dim, p.vdim, p.T, p.cbf16),
          "attn_bias: transposed-value workspace too small");
    p.vt_ws = vt_ws->data_ptr();
  }
  if (turn_pos.has_value()) {
    check(p.S == 1 && maps == 1, "attn_bias: one query per row is turned");
    p.turn_pos = i32(*turn_pos, "turn_pos", p.B);
    if (turn_freq.has_value()) {
      check(2 * turn_freq->numel() <= p.vdim, "attn_bias: more rotated numbers than a head holds");
      p.turn_freq = f64(*turn_freq, "turn_freq");
      p.turn_half = turn_freq->numel();
    }
    p.turn_sign = turn_sign; p.turn_gain = turn_gain;
  }
  rc(jla::hy_attn_bias(p, stream()), "attn_bias");
}

// One token of an attention layer in one launch; false (nothing done) where its shapes are not the kernel's.
bool attn_step(Tensor proj, Tensor kc, Tensor vc, Tensor slot, Tensor positions, int64_t H, bool own, Tensor tickets, double scale,
               double softcap, OptT bias, Tensor out, int64_t seen, OptT sink, int64_t chunk, OptT head_scale, bool rope,
               double eps, double temp_coef, int64_t temp_every, OptT col_bias, OptT qk_freq, OptT v_freq, bool turn,
               double turn_sign, double turn_gain) {
  jla::AttnStep p{};
  jla::AttnBias& a = p.a;
  check(kc.dim() == 4 && vc.dim() == 4 && kc.size(0) == vc.size(0) && kc.size(1) == vc.size(1) && kc.size(2) == vc.size(2),
        "attn_step: cache shapes");
  a.cbf16 = wtype(kc, "k cache");
  check(wtype(vc, "v cache") == a.cbf16, "attn_step: cache dtypes differ");
  a.B = kc.size(0); a.G = kc.size(1); a.T = kc.size(2); a.dim = a.ldk = kc.size(3); a.vdim = a.ldv = vc.size(3);
  a.S = 1; a.H = H; a.maps = 1;
  check(H >= 1 && H % a.G == 0, "attn_step: heads");
  a.kc = kc.data_ptr();
  a.vc = vc.data_ptr();
  a.splits = jla::hy_attn_decode_splits(a.B, a.H, std::max<int64_t>(1, std::min<int64_t>(seen, a.T)));
  if (!jla::hy_attn_step_takes(p) || tickets.numel() < (int64_t)a.B * H * jla::AS_TICKET) return false;
  const int64_t cols = H * a.dim + (own ? (int64_t)a.G * (a.dim + a.vdim) : 0);
  check(proj.dim() == 2 && proj.size(0) == a.B, "attn_step: proj rows");
  p.proj = rows2d(proj, "proj", cols, &p.ld);
  p.own = own;
  p.positions = i32(positions, "positions", a.B);
  a.slot = i32(slot, "slot", 1);
  a.scale = scale;
  a.softcap = softcap;
  if (bias.has_value()) {
    check(bias->dim() == 2 && bias->size(1) == H, "attn_step: bias is [distances, heads]");
    a.bias = f32(*bias, "bias");
    a.nbias = bias->size(0);
  }
  if (sink.has_value()) {
    check(sink->numel() == H, "attn_step: one sink per head");
    a.sink = f32(*sink, "sink");
  }
  check(chunk >= 0 && chunk <= INT32_MAX, "attn_step: chunk");
  a.chunk = chunk;
  if (head_scale.has_value()) {
    check(head_scale->numel() == H, "attn_step: one factor per head");
    a.head_scale = f32(*head_scale, "head_scale");
  }
  a.out = slice2d_any(out, "out", a.B, (int64_t)H * a.vdim, &a.ldo, &a.out_bf16);
  p.rope = rope;
  p.eps = eps; p.temp_coef = temp_coef; p.temp_every = temp_every;
  if (col_bias.has_value()) {
    check(col_bias->numel() == H * a.dim + (int64_t)a.G * (a.dim + a.vdim), "attn_step: one bias per projection column");
    p.col_bias = f32(*col_bias, "col_bias");
  }
  if (qk_freq.has_value() && qk_freq->numel() > 0) {
    p.qk_half = qk_freq->numel();
    check(2 * p.qk_half <= a.dim, "attn_step: more rotated numbers than a head holds");
    p.qk_freq = f64(*qk_freq, "qk_freq");
  }
  if (v_freq.has_value() && v_freq->numel() > 0) {
    p.v_half = v_freq->numel();
    check(2 * p.v_half <= a.vdim, "attn_step: more rotated numbers than a value head holds");
    p.v_freq = f64(*v_freq, "v_freq");
  }
  p.turn = turn;
  p.turn_sign = turn_sign; p.turn_gain = turn_gain;
  p.tickets = i32w(tickets, "tickets", (int64_t)a.B * H * jla::AS_TICKET);
  const Tensor ws = torch::empty({(int64_t)a.B * H * a.splits * (a.vdim + 2)}, out.options().dtype(torch::kFloat32));
  a.ws = f32w(ws, "ws");
  rc(jla::hy_attn_step(p, stream()), "attn_step");
  return true;
}

jla::DeltaPrep delta_args(const Tensor& proj, int64_t B, int64_t S, int64_t H, int64_t G, int64_t dim, int64_t vdim,
                          const Tensor& conv_w, const Tensor& conv_state) {
  jla::DeltaPrep p{};
  const int64_t C = 2 * G * dim + H * vdim;
  check(proj.dim() == 2 && proj.size(0) == B * S, "delta: proj rows");
  p.proj = rows2d(proj, "proj", C + H * vdim + 2 * H, &p.ld);
  p.B = B; p.S = S; p.H = H; p.G = G; p.dim = dim; p.vdim = vdim;
  check(conv_w.dim() == 2 && conv_w.size(0) == C, "delta: conv_w is [channels, taps]");
  p.taps = conv_w.size(1);
  p.conv_w = f32(conv_w, "conv_w");
  check(conv_state.numel() == B * C * (p.taps - 1), "delta: conv_state is [B, channels, taps - 1]");
  p.conv_state = f32w(conv_state, "conv_state");
  return p;
}

void delta_prep(Tensor proj, int64_t B, int64_t S, int64_t H, int64_t G, int64_t dim, int64_t vdim, Tensor conv_w,
                Tensor conv_state, Tensor a_log, Tensor dt_bias, Tensor qn, Tensor kn, Tensor vcv, Tensor beta,
                Tensor decay) {
  jla::DeltaPrep p = delta_args(proj, B, S, H, G, dim, vdim, conv_w, conv_state);
  const int64_t M = B * S;
  check(a_log.numel() == H && dt_bias.numel() == H, "delta_prep: per-head constants");
  p.a_log = f32(a_log, "a_log");
  p.dt_bias = f32(dt_bias, "dt_bias");
  check(qn.numel() == M * G * dim && kn.numel() == M * G * dim && vcv.numel() == M * H * vdim &&
            beta.numel() == M * H && decay.numel() == M * H,
        "delta_prep: output shapes");
  p.qn = f32w(qn, "qn");
  p.kn = f32w(kn, "kn");
  p.vc = f32w(vcv, "v");
  p.beta = f32w(beta, "beta");
  p.decay = f32w(decay, "decay");
  rc(jla::hy_delta_prep(p, stream()), "delta_prep");
}

void conv_state_update(Tensor proj, int64_t B, int64_t S, int64_t H, int64_t G, int64_t dim, int64_t vdim, Tensor conv_w,
                       Tensor conv_state) {
  jla::DeltaPrep p = delta_args(proj, B, S, H, G, dim, vdim, conv_w, conv_state);
  rc(jla::hy_conv_state_update(p, stream()), "conv_state_update");
}

void delta_scan(Tensor qn, Tensor kn, Tensor v, Tensor beta, Tensor decay, Tensor state, Tensor o, int64_t B, int64_t S,
                int64_t H, int64_t G, int64_t dim, int64_t vdim) {
  jla::DeltaScan p{};
  const int64_t M = B * S;
  check(qn.numel() == M * G * dim && kn.numel() == M * G * dim && v.numel() == M * H * vdim && beta.numel() == M * H &&
            decay.numel() == M * H && o.numel() == M * H * vdim && state.numel() == B * H * dim * vdim,
        "delta_scan shapes");
  p.qn = f32(qn, "qn");
  p.kn = f32(kn, "kn");
  p.v = f32(v, "v");
  p.beta = f32(beta, "beta");
  p.decay = f32(decay, "decay");
  p.state = f32w(state, "state");
  p.o = f32w(o, "o");
  p.B = B; p.S = S; p.H = H; p.G = G; p.dim = dim; p.vdim = vdim;
  // a prompt whose rows the chunked form can read (16-byte rows) runs on the matrix cores, the rest token by token
  const long long floats = ((uintptr_t)p.qn | (uintptr_t)p.kn) & 15 ? 0 : jla::hy_delta_chunk_floats(p);
  if (floats > 0) {
    Tensor ws = torch::empty({floats}, qn.options());
    rc(jla::hy_delta_chunk(p, reinterpret_cast<float*>(ws.data_ptr()), stream()), "delta_scan");
    return;
  }
  rc(jla::hy_delta_scan(p, stream()), "delta_scan");
}

// a 2-d float32 view with unit inner stride whose rows hold at least `cols` numbers
float* slice2d(const Tensor& t, const char* name, int64_t rows, int64_t cols, int* ld) {
  TORCH_CHECK(t.is_cuda() && t.scalar_type() == torch::kFloat32 && t.dim() == 2 && t.stride(1) == 1 &&
                  t.size(0) == rows && t.size(1) == cols && (rows <= 1 || t.stride(0) >= cols),
              "jax_llama_amd._C_hybrid: ", name, " must be a float32 [", rows, ", ", cols,
              "] GPU view with unit inner stride");
  *ld = rows > 1 ? (int)t.stride(0) : (int)cols;
  return reinterpret_cast<float*>(t.data_ptr());
}

// the same, float32 or bfloat16 (*bf = 1)
void* slice2d_any(const Tensor& t, const char* name, int64_t rows, int64_t cols, int* ld, int* bf) {
  TORCH_CHECK(t.is_cuda() && (t.scalar_type() == torch::kFloat32 || t.scalar_type() == torch::kBFloat16) &&
                  t.dim() == 2 && (t.size(1) <= 1 || t.stride(1) == 1) && t.size(0) == rows && t.size(1) == cols &&
                  (rows <= 1 || t.stride(0) >= cols),
              "jax_llama_amd._C_hybrid: ", name, " must be a float32 / bfloat16 [", rows, ", ", cols,
              "] GPU view with unit inner stride");
  *ld = rows > 1 ? (int)t.stride(0) : (int)cols;
  *bf = t.scalar_type() == torch::kBFloat16;
  return t.data_ptr();
}

// a [M, H, n] float32 view whose heads are adjacent (stride(1) == n, unit inner stride): rows may be strided
const float* heads3d(const Tensor& t, const char* name, int64_t M, int64_t H, int64_t n, int* ld) {
  TORCH_CHECK(t.is_cuda() && t.scalar_type() == torch::kFloat32 && t.dim() == 3 && t.size(0) == M && t.size(1) == H &&
                  t.size(2) == n && t.stride(2) == 1 && (H == 1 || t.stride(1) == n) && (M <= 1 || t.stride(0) >= H * n),
              "jax_llama_amd._C_hybrid: ", name, " must be a float32 [", M, ", ", H, ", ", n,
              "] GPU view with adjacent heads");
  *ld = M > 1 ? (int)t.stride(0) : (int)(H * n);
  return reinterpret_cast<const float*>(t.data_ptr());
}

const double* f64(const Tensor& t, const char* name) {
  gpu(t, name);
  TORCH_CHECK(t.scalar_type() == torch::kFloat64, "jax_llama_amd._C_hybrid: ", name, " must be float64");
  return reinterpret_cast<const double*>(t.data_ptr());
}

void gated_rmsnorm(Tensor o, OptT gate, Tensor w, double eps, Tensor out, int64_t H, int64_t vdim, int64_t gate_act,
                   OptT denom_floor, double gain) {
  jla::GatedNorm p{};
  const int64_t ov = denom_floor.has_value() ? vdim + 1 : vdim;
  const int64_t M = o.numel() / (H * ov);
  check(o.numel() == M * H * ov && (w.numel() == vdim || w.numel() == H * vdim), "gated_rmsnorm shapes");
  check(gate.has_value() == (gate_act != 2), "gated_rmsnorm: gate_act 2 has no gate, the others need one");
  p.o = f32(o, "o");
  if (gate.has_value()) {
    check(gate->dim() == 2 && gate->size(0) == M, "gated_rmsnorm: gate rows");
    p.gate = rows2d(*gate, "gate", H * vdim, &p.ldg);
  }
  p.w = f32(w, "w");
  p.w_heads = w.numel() != vdim || H == 1;
  p.eps = eps;
  p.out = slice2d_any(out, "out", M, H * vdim, &p.ldo, &p.out_bf16);
  p.M = M; p.H = H; p.vdim = vdim;
  p.gate_act = gate_act;
  if (denom_floor.has_value()) {
    check(denom_floor->numel() == M * H, "gated_rmsnorm: denom_floor is [M, H]");
    p.denom_floor = f32(*denom_floor, "denom_floor");
  }
  p.gain = gain;
  rc(jla::hy_gated_rmsnorm(p, stream()), "gated_rmsnorm");
}

void rope_prep(Tensor proj, OptT bias, Tensor positions, Tensor slot, int64_t B, int64_t S, int64_t H, int64_t G,
               int64_t dim, int64_t vdim, Tensor kc, Tensor vc, Tensor q, Tensor qk_freq, OptT v_freq) {
  jla::RopePrep p{};
  const int64_t cols = (H + G) * dim + G * vdim;
  check(proj.dim() == 2 && proj.size(0) == B * S, "rope_prep: proj rows");
  p.proj = rows2d(proj, "proj", cols, &p.ld);
  if (bias.has_value()) {
    check(bias->numel() == cols, "rope_prep: one bias per projection column");
    p.bias = f32(*bias, "bias");
  }
  p.positions = i32(positions, "positions", B * S);
  p.slot = i32(slot, "slot", 1);
  p.B = B; p.S = S; p.H = H; p.G = G; p.dim = dim; p.vdim = vdim;
  p.cbf16 = wtype(kc, "k cache");
  check(wtype(vc, "v cache") == p.cbf16, "rope_prep: cache dtypes differ");
  check(kc.dim() == 4 && kc.size(0) == B && kc.size(1) == G && kc.size(3) == dim, "rope_prep: k cache shape");
  p.T = kc.size(2);
  check(vc.dim() == 4 && vc.size(0) == B && vc.size(1) == G && vc.size(2) == p.T && vc.size(3) == vdim,
        "rope_prep: v cache shape");
  p.kc = kc.data_ptr();
  p.vc = vc.data_ptr();
  check(q.numel() == B * S * H * dim, "rope_prep: q shape");
  p.q = f32w(q, "q");
  p.qk_half = qk_freq.numel();
  check(2 * p.qk_half <= dim, "rope_prep: more rotated numbers than a head holds");
  p.qk_freq = p.qk_half ? f64(qk_freq, "qk_freq") : nullptr;
  if (v_freq.has_value() && v_freq->numel() > 0) {
    p.v_half = v_freq->numel();
    check(2 * p.v_half <= vdim, "rope_prep: more rotated numbers than a value head holds");
    p.v_freq = f64(*v_freq, "v_freq");
  }
  rc(jla::hy_rope_prep(p, stream()), "rope_prep");
}

void qkv_prep(Tensor proj, OptT bias, OptT q_w, OptT k_w, double eps, Tensor positions, Tensor slot, int64_t B, int64_t S,
              int64_t H, int64_t G, int64_t dim, int64_t vdim, OptT kc, OptT vc, Tensor q, OptT freq, bool halves,
              OptT v_prev, OptT lambda, OptT v_out, int64_t maps, bool v_is_k, double rot_gain) {
  jla::QkvPrep p{};
  check(maps == 1 || maps == 2, "qkv_prep: one or two maps per head");
  check(kc.has_value() == vc.has_value(), "qkv_prep: k and v caches together");
  p.q_only = !kc.has_value();
  p.maps = maps;
  p.rot_gain = rot_gain;
  check(!v_is_k || (vdim == maps * dim && !p.q_only), "qkv_prep: values that are the keys have their width");
  const int64_t nq = H * maps * dim, nk = p.q_only ? 0 : G * maps * dim;
  const int64_t cols = nq + nk + (p.q_only || v_is_k ? 0 : G * vdim);
  p.v_col = v_is_k ? nq : nq + nk;
  check(proj.dim() == 2 && proj.size(0) == B * S && proj.size(1) >= cols, "qkv_prep: proj is [B * S, >= q | k | v columns]");
  p.proj = rows2d(proj, "proj", proj.size(1), &p.ld);
  if (bias.has_value()) {
    check(bias->numel() == cols, "qkv_prep: one bias per projection column");
    p.bias = f32(*bias, "bias");
  }
  if (q_w.has_value()) {
    check(q_w->numel() == nq, "qkv_prep: q_w has one gain per query column");
    p.q_w = f32(*q_w, "q_w");
  }
  if (k_w.has_value()) {
    check(k_w->numel() == nk, "qkv_prep: k_w has one gain per key column");
    p.k_w = f32(*k_w, "k_w");
  }
  p.eps = eps;
  p.positions = i32(positions, "positions", B * S);
  p.slot = i32(slot, "slot", 1);
  p.B = B; p.S = S; p.H = H; p.G = G; p.dim = dim; p.vdim = vdim;
  p.T = 1;
  if (!p.q_only) {
    p.cbf16 = wtype(*kc, "k cache");
    check(wtype(*vc, "v cache") == p.cbf16, "qkv_prep: cache dtypes differ");
    check(kc->dim() == 4 && kc->size(0) == B && kc->size(1) == G && kc->size(3) == maps * dim, "qkv_prep: k cache shape");
    p.T = kc->size(2);
    check(vc->dim() == 4 && vc->size(0) == B && vc->size(1) == G && vc->size(2) == p.T && vc->size(3) == vdim,
          "qkv_prep: v cache shape");
    p.kc = kc->data_ptr();
    p.vc = vc->data_ptr();
  }
  check(q.numel() == B * S * nq, "qkv_prep: q shape");
  p.q = f32w(q, "q");
  if (freq.has_value() && freq->numel() > 0) {
    p.half = freq->numel();
    check(2 * p.half <= dim, "qkv_prep: more rotated numbers than a head holds");
    p.freq = f64(*freq, "freq");
  }
  p.halves = halves;
  if (v_prev.has_value()) {
    check(v_prev->numel() == B * S * G * vdim && lambda.has_value() && lambda->numel() == 1,
          "qkv_prep: v_prev is [B * S, G * vdim], lambda one number");
    p.v_prev = f32(*v_prev, "v_prev");
    p.lambda = f32(*lambda, "lambda");
  }
  if (v_out.has_value()) {
    check(v_out->numel() == B * S * G * vdim, "qkv_prep: v_out is [B * S, G * vdim]");
    p.v_out = f32w(*v_out, "v_out");
  }
  rc(jla::hy_qkv_prep(p, stream()), "qkv_prep");
}

void rotate_heads(Tensor a, Tensor positions, OptT freq, int64_t H, double sign, double gain, Tensor out, int64_t offset,
                  bool interleaved) {
  check(a.dim() == 2 && a.size(1) % H == 0, "rotate_heads: a is [M, H * n]");
  const int64_t M = a.size(0), n = a.size(1) / H;
  int lda = 0, ldo = 0;
  const float* ap = slice2d(a, "a", M, H * n, &lda);
  int bf = 0;
  void* op = slice2d_any(out, "out", M, H * n, &ldo, &bf);
  const int half = freq.has_value() ? (int)freq->numel() : 0;
  check(offset >= 0 && offset + 2 * half <= n, "rotate_heads: more rotated numbers than a head holds");
  rc(jla::hy_rotate_heads(ap, lda, i32(positions, "positions", M), half ? f64(*freq, "freq") : nullptr, half, M, H, n,
                          (float)sign, (float)gain, op, bf, ldo, offset, interleaved, stream()),
     "rotate_heads");
}

void token_shift(Tensor h, Tensor prev, Tensor mu, Tensor out, int64_t B, int64_t S, OptT w, double eps) {
  check(mu.dim() == 2, "token_shift: mu is [n, D]");
  const int64_t n = mu.size(0), D = mu.size(1);
  check(!w.has_value() || w->numel() == D, "token_shift: w is [D]");
  check(h.numel() == B * S * D && prev.numel() == B * D && out.numel() == n * B * S * D, "token_shift shapes");
  const int bf = wtype(out, "out");
  check(out.is_contiguous(), "token_shift: out is contiguous");
  rc(jla::hy_token_shift(f32(h, "h"), f32w(prev, "prev"), f32(mu, "mu"), n, out.data_ptr(), bf, B, S, D,
                         w.has_value() ? f32(*w, "w") : nullptr, eps, stream()),
     "token_shift");
}

void mlstm_prep(Tensor proj, int64_t col_i, int64_t col_f, Tensor gate_bias, double cap, Tensor mstate, Tensor out,
                int64_t B, int64_t S, int64_t H) {
  jla::MlstmPrep p{};
  check(proj.dim() == 2 && proj.size(0) == B * S, "mlstm_prep: proj rows");
  p.proj = rows2d(proj, "proj", proj.size(1), &p.ld);
  check(col_i >= 0 && col_f >= 0 && col_i + H <= proj.size(1) && col_f + H <= proj.size(1), "mlstm_prep: gate columns");
  p.col_i = col_i; p.col_f = col_f;
  check(gate_bias.numel() == 2 * H && mstate.numel() == B * H && out.numel() == 3 * B * S * H, "mlstm_prep shapes");
  p.gate_bias = f32(gate_bias, "gate_bias");
  p.cap = cap;
  p.mstate = f32w(mstate, "mstate");
  float* o = f32w(out, "out");
  p.keep = o; p.write = o + B * S * H; p.floor = o + 2 * B * S * H;
  p.B = B; p.S = S; p.H = H;
  rc(jla::hy_mlstm_prep(p, stream()), "mlstm_prep");
}

void timemix_run(const jla::TimeMixChunk& t, const Tensor& like) {
  Tensor ws;  // scratch of this call, from the allocator of the stream that uses it
  const long long floats = jla::hy_timemix_chunk_floats(t);
  if (floats > 0) ws = torch::empty({floats}, like.options());
  rc(jla::hy_timemix_chunk(t, floats > 0 ? reinterpret_cast<float*>(ws.data_ptr()) : nullptr, stream()), "timemix_chunk");
}

// A prompt's time-mix memory with its gated head norm; false (nothing done) where the chunked kernel does not apply.
bool timemix_norm(Tensor r, Tensor k, Tensor v, Tensor pre, Tensor w0, Tensor u, Tensor state, int64_t B, int64_t S, Tensor gate, Tensor w,
                  double eps, double gain, Tensor out) {
  check(r.dim() == 3 && v.dim() == 3, "timemix_norm: r, k are [M, H, dim], v is [M, H, vdim]");
  const int64_t M = B * S, H = r.size(1), dim = r.size(2), vdim = v.size(2);
  jla::TimeMixChunk t{};
  jla::LinScan& p = t.s;
  p.mode = 1;
  p.q = heads3d(r, "r", M, H, dim, &p.ldq);
  p.k = heads3d(k, "k", M, H, dim, &p.ldk);
  p.v = heads3d(v, "v", M, H, vdim, &p.ldv);
  p.decay = heads3d(pre, "pre", M, H, dim, &p.ldd);
  check(w0.numel() == H * dim && u.numel() == H * dim, "timemix_norm: w0, u are [H, dim]");
  p.w0 = f32(w0, "w0");
  p.u = f32(u, "u");
  check(state.numel() == B * H * dim * vdim, "timemix_norm: state");
  p.state = f32w(state, "state");
  p.B = B; p.S = S; p.H = H; p.dim = dim; p.vdim = vdim;
  t.norm = 1;
  check(gate.dim() == 2 && gate.size(0) == M && (w.numel() == vdim || w.numel() == H * vdim), "timemix_norm: gate, w");
  t.gate = rows2d(gate, "gate", H * vdim, &t.ldg);
  t.w = f32(w, "w");
  t.w_heads = w.numel() != vdim || H == 1;
  t.eps = eps; t.gain = gain;
  t.out = slice2d_any(out, "out", M, H * vdim, &t.ldo, &t.out_bf16);
  if (M == 0 || !jla::hy_timemix_chunk_takes(t)) return false;
  timemix_run(t, r);
  return true;
}

void lin_scan(int64_t mode, Tensor q, Tensor k, Tensor v, Tensor decay, OptT write, OptT w0, OptT u, Tensor state,
              Tensor o, int64_t B, int64_t S, double q_scale, int64_t nseg, int64_t seg_len) {
  jla::LinScan p{};
  check(mode >= 0 && mode <= 2, "lin_scan: mode");
  check(q.dim() == 3 && v.dim() == 3, "lin_scan: q, k are [M, H, dim], v is [M, H, vdim]");
  const int64_t M = B * S, H = q.size(1), dim = q.size(2), vdim = v.size(2);
  const int64_t cols = mode == 0 ? vdim + 1 : vdim;
  p.mode = mode;
  p.q = heads3d(q, "q", M, H, dim, &p.ldq);
  p.k = heads3d(k, "k", M, H, dim, &p.ldk);
  p.v = heads3d(v, "v", M, H, vdim, &p.ldv);
  if (mode == 0) {
    check(decay.numel() == M * H && write.has_value() && write->numel() == M * H, "lin_scan: keep, write are [M, H]");
    p.decay = f32(decay, "keep");
    p.write = f32(*write, "write");
  } else {
    if (mode == 1) p.decay = heads3d(decay, "decay", M, H, dim, &p.ldd);
    check(w0.has_value() && u.has_value() && w0->numel() == H * dim && u->numel() == H * dim, "lin_scan: w0, u are [H, dim]");
    p.w0 = f32(*w0, "w0");
    p.u = f32(*u, "u");
  }
  check(state.numel() == B * H * dim * cols && o.numel() == M * H * cols, "lin_scan: state / output shapes");
  p.state = f32w(state, "state");
  p.o = f32w(o, "o");
  p.B = B; p.S = S; p.H = H; p.dim = dim; p.vdim = vdim;
  p.q_scale = q_scale;
  check(nseg >= 1 && seg_len >= 1 && nseg * seg_len >= S && (nseg - 1) * seg_len < S, "lin_scan: segments cover the tokens");
  jla::TimeMixChunk t{};
  t.s = p;
  if (jla::hy_timemix_chunk_takes(t)) return timemix_run(t, q);
  p.nseg = nseg;
  p.seg_len = seg_len;
  Tensor ws;  // scratch of this call, from the allocator of the stream that uses it
  const long long floats = jla::hy_scalar_chunk_floats(p);
  if (floats > 0) {  // (a prompt with scalar gates: chunks on the matrix cores)
    ws = torch::empty({floats}, q.options());
    rc(jla::hy_scalar_chunk(p, reinterpret_cast<float*>(ws.data_ptr()), stream()), "lin_scan");
    return;
  }
  if (nseg > 1) {  // each segment's own state and the product of its decays
    const int64_t ns = B * nseg * H * dim * cols, nd = B * nseg * H * (mode != 0 ? dim : 1);
    ws = torch::empty({ns + nd}, q.options());
    p.seg_state = reinterpret_cast<float*>(ws.data_ptr());
    p.seg_decay = p.seg_state + ns;
  }
  rc(jla::hy_lin_scan(p, stream()), "lin_scan");
}

bool rec_step_takes(int64_t dim, int64_t vdim) {
  return dim <= 0x7fffffff && vdim <= 0x7fffffff && jla::hy_rec_step_takes((int)dim, (int)vdim);
}

// gates: mode 0: (projection [B, .], column of the input gates, column of the forget gates, biases, running maximum [B, H])
void rec_step(int64_t mode, Tensor q, OptT k, Tensor v, OptT pre, OptT w0, OptT u, OptT beta, OptT decay, OptT proj, int64_t col_i,
              int64_t col_f, OptT gate_bias, double cap, OptT mstate, double q_scale, Tensor state, OptT gate, Tensor w,
              double eps, int64_t gate_act, double gain, Tensor out, OptT pre_x, OptT pre_w, OptT prev, OptT row) {
  jla::RecStep p{};
  check(mode >= 0 && mode <= 3, "rec_step: mode");
  check(q.dim() == 3 && v.dim() == 3, "rec_step: q is [B, H (mode 3: G), dim], v is [B, H, vdim]");
  const int64_t B = v.size(0), H = v.size(1), dim = q.size(2), vdim = v.size(2), G = q.size(1);
  check(rec_step_takes(dim, vdim), "rec_step: head sizes");
  check(mode == 3 ? (G >= 1 && H % G == 0) : G == H, "rec_step: heads");
  p.mode = mode; p.B = B; p.H = H; p.G = G; p.dim = dim; p.vdim = vdim;
  p.q = heads3d(q, "q", B, G, dim, &p.ldq);
  check(k.has_value() == (mode != 2), "rec_step: k");
  if (k.has_value()) p.k = heads3d(*k, "k", B, G, dim, &p.ldk);
  p.v = heads3d(v, "v", B, H, vdim, &p.ldv);
  if (mode == 0) {
    check(proj.has_value() && gate_bias.has_value() && mstate.has_value() && cap > 0, "rec_step: gates");
    check(proj->dim() == 2 && proj->size(0) == B && col_i >= 0 && col_f >= 0 && col_i + H <= proj->size(1) &&
              col_f + H <= proj->size(1), "rec_step: gate columns");
    const float* base = rows2d(*proj, "proj", proj->size(1), &p.ldgate);
    p.gate_i = base + col_i;
    p.gate_f = base + col_f;
    check(gate_bias->numel() == 2 * H && mstate->numel() == B * H, "rec_step: gate biases, running maximum");
    p.gate_bias = f32(*gate_bias, "gate_bias");
    p.mstate = f32w(*mstate, "mstate");
    p.cap = cap;
  } else if (mode == 3) {
    check(beta.has_value() && decay.has_value() && beta->numel() == B * H && decay->numel() == B * H, "rec_step: beta, decay");
    p.beta = f32(*beta, "beta");
    p.decay = f32(*decay, "decay");
  } else {
    check((pre.has_value() || (mode == 1 && pre_x.has_value())) && w0.has_value() && u.has_value() && w0->numel() == H * dim &&
              u->numel() == H * dim,
          "rec_step: pre, w0, u");
    if (pre_x.has_value()) {
      check(mode == 1 && !pre.has_value() && pre_w.has_value() && pre_w->dim() == 2 && pre_w->size(0) == H * dim &&
                pre_x->dim() == 2 && pre_x->size(0) == B && pre_x->size(1) == pre_w->size(1) && pre_w->size(1) % 4 == 0,
            "rec_step: low-rank gate product");
      p.pre_x = f32(*pre_x, "pre_x");
      p.pre_bf16 = wtype(*pre_w, "pre_w");
      p.pre_w = pre_w->data_ptr();
      p.rank = pre_w->size(1);
      check(((uintptr_t)p.pre_x & 15) == 0 && ((uintptr_t)p.pre_w & 15) == 0, "rec_step: alignment");
      check(prev.has_value() == row.has_value(), "rec_step: prev and row");
      if (row.has_value()) {
        check(prev->numel() == row->numel() && row->numel() % B == 0, "rec_step: prev and row are [B, width]");
        p.prev = f32w(*prev, "prev");
        p.row = f32(*row, "row");
        p.width = row->numel() / B;
      }
    } else {
      p.pre = heads3d(*pre, "pre", B, H, dim, &p.ldpre);
    }
    p.w0 = f32(*w0, "w0");
    p.u = f32(*u, "u");
  }
  p.q_scale = q_scale;
  check(state.numel() == B * H * dim * (mode == 0 ? vdim + 1 : vdim), "rec_step: state");
  p.state = f32w(state, "state");
  check(gate_act >= 0 && gate_act <= 2 && gate.has_value() == (gate_act != 2), "rec_step: gate");
  if (gate.has_value()) {
    check(gate->dim() == 2 && gate->size(0) == B, "rec_step: gate rows");
    p.gate = rows2d(*gate, "gate", H * vdim, &p.ldg);
  }
  check(w.numel() == vdim || w.numel() == H * vdim, "rec_step: norm gain");
  p.w = f32(w, "w");
  p.w_heads = w.numel() != vdim || H == 1;
  p.eps = eps; p.gate_act = gate_act; p.gain = gain;
  p.out = slice2d_any(out, "out", B, H * vdim, &p.ldo, &p.out_bf16);
  rc(jla::hy_rec_step(p, stream()), "rec_step");
}

// The delta rule of one token from its fused projection; false (nothing done) where its shapes are not the kernel's.
bool delta_step(Tensor proj, int64_t B, int64_t H, int64_t G, int64_t dim, int64_t vdim, Tensor conv_w, Tensor conv_state, Tensor a_log,
                Tensor dt_bias, Tensor tickets, Tensor state, Tensor w, double eps, Tensor out) {
  const jla::DeltaPrep d = delta_args(proj, B, 1, H, G, dim, vdim, conv_w, conv_state);
  if (d.taps != 4 || !rec_step_takes(dim, vdim) || G < 1 || H % G || B > 65535 || tickets.numel() < B * G * 4 * 32 ||
      ((uintptr_t)d.conv_w & 15) != 0)
    return false;
  jla::RecStep p{};
  p.mode = 4; p.B = B; p.H = H; p.G = G; p.dim = dim; p.vdim = vdim;
  p.proj = d.proj; p.ldproj = d.ld;
  p.conv_w = d.conv_w;
  p.conv_state = d.conv_state;
  check(a_log.numel() == H && dt_bias.numel() == H, "delta_step: per-head constants");
  p.a_log = f32(a_log, "a_log");
  p.dt_bias = f32(dt_bias, "dt_bias");
  p.tickets = i32w(tickets, "tickets", B * G * 4 * 32);
  check(state.numel() == B * H * dim * vdim, "delta_step: state");
  p.state = f32w(state, "state");
  p.gate = p.proj + 2 * G * dim + H * vdim;
  p.ldg = p.ldproj;
  check(w.numel() == vdim || w.numel() == H * vdim, "delta_step: norm gain");
  p.w = f32(w, "w");
  p.w_heads = w.numel() != vdim || H == 1;
  p.eps = eps; p.gate_act = 0; p.gain = 1.f;
  p.out = slice2d_any(out, "out", B, H * vdim, &p.ldo, &p.out_bf16);
  rc(jla::hy_rec_step(p, stream()), "delta_step");
  return true;
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.attr("GEMV_MAX_R") = jla::HY_GEMV_MAX_R;
  m.def("embed_rows", &embed_rows, py::arg("ids"), py::arg("table"), py::arg("col0"), py::arg("out"), py::arg("scale"),
        py::arg("copies") = 1, py::arg("norm") = py::none(), py::arg("eps") = 0.0);
  m.def("route_grouped", &route_grouped, py::arg("z"), py::arg("correction"), py::arg("E"), py::arg("top"),
        py::arg("groups"), py::arg("keep"), py::arg("row_expert"), py::arg("row_tok"), py::arg("row_w"),
        py::arg("sort_tok"), py::arg("sort_dst"), py::arg("sort_w"), py::arg("offs"), py::arg("sigmoid") = false,
        py::arg("group_top") = 1, py::arg("normalise") = false, py::arg("w_scale") = 1.0,
        py::arg("z_bias") = py::none());
  m.def("hc_update", &hc_update);
  m.def("linear_rows", &linear_rows, py::arg("a"), py::arg("a_idx"), py::arg("w"), py::arg("out"), py::arg("dst_idx"),
        py::arg("offs"), py::arg("row_expert"), py::arg("R"), py::arg("act"), py::arg("act_limit"), py::arg("act_alpha"),
        py::arg("a_scale"), py::arg("a_norm_w"), py::arg("a_norm_eps"), py::arg("even_rows") = 0,
        py::arg("add_out") = false);
  py::class_<jla::RowLinear>(m, "RowLinear");
  m.def("row_linear", &row_linear, py::arg("a"), py::arg("a_idx"), py::arg("w"), py::arg("out"), py::arg("dst_idx"),
        py::arg("offs"), py::arg("row_expert"), py::arg("R"), py::arg("act"), py::arg("act_limit"), py::arg("act_alpha"),
        py::arg("a_scale"), py::arg("a_norm_w"), py::arg("a_norm_eps"), py::arg("even_rows") = 0,
        py::arg("add_out") = false);
  m.def("linear_rows_pair", &linear_rows_pair);
  m.def("route_table", &route_table);
  m.def("route_topk", &route_topk);
  m.def("dense_is_gemv", &dense_is_gemv);
  m.def("rows_gemm_pays", &rows_gemm_pays);
  m.def("rows_mid_takes", &rows_mid_takes);
  m.def("rows_bf16_takes", &rows_bf16_takes);
  m.def("latent_prep", &latent_prep, py::arg("proj"), py::arg("col0"), py::arg("w"), py::arg("slot"), py::arg("B"),
        py::arg("S"), py::arg("cache"), py::arg("eps"), py::arg("q"), py::arg("q_col0") = 0,
        py::arg("q_norm_w") = py::none(), py::arg("rot_freq") = py::none(), py::arg("positions") = py::none(),
        py::arg("rot_halves") = false);
  m.attr("ACT_NONE") = (int)jla::HY_ACT_NONE;
  m.attr("ACT_RELU2") = (int)jla::HY_ACT_RELU2;
  m.attr("ACT_SWIGLU") = (int)jla::HY_ACT_SWIGLU;
  m.attr("ACT_CLAMP_GLU") = (int)jla::HY_ACT_CLAMP_GLU;
  m.def("norm_residual", &norm_residual, py::arg("y"), py::arg("nsum"), py::arg("ysc"), py::arg("w"), py::arg("eps"), py::arg("x"),
        py::arg("out"), py::arg("extra"), py::arg("extra_gate"), py::arg("rounded") = py::none());
  m.def("gelu_gate_rows", &gelu_gate_rows);
  m.def("cast_bf16", &cast_bf16, py::arg("x"), py::arg("y"), py::arg("act") = 0);
  m.def("softcap", &softcap);
  m.def("attn_prep", &attn_prep, py::arg("proj"), py::arg("positions"), py::arg("slot"), py::arg("B"), py::arg("S"),
        py::arg("H"), py::arg("G"), py::arg("dim"), py::arg("vdim"), py::arg("kc"), py::arg("vc"), py::arg("q"),
        py::arg("eps"), py::arg("temp_coef"), py::arg("temp_every"), py::arg("q_w") = py::none(),
        py::arg("k_w") = py::none(), py::arg("norm_v") = true);
  m.def("attn_decode_splits", &attn_decode_splits);
  m.def("attn_bias", &attn_bias, py::arg("q"), py::arg("kc"), py::arg("vc"), py::arg("slot"), py::arg("scale"),
        py::arg("softcap"), py::arg("bias"), py::arg("out"), py::arg("t_cap"), py::arg("ws"), py::arg("splits"),
        py::arg("vt_ws"), py::arg("sink"), py::arg("chunk") = 0, py::arg("head_scale") = py::none(),
        py::arg("window") = 0, py::arg("keep_first") = 0, py::arg("gate") = py::none(), py::arg("vdim") = py::none(),
        py::arg("gate_cols") = false, py::arg("maps") = 1, py::arg("diff_lambda") = 0.0, py::arg("diff_eps") = 0.0,
        py::arg("diff_gain") = 1.0, py::arg("turn_pos") = py::none(), py::arg("turn_freq") = py::none(),
        py::arg("turn_sign") = 1.0, py::arg("turn_gain") = 1.0);
  m.def("attn_step", &attn_step, py::arg("proj"), py::arg("kc"), py::arg("vc"), py::arg("slot"), py::arg("positions"), py::arg("H"),
        py::arg("own"), py::arg("tickets"), py::arg("scale"), py::arg("softcap"), py::arg("bias"), py::arg("out"), py::arg("seen"),
        py::arg("sink") = py::none(), py::arg("chunk") = 0, py::arg("head_scale") = py::none(), py::arg("rope") = false,
        py::arg("eps") = 0.0, py::arg("temp_coef") = 0.0, py::arg("temp_every") = 1, py::arg("col_bias") = py::none(),
        py::arg("qk_freq") = py::none(), py::arg("v_freq") = py::none(), py::arg("turn") = false, py::arg("turn_sign") = 1.0, py::arg("turn_gain") = 1.0);
  m.def("attn_prefill_ws_bytes", &attn_prefill_ws_bytes);
  m.def("timemix_norm", &timemix_norm);
  m.def("rows_parts", &rows_parts);
  m.def("rows_best", &rows_best);
  m.def("delta_step", &delta_step);
  m.def("delta_prep", &delta_prep);
  m.def("conv_state_update", &conv_state_update);
  m.def("delta_scan", &delta_scan);
  m.def("rows_fused", &rows_fused, py::arg("a"), py::arg("w"), py::arg("out"), py::arg("y"), py::arg("nsum"), py::arg("ysc"),
        py::arg("res_w"), py::arg("eps"), py::arg("x_out"), py::arg("ids") = py::none(), py::arg("table") = py::none(),
        py::arg("col0") = 0, py::arg("a_norm_w") = py::none(), py::arg("a_norm_eps") = 0.0, py::arg("act") = 0,
        py::arg("act_limit") = 0.0);
  m.def("table_rows", &table_rows);
  m.def("rec_step_takes", &rec_step_takes);
  m.def("rec_step", &rec_step, py::arg("mode"), py::arg("q"), py::arg("k"), py::arg("v"), py::arg("pre") = py::none(),
        py::arg("w0") = py::none(), py::arg("u") = py::none(), py::arg("beta") = py::none(), py::arg("decay") = py::none(),
        py::arg("proj") = py::none(), py::arg("col_i") = 0, py::arg("col_f") = 0, py::arg("gate_bias") = py::none(),
        py::arg("cap") = 1.0, py::arg("mstate") = py::none(), py::arg("q_scale") = 1.0, py::arg("state"), py::arg("gate"),
        py::arg("w"), py::arg("eps"), py::arg("gate_act"), py::arg("gain"), py::arg("out"), py::arg("pre_x") = py::none(),
        py::arg("pre_w") = py::none(), py::arg("prev") = py::none(), py::arg("row") = py::none());
  m.def("gated_rmsnorm", &gated_rmsnorm, py::arg("o"), py::arg("gate"), py::arg("w"), py::arg("eps"), py::arg("out"),
        py::arg("H"), py::arg("vdim"), py::arg("gate_act") = 0, py::arg("denom_floor") = py::none(),
        py::arg("gain") = 1.0);
  m.attr("ACT_SOFTCAP") = (int)jla::HY_ACT_SOFTCAP;
  m.def("rope_prep", &rope_prep);
  m.def("qkv_prep", &qkv_prep, py::arg("proj"), py::arg("bias"), py::arg("q_w"), py::arg("k_w"), py::arg("eps"),
        py::arg("positions"), py::arg("slot"), py::arg("B"), py::arg("S"), py::arg("H"), py::arg("G"), py::arg("dim"),
        py::arg("vdim"), py::arg("kc"), py::arg("vc"), py::arg("q"), py::arg("freq"), py::arg("halves") = false,
        py::arg("v_prev") = py::none(), py::arg("lambda_") = py::none(), py::arg("v_out") = py::none(),
        py::arg("maps") = 1, py::arg("v_is_k") = false, py::arg("rot_gain") = 1.0);
  m.def("sandwich_update", &sandwich_update);
  m.def("glu_rows", &glu_rows);
  m.def("squash_rows", &squash_rows);
  m.def("depth_update", &depth_update);
  m.def("rotate_heads", &rotate_heads, py::arg("a"), py::arg("positions"), py::arg("freq"), py::arg("H"), py::arg("sign"),
        py::arg("gain"), py::arg("out"), py::arg("offset") = 0, py::arg("interleaved") = false);
  m.def("token_shift", &token_shift, py::arg("h"), py::arg("prev"), py::arg("mu"), py::arg("out"), py::arg("B"), py::arg("S"),
        py::arg("w") = py::none(), py::arg("eps") = 0.0);
  m.def("mlstm_prep", &mlstm_prep);
  m.def("lin_scan", &lin_scan, py::arg("mode"), py::arg("q"), py::arg("k"), py::arg("v"), py::arg("decay"),
        py::arg("write"), py::arg("w0"), py::arg("u"), py::arg("state"), py::arg("o"), py::arg("B"), py::arg("S"),
        py::arg("q_scale"), py::arg("nseg") = 1, py::arg("seg_len") = (int64_t)1 << 40);
}
