// Native launchers of the torch ops: output allocation, argument blocks and the C-ABI calls of the ops whose
// Python bodies did the same through ctypes. A body's allocations, views and argument fields took 18 to
// 25 us of interpreter time a call (the forward 18.0, the backward 25.1), 7.9 and 10.8 here, and a small
// layer's step is paced by them. Dispatch, autograd and fake implementations stay with the Python ops, and
// so do checks of what a call may pass, except the sizes, types and devices of operands whose extent the
// kernel takes from another one: those are compared here. RuntimeError with the library's message
// when a call fails. Host code only; streams come as raw handles.
#include <torch/extension.h>

#include <string>
#include <tuple>

#include "../../include/mote_relation.h"

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;

[[noreturn]] void fail(int rc, const char* what) {
  throw std::runtime_error(std::string(what) + " failed (status " + std::to_string(rc) + "): " + mote_last_error());
}
void check(int rc, const char* what) {
  if (rc != MOTE_OK) fail(rc, what);
}

int code(at::ScalarType t) {
  if (t == at::kFloat) return MOTE_F32;
  if (t == at::kBFloat16) return MOTE_BF16;
  throw py::type_error(std::string("Relation kernels take float32 or bfloat16 tensors, got ") + c10::toString(t));
}
int code(const Tensor& t) { return code(t.scalar_type()); }

mote_view view(const Tensor& t) {
  TORCH_CHECK(t.dim() == 4 && t.stride(3) == 1, "last axis must be contiguous");
  return mote_view{t.data_ptr(), t.stride(0), t.stride(1), t.stride(2)};
}
float* fptr(const Tensor& t) { return static_cast<float*>(t.data_ptr()); }
int32_t* iptr(const Tensor& t) { return static_cast<int32_t*>(t.data_ptr()); }

Tensor empty(at::IntArrayRef sizes, const Tensor& like, at::ScalarType dt) {
  return at::empty(sizes, like.options().dtype(dt).memory_format(std::nullopt));
}
// [B, H, T, D] view over new [B, T, H, D] memory
Tensor heads(int64_t B, int64_t T, int64_t H, int64_t D, const Tensor& like, at::ScalarType dt) {
  return empty({B, T, H, D}, like, dt).transpose(1, 2);
}
Tensor bytes(size_t n, const Tensor& like) { return empty({int64_t(n < 16 ? 16 : n)}, like, at::kByte); }
// a small parameter as contiguous fp32 on the operands' device (itself when it is that already)
Tensor f32(const Tensor& t, const Tensor& like) { return t.detach().to(like.device(), at::kFloat).contiguous(); }

// unit stride on the last axis, strides of whole 16-byte chunks and an aligned base, else a copy
Tensor aligned(const Tensor& t) {
  const int64_t epc = 16 / t.element_size();
  bool ok = t.stride(-1) == 1 && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
  for (int64_t i = 0; i + 1 < t.dim(); ++i) ok = ok && t.stride(i) % epc == 0;
  return ok ? t : t.contiguous();
}
Tensor unit(const Tensor& t) { return t.stride(-1) == 1 ? t : t.contiguous(); }

std::tuple<Tensor, Tensor, Tensor, Tensor> relation_fwd(Tensor p1, Tensor p2, Tensor info, const Tensor& lam, double tau,
                                                        int64_t q_start, const OptTensor& cu, int64_t max_seqlen,
                                                        int64_t stream) {
  const bool varlen = cu.has_value();  // p1, p2, info are then [1, H, total, D]
  p1 = aligned(p1); p2 = aligned(p2); info = aligned(info);
  const int64_t B = p1.size(0), H = p1.size(1), TQ = p1.size(2), D = p1.size(3), TK = p2.size(2);
  const Tensor lam32 = lam.detach().to(at::kFloat).reshape({1}).contiguous();
  Tensor y = heads(B, TQ, H, D, p1, info.scalar_type());
  Tensor ibar = empty({B, H, TQ, D}, p1, at::kFloat), lse = empty({B, H, TQ}, p1, at::kFloat), g = empty({B, H, TQ}, p1, at::kFloat);
  mote_relation_fwd_args a{};
  a.dtype = code(p1);
  a.B = int(varlen ? cu->numel() - 1 : B); a.H = int(H); a.D = int(D);
  a.TQ = int(varlen ? max_seqlen : TQ); a.TK = int(varlen ? max_seqlen : TK); a.q_start = int(q_start);
  a.tau_s = float(tau);
  a.p1 = view(p1); a.p2 = view(p2); a.info = view(info); a.y = view(y);
  a.ibar = fptr(ibar); a.lse = fptr(lse); a.g = fptr(g); a.lam = fptr(lam32);
  if (varlen) {
    a.cu_seqlens = iptr(*cu);
    a.total_rows = int(TQ);
  }
  // scratch of the key-range pieces or the job counters; held until the launch is queued (the caching
  // allocator orders its reuse)
  Tensor ws;
  const size_t n = mote_relation_fwd_workspace(&a);
  if (n) {
    ws = bytes(n, p1);
    a.workspace = ws.data_ptr();
    a.workspace_bytes = n;
  }
  check(mote_relation_fwd(&a, reinterpret_cast<void*>(stream)), varlen ? "mote_relation_fwd (varlen)" : "mote_relation_fwd");
  return {y, g, ibar, lse};
}

std::tuple<Tensor, Tensor, Tensor, Tensor> relation_bwd(Tensor p1, Tensor p2, Tensor info, Tensor ibar, Tensor lse, Tensor g,
                                                        Tensor dy, double tau, int64_t q_start, bool deterministic,
                                                        int64_t stream) {
  p1 = aligned(p1); p2 = aligned(p2); info = aligned(info);
  dy = aligned(dy.to(p1.scalar_type()));
  ibar = ibar.contiguous(); lse = lse.contiguous(); g = g.contiguous();
  const int64_t B = p1.size(0), H = p1.size(1), TQ = p1.size(2), D = p1.size(3), TK = p2.size(2);
  Tensor dp1 = heads(B, TQ, H, D, p1, p1.scalar_type()), dp2 = heads(B, TK, H, D, p1, p2.scalar_type()),
         dinfo = heads(B, TK, H, D, p1, info.scalar_type()), dlam = empty({}, p1, at::kFloat);
  mote_relation_bwd_args a{};
  a.dtype = code(p1);
  a.B = int(B); a.H = int(H); a.TQ = int(TQ); a.TK = int(TK); a.D = int(D); a.q_start = int(q_start);
  a.tau_s = float(tau);
  a.deterministic = deterministic;
  a.p1 = view(p1); a.p2 = view(p2); a.info = view(info); a.dy = view(dy);
  a.ibar = fptr(ibar); a.lse = fptr(lse); a.g = fptr(g);
  a.dp1 = view(dp1); a.dp2 = view(dp2); a.dinfo = view(dinfo);
  a.dlam = fptr(dlam);
  // a step that leaves too little memory for the stored dU runs without it
  const size_t full = mote_relation_bwd_workspace(&a), least = mote_relation_bwd_workspace_min(&a);
  Tensor ws;
  try {
    ws = bytes(full, p1);
  } catch (const c10::OutOfMemoryError&) {
    if (least == full) throw;
    ws = bytes(least, p1);
  }
  a.workspace = ws.data_ptr();
  a.workspace_bytes = size_t(ws.numel());
  check(mote_relation_bwd(&a, reinterpret_cast<void*>(stream)), "mote_relation_bwd");
  return {dp1, dp2, dinfo, dlam};
}

std::tuple<Tensor, Tensor, Tensor> rope_givens(Tensor qkv, const OptTensor& inv_freq, const OptTensor& theta, int64_t H,
                                               int64_t parity, int64_t pos0, int64_t stream) {
  qkv = unit(qkv);
  const int64_t B = qkv.size(0), T = qkv.size(1), D = qkv.size(2) / (3 * H);
  Tensor p1 = heads(B, T, H, D, qkv, qkv.scalar_type()), p2 = heads(B, T, H, D, qkv, qkv.scalar_type()),
         info = heads(B, T, H, D, qkv, qkv.scalar_type());
  Tensor inv, th;
  if (inv_freq) inv = f32(*inv_freq, qkv);
  if (theta) th = f32(*theta, qkv);
  mote_rope_givens_args a{};
  a.dtype = code(qkv);
  a.B = int(B); a.T = int(T); a.H = int(H); a.D = int(D); a.pos0 = int(pos0); a.layer_parity = int(parity);
  a.inv_freq = inv_freq ? fptr(inv) : nullptr;
  a.theta = theta ? fptr(th) : nullptr;
  a.qkv = qkv.data_ptr(); a.qkv_sb = qkv.stride(0); a.qkv_sr = qkv.stride(1);
  a.p1 = view(p1); a.p2 = view(p2); a.info = view(info);
  check(mote_rope_givens_fwd(&a, reinterpret_cast<void*>(stream)), "mote_rope_givens_fwd");
  return {p1, p2, info};
}

std::tuple<Tensor, Tensor> rope_givens_bwd(const Tensor& dp1_, const Tensor& dp2_, const Tensor& dinfo_, Tensor qkv,
                                           const OptTensor& inv_freq, const OptTensor& theta, int64_t H, int64_t parity,
                                           int64_t pos0, bool info_only, int64_t stream) {
  const int64_t B = qkv.size(0), T = qkv.size(1), D = info_only ? qkv.size(2) / H : qkv.size(2) / (3 * H), D3 = 3 * H * D;
  qkv = unit(qkv);
  const at::ScalarType dt = qkv.scalar_type();
  auto grad = [&](const Tensor& t) { return t.stride(-1) == 1 ? t.to(dt) : t.to(dt).contiguous(); };
  const Tensor dp1 = grad(dp1_), dp2 = grad(dp2_), dinfo = grad(dinfo_);
  Tensor dqkv = empty({B, T, D3}, qkv, dt);
  // written whole by the kernel when theta is given
  Tensor dtheta = empty({H / 2 > 1 ? H / 2 : 1}, qkv, at::kFloat);
  if (!theta) dtheta.zero_();
  Tensor inv, th;
  if (inv_freq) inv = f32(*inv_freq, qkv);
  if (theta) th = f32(*theta, qkv);
  mote_rope_givens_bwd_args a{};
  a.dtype = code(qkv);
  a.B = int(B); a.T = int(T); a.H = int(H); a.D = int(D); a.pos0 = int(pos0); a.layer_parity = int(parity);
  a.inv_freq = inv_freq ? fptr(inv) : nullptr;
  a.theta = theta ? fptr(th) : nullptr;
  a.qkv = qkv.data_ptr(); a.qkv_sb = qkv.stride(0); a.qkv_sr = qkv.stride(1);
  a.qkv_info_only = info_only;
  a.dp1 = view(dp1); a.dp2 = view(dp2); a.dinfo = view(dinfo);
  a.dqkv = dqkv.data_ptr(); a.dqkv_sb = dqkv.stride(0); a.dqkv_sr = dqkv.stride(1);
  a.dtheta = fptr(dtheta);
  const Tensor ws = bytes(mote_rope_givens_bwd_workspace(&a), qkv);
  a.workspace = ws.data_ptr();
  a.workspace_bytes = size_t(ws.numel());
  check(mote_rope_givens_bwd(&a, reinterpret_cast<void*>(stream)), "mote_rope_givens_bwd");
  return {dqkv, dtheta};
}

Tensor linear_wgrad(Tensor a_, Tensor x, at::ScalarType dtype, int64_t stream) {
  TORCH_CHECK(a_.dim() == 2 && x.dim() == 2 && a_.size(0) == x.size(0) && a_.scalar_type() == x.scalar_type() &&
                  a_.device() == x.device(),
              "linear_wgrad: a [M, N] and x [M, K] of one dtype and device, got ", a_.sizes(), " ", a_.scalar_type(), " and ",
              x.sizes(), " ", x.scalar_type());
  // rows the kernel can walk: apart (an expanded gradient has stride 0), within its 32-bit offsets, aligned
  auto rows = [](const Tensor& t) {
    const int64_t sr = t.stride(0);
    const bool ok = t.stride(1) == 1 && sr >= t.size(1) && sr < (int64_t(1) << 24) && sr % 8 == 0 &&
                    reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
    return ok ? t : t.clone(at::MemoryFormat::Contiguous);  // (contiguous() keeps a contiguous tensor off a boundary)
  };
  a_ = rows(a_);
  x = rows(x);
  Tensor dw = empty({a_.size(1), x.size(1)}, a_, dtype);
  mote_linear_wgrad_args a{};
  a.dtype = code(a_); a.dw_dtype = code(dw);
  a.M = int(a_.size(0)); a.N = int(a_.size(1)); a.K = int(x.size(1));
  a.a = a_.data_ptr(); a.a_sr = a_.stride(0);
  a.x = x.data_ptr(); a.x_sr = x.stride(0);
  a.dw = dw.data_ptr(); a.dw_sr = dw.stride(0);
  const Tensor ws = bytes(mote_linear_wgrad_workspace(&a), a_);
  a.workspace = ws.data_ptr();
  a.workspace_bytes = size_t(ws.numel());
  check(mote_linear_wgrad(&a, reinterpret_cast<void*>(stream)), "mote_linear_wgrad");
  return dw;
}

// [..., D] -> [rows, D] with unit element stride (a view when possible)
Tensor rows2d(const Tensor& t_) { return unit(t_).reshape({-1, t_.size(-1)}); }

// (y, s or an empty stand-in when s is x itself, rstd); s_dtype: the summed stream's type
std::tuple<Tensor, Tensor, Tensor> add_rms_norm(const Tensor& x, const Tensor& weight, const OptTensor& residual, double eps,
                                                at::ScalarType s_dtype, int64_t stream) {
  const int64_t D = x.size(-1);
  const Tensor x2 = rows2d(x), w = f32(weight, x);
  const int64_t rows = x2.size(0);
  Tensor r2;
  if (residual) r2 = rows2d(*residual);
  Tensor y = empty(x.sizes(), x, x.scalar_type());
  const bool sum = residual.has_value() || s_dtype != x.scalar_type();
  Tensor s = sum ? empty(x.sizes(), x, s_dtype) : empty({0}, x, x.scalar_type());
  Tensor rstd = empty({rows}, x, at::kFloat);
  mote_add_rms_norm_args a{};
  a.dtype = code(x2); a.out_dtype = code(y);
  a.res_dtype = residual ? code(r2) : a.dtype;
  a.res_out_dtype = sum ? code(s) : a.dtype;
  a.rows = int(rows); a.D = int(D); a.eps = float(eps);
  a.x = x2.data_ptr(); a.x_sr = x2.stride(0);
  if (residual) {
    a.residual = r2.data_ptr();
    a.res_sr = r2.stride(0);
  }
  a.weight = fptr(w);
  a.y = y.data_ptr(); a.y_sr = D;
  if (sum) {
    a.residual_out = s.data_ptr();
    a.res_out_sr = D;
  }
  a.rstd = fptr(rstd);
  check(mote_add_rms_norm_fwd(&a, reinterpret_cast<void*>(stream)), "mote_add_rms_norm_fwd");
  return {y, s, rstd};
}

std::tuple<Tensor, Tensor, Tensor> add_rms_norm_bwd(const Tensor& dy, const OptTensor& dres_out, const Tensor& s, const Tensor& rstd,
                                                    const Tensor& weight, at::ScalarType x_dtype, bool has_res,
                                                    at::ScalarType res_dtype, int64_t stream) {
  const int64_t D = s.size(-1);
  const Tensor dy2 = rows2d(dy), s2 = rows2d(s), w = f32(weight, s);
  Tensor dro2;
  if (dres_out) dro2 = rows2d(*dres_out);
  Tensor dx = empty(s.sizes(), s, x_dtype);
  Tensor dres = has_res ? empty(s.sizes(), s, res_dtype) : empty({0}, s, res_dtype);
  Tensor dw = empty({D}, s, at::kFloat);
  mote_add_rms_norm_bwd_args a{};
  a.dtype = code(dy2); a.s_dtype = code(s2); a.dx_dtype = code(dx);
  a.dres_out_dtype = dres_out ? code(dro2) : a.dtype;
  a.dres_dtype = has_res ? code(dres) : a.dtype;
  a.rows = int(s2.size(0)); a.D = int(D);
  a.dy = dy2.data_ptr(); a.dy_sr = dy2.stride(0);
  if (dres_out) {
    a.dres_out = dro2.data_ptr();
    a.dres_out_sr = dro2.stride(0);
  }
  a.s = s2.data_ptr(); a.s_sr = s2.stride(0);
  a.rstd = fptr(rstd); a.weight = fptr(w);
  a.dx = dx.data_ptr(); a.dx_sr = D;
  if (has_res) {
    a.dresidual = dres.data_ptr();
    a.dres_sr = D;
  }
  a.dweight = fptr(dw);
  const Tensor ws = bytes(mote_add_rms_norm_bwd_workspace(&a), s);
  a.workspace = ws.data_ptr();
  a.workspace_bytes = size_t(ws.numel());
  check(mote_add_rms_norm_bwd(&a, reinterpret_cast<void*>(stream)), "mote_add_rms_norm_bwd");
  return {dx, dres, dw};
}

// The fused prologue; ws: the stacked weight, or the three (p1, p2, I~ projections); p2 / info: views to
// write instead of new tensors. The kernel reads its operands at the sizes that x and H give: they are checked
// against those here (a longer stack, frequency or angle tensor is read at its start). The cos / sin table (memoised by the caller) comes as `table`.
std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor> qkv_rope(const Tensor& x, const std::vector<Tensor>& ws, const OptTensor& inv_freq,
                                                            const OptTensor& theta, int64_t H, int64_t parity, int64_t pos0,
                                                            bool keep_info, const OptTensor& norm_w1, const OptTensor& norm_w2,
                                                            double eps, const Tensor& table, bool table_ready, const OptTensor& p2_,
                                                            const OptTensor& info_, int64_t stream) {
  const int64_t B = x.size(0), T = x.size(1), K = x.size(2), D = K / H;
  const at::ScalarType dt = x.scalar_type();
  TORCH_CHECK(dt == at::kBFloat16 && K == H * D && x.is_contiguous(), "qkv_rope: x must be bf16 of ", H, " heads, got ", dt, " rows of ", K);
  for (const Tensor& w : ws)
    TORCH_CHECK(w.dim() == 2 && (ws.size() == 3 ? w.size(0) == K : w.size(0) >= 3 * K) && w.size(1) == K &&
                    w.scalar_type() == dt && w.device() == x.device() && w.is_contiguous(),
                "qkv_rope: weights must be contiguous bf16 [", K, ", ", K, "] each or [", 3 * K, ", ", K, "] stacked, on x's device");
  TORCH_CHECK(!inv_freq || inv_freq->numel() >= D / 2, "qkv_rope: inv_freq needs ", D / 2, " values");
  TORCH_CHECK(!theta || theta->numel() >= H / 2, "qkv_rope: theta needs ", H / 2, " values");
  for (const OptTensor* t : {&p2_, &info_})  // the caller's memory: the kernel writes all of [B, H, T, D]
    TORCH_CHECK(!t->has_value() || ((*t)->sizes() == at::IntArrayRef({B, H, T, D}) && (*t)->scalar_type() == dt &&
                                    (*t)->device() == x.device()),
                "qkv_rope: P2 and I~ must be [", B, ", ", H, ", ", T, ", ", D, "] in x's dtype on x's device");
  Tensor p1 = heads(B, T, H, D, x, dt);
  Tensor p2 = p2_ ? *p2_ : heads(B, T, H, D, x, dt), info = info_ ? *info_ : heads(B, T, H, D, x, dt);
  const bool norm = norm_w1.has_value();
  Tensor iraw = keep_info ? empty({B, T, K}, x, dt) : empty({0}, x, dt);
  Tensor qkraw = keep_info && norm ? empty({B, T, 2 * K}, x, dt) : empty({0}, x, dt);
  mote_qkv_rope_args a{};
  a.B = int(B); a.T = int(T); a.H = int(H); a.D = int(D); a.pos0 = int(pos0); a.layer_parity = int(parity);
  a.x = x.data_ptr(); a.x_sb = T * K; a.x_sr = K;  // contiguous (the strides of axes of one element may be any)
  a.w = ws[0].data_ptr(); a.w_sr = K;
  Tensor inv, th, n1, n2;
  if (inv_freq) {
    inv = f32(*inv_freq, x);
    a.inv_freq = fptr(inv);
  }
  if (theta) {
    th = f32(*theta, x);
    a.theta = fptr(th);
  }
  a.p1 = view(p1); a.p2 = view(p2); a.info = view(info);
  if (keep_info) {
    a.info_raw = iraw.data_ptr(); a.ir_sb = iraw.stride(0); a.ir_sr = iraw.stride(1);
  }
  if (norm) {
    n1 = f32(*norm_w1, x);
    n2 = f32(*norm_w2, x);
    a.norm_w1 = fptr(n1); a.norm_w2 = fptr(n2); a.norm_eps = float(eps);
    if (keep_info) {
      a.qk_raw = qkraw.data_ptr(); a.qr_sb = qkraw.stride(0); a.qr_sr = qkraw.stride(1);
    }
  }
  a.workspace = table.data_ptr(); a.workspace_bytes = size_t(table.numel()); a.table_ready = table_ready;
  void* st = reinterpret_cast<void*>(stream);
  if (ws.size() == 3) check(mote_qkv_rope_parts_fwd(&a, ws[1].data_ptr(), ws[2].data_ptr(), st), "mote_qkv_rope_parts_fwd");
  else check(mote_qkv_rope_fwd(&a, st), "mote_qkv_rope_fwd");
  return {p1, p2, info, iraw, qkraw};
}

std::tuple<Tensor, Tensor, Tensor, Tensor> chunk_route(const Tensor& m, int64_t stream) {
  const int64_t B = m.size(0), L = m.size(1);
  Tensor cum = empty({B, L}, m, at::kInt), perm = empty({B, L}, m, at::kInt), num = empty({B}, m, at::kInt),
         cu = empty({B + 1}, m, at::kInt);
  mote_chunk_route_args a{};
  a.B = int(B); a.L = int(L);
  a.mask = static_cast<const uint8_t*>(m.data_ptr()); a.mask_sr = m.stride(0);
  a.cum = iptr(cum); a.perm = iptr(perm); a.num = iptr(num); a.cu_seqlens = iptr(cu);
  if (B == 0) cu.zero_();
  check(mote_chunk_route(&a, reinterpret_cast<void*>(stream)), "mote_chunk_route");
  return {cum, perm, num, cu};
}

std::tuple<Tensor, Tensor> dechunk(const Tensor& h, const Tensor& pr, const Tensor& perm, const Tensor& num, const Tensor& cum,
                                   int64_t L, double eps, const OptTensor& init, int64_t stream) {
  const int64_t B = h.size(0), M = h.size(1), D = h.size(2);
  Tensor out = empty({B, L, D}, h, h.scalar_type()), w = empty({B, M, D}, h, at::kFloat), ini;
  if (init) ini = f32(*init, h);
  mote_dechunk_args a{};
  a.dtype = code(h); a.prob_dtype = code(pr); a.out_dtype = a.dtype;
  a.B = int(B); a.L = int(L); a.M = int(M); a.D = int(D); a.eps = float(eps);
  a.hidden = h.data_ptr(); a.h_sb = h.stride(0); a.h_sr = h.stride(1);
  a.prob = pr.data_ptr(); a.p_sb = pr.stride(0); a.p_sr = pr.stride(1);
  a.perm = iptr(perm); a.num = iptr(num); a.cum = iptr(cum);
  a.init = init ? fptr(ini) : nullptr;
  a.out = out.data_ptr(); a.o_sb = out.stride(0); a.o_sr = out.stride(1);
  a.w = fptr(w);
  const Tensor ws = bytes(mote_dechunk_workspace(&a), h);
  a.workspace = ws.data_ptr();
  a.workspace_bytes = size_t(ws.numel());
  check(mote_dechunk_fwd(&a, reinterpret_cast<void*>(stream)), "mote_dechunk_fwd");
  return {out, w};
}

std::tuple<Tensor, Tensor> dechunk_bwd(const Tensor& g, const Tensor& h, const Tensor& pr, const Tensor& perm, const Tensor& num,
                                       const Tensor& m, const Tensor& cum, const Tensor& w, double eps, int64_t stream) {
  const int64_t B = h.size(0), M = h.size(1), D = h.size(2), L = g.size(1);
  Tensor dh = empty({B, M, D}, h, h.scalar_type()), dp = empty({B, L, 2}, h, pr.scalar_type());
  mote_dechunk_bwd_args a{};
  a.dtype = code(h); a.prob_dtype = code(pr); a.dout_dtype = code(g); a.dx_dtype = code(dh); a.dprob_dtype = code(dp);
  a.B = int(B); a.L = int(L); a.M = int(M); a.D = int(D); a.eps = float(eps);
  a.dout = g.data_ptr(); a.g_sb = g.stride(0); a.g_sr = g.stride(1);
  a.hidden = h.data_ptr(); a.h_sb = h.stride(0); a.h_sr = h.stride(1);
  a.prob = pr.data_ptr(); a.p_sb = pr.stride(0); a.p_sr = pr.stride(1);
  a.perm = iptr(perm); a.num = iptr(num);
  a.mask = static_cast<const uint8_t*>(m.data_ptr()); a.mask_sr = m.stride(0);
  a.cum = iptr(cum); a.w = fptr(w);
  a.dhidden = dh.data_ptr(); a.dh_sb = dh.stride(0); a.dh_sr = dh.stride(1);
  a.dprob = dp.data_ptr(); a.dp_sb = dp.stride(0); a.dp_sr = dp.stride(1);
  const Tensor ws = bytes(mote_dechunk_bwd_workspace(&a), h);
  a.workspace = ws.data_ptr();
  a.workspace_bytes = size_t(ws.numel());
  check(mote_dechunk_bwd(&a, reinterpret_cast<void*>(stream)), "mote_dechunk_bwd");
  return {dh, dp};
}

}  // namespace

PYBIND11_MODULE(_torch_launch, m) {
  // the interpreter lock is free while a call allocates and launches, as it was during the ctypes calls
  using nogil = py::call_guard<py::gil_scoped_release>;
  m.def("relation_fwd", &relation_fwd, nogil());
  m.def("relation_bwd", &relation_bwd, nogil());
  m.def("rope_givens", &rope_givens, nogil());
  m.def("rope_givens_bwd", &rope_givens_bwd, nogil());
  m.def("linear_wgrad", &linear_wgrad, nogil());
  m.def("add_rms_norm", &add_rms_norm, nogil());
  m.def("add_rms_norm_bwd", &add_rms_norm_bwd, nogil());
  m.def("qkv_rope", &qkv_rope, nogil());
  m.def("chunk_route", &chunk_route, nogil());
  m.def("dechunk", &dechunk, nogil());
  m.def("dechunk_bwd", &dechunk_bwd, nogil());
}
