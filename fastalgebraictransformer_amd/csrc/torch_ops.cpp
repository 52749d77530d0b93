// The autograd entry points of the package as native torch autograd functions
// over the C ABI (kat.h): the module _katops.
//
// A fwd + bwd pass of a small op through torch.autograd.Function spends its
// time in Python: the backward runs in autograd's device thread, which takes
// the GIL and builds its ctypes calls there (softmax fwd + bwd 44 us of host
// time a pass with both threads on one core complex, 88 us otherwise, against
// 37 us of GPU time at 4096 x 4096 bf16). Here the backward runs without the
// GIL; the launches, their arguments and the results are the same.
//
// Every function takes the common case only -- plain strided CUDA (HIP)
// tensors of one dtype in the layouts the kernels read -- and returns None for
// anything else (tensor subclasses, functorch transforms, tracing, dispatch
// modes, empty inputs, mixed dtypes, wrong shapes, attention outside the MFMA
// kernels' envelope): the Python functions then run the torch.autograd.Function
// classes, which convert, warn and raise as they do. What a backward gets (from
// autograd, or from saved-tensor hooks, which may return other layouts) is
// examined again there.

#include <ATen/ATen.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/extension.h>

#include <initializer_list>
#include <optional>
#include <stdexcept>
#include <string>
#include <tuple>

#include "kat.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::Function;
using torch::autograd::variable_list;

int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return KAT_F32;
    case at::kBFloat16: return KAT_BF16;
    case at::kHalf: return KAT_F16;
    case at::kDouble: return KAT_F64;
    default: return -1;
  }
}
int code(const Tensor& t) { return dtype_code(t.scalar_type()); }

// a strided device tensor whose data the kernels may read: no subclass,
// wrapper of a transform, or lazily materialised tensor
bool plain(const Tensor& t) {
  constexpr c10::DispatchKeySet odd{c10::DispatchKey::Python,           c10::DispatchKey::PythonTLSSnapshot,
                                    c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                    c10::DispatchKey::Functionalize,    c10::DispatchKey::ZeroTensor,
                                    c10::DispatchKey::Conjugate,        c10::DispatchKey::Negative};
  return t.defined() && t.is_cuda() && t.layout() == at::kStrided && !t.key_set().has_any(odd) && code(t) >= 0;
}

// no transform, dispatch mode or tracer sees this call
bool untraced() {
  return !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) &&
         !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::Python) &&
         !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::Functionalize) &&
         !torch::jit::tracer::isTracing();
}

bool same_place(const Tensor& a, std::initializer_list<const Tensor*> ts) {
  for (const Tensor* t : ts)
    if (!plain(*t) || t->device() != a.device()) return false;
  return true;
}

void check(int rc, const char* name) {
  if (rc != 0)
    throw std::runtime_error(std::string(name) + " failed (status " + std::to_string(rc) + "): " + kat_last_error());
}

// What a backward unpacked (a hook may return another tensor than it was given)
// or was handed: `a` and tensors on its device of the sizes the launch reads, or
// no launch. Call it on what as() returned, whose dtypes are the launch's.
struct Want {
  const Tensor& t;
  at::IntArrayRef sizes;
};
void need(const Tensor& a, std::initializer_list<Want> ts) {
  bool ok = plain(a);
  for (const Want& w : ts) ok = ok && plain(w.t) && w.t.device() == a.device() && w.t.sizes() == w.sizes;
  if (!ok)
    throw std::runtime_error(
        "backward: saved tensors and gradients must be tensors of one CUDA device with the sizes of the forward");
}

void* stream(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

// The tensor as [rows, cols] over its last dim: in place when the layout
// allows (unit last-dim stride, collapsible leading dims, rows that do not
// overlap), else a contiguous copy -- _lib.rows2d.
struct Rows {
  Tensor t;
  int64_t rows = 0, cols = 0, ld = 0;
  explicit Rows(const Tensor& x) : t(x) {
    if (!in_place()) {
      t = x.contiguous();
      rows = cols ? t.numel() / cols : 0;
      ld = cols;
    }
  }
  void* p() const { return t.data_ptr(); }

 private:
  bool in_place() {
    const int64_t n = t.dim();
    cols = n ? t.size(-1) : 1;
    rows = cols ? t.numel() / cols : 0;
    ld = cols;
    if (t.is_contiguous()) return true;
    if (cols != 1 && t.stride(-1) != 1) return false;
    int64_t st = -1, ext = 0;  // stride of the collapsed rows; the next outer dim's stride
    for (int64_t d = n - 2; d >= 0; --d) {
      if (t.size(d) == 1) continue;
      if (st < 0) st = t.stride(d);
      else if (t.stride(d) != ext) return false;
      ext = t.stride(d) * t.size(d);
    }
    if (st < 0) return true;  // one row
    ld = st;
    return ld >= cols;
  }
};

Tensor as(const Tensor& t, at::ScalarType dt) {
  const Tensor r = t.is_neg() ? t.resolve_neg() : t;
  return r.scalar_type() == dt ? r : r.to(dt);
}

// a weight or slopes tensor, which may come with leading dims of 1 (a view op costs
// a microsecond of host time)
Tensor flat(const Tensor& t) { return t.dim() == 1 ? t : t.reshape({-1}); }

Tensor bytes(size_t n, const Tensor& like) {
  return at::empty({(int64_t)std::max<size_t>(n, 1)}, like.options().dtype(at::kByte));
}

// ---------------------------------------------------------------------------
// row ops
// ---------------------------------------------------------------------------

struct Softmax : Function<Softmax> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, double eps) {
    const Rows r(x);
    Tensor out = at::empty(x.sizes(), x.options().memory_format(at::MemoryFormat::Contiguous));
    check(kat_rsoftmax_fwd(r.p(), out.data_ptr(), r.rows, r.cols, r.ld, r.cols, (float)eps, code(x), stream(x)),
          "kat_rsoftmax_fwd");
    ctx->save_for_backward({x, out});
    ctx->saved_data["eps"] = eps;
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &x = saved[0], out = as(saved[1], x.scalar_type()), dy = as(g[0], x.scalar_type());
    need(x, {{out, x.sizes()}, {dy, x.sizes()}});
    const Rows rx(x), rp(out), rg(dy);
    Tensor dx = at::empty(x.sizes(), x.options().memory_format(at::MemoryFormat::Contiguous));
    check(kat_rsoftmax_bwd(rg.p(), rx.p(), rp.p(), dx.data_ptr(), rx.rows, rx.cols, rg.ld, rx.ld, rp.ld, rx.cols,
                           (float)ctx->saved_data["eps"].toDouble(), code(x), stream(x)),
          "kat_rsoftmax_bwd");
    return {dx, Tensor()};
  }
};

std::optional<Tensor> softmax(const Tensor& x, double eps) {
  if (!untraced() || !plain(x) || x.numel() == 0) return std::nullopt;
  return Softmax::apply(x, eps);
}

struct Swiglu : Function<Swiglu> {
  static Tensor forward(AutogradContext* ctx, const Tensor& gate, const Tensor& value) {
    const Rows g(gate), v(value);
    Tensor out = at::empty(gate.sizes(), gate.options().memory_format(at::MemoryFormat::Contiguous));
    check(kat_rswiglu_fwd(g.p(), v.p(), out.data_ptr(), g.rows, g.cols, g.ld, v.ld, g.cols, code(gate), stream(gate)),
          "kat_rswiglu_fwd");
    ctx->save_for_backward({gate, value});
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list gr) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &gate = saved[0], value = as(saved[1], gate.scalar_type()), dy = as(gr[0], gate.scalar_type());
    need(gate, {{value, gate.sizes()}, {dy, gate.sizes()}});
    const Rows g(gate), v(value), y(dy);
    const auto opt = gate.options().memory_format(at::MemoryFormat::Contiguous);
    Tensor dg = at::empty(gate.sizes(), opt), dv = at::empty(gate.sizes(), opt);
    check(kat_rswiglu_bwd(y.p(), g.p(), v.p(), dg.data_ptr(), dv.data_ptr(), g.rows, g.cols, y.ld, g.ld, v.ld, g.cols,
                          g.cols, code(gate), stream(gate)),
          "kat_rswiglu_bwd");
    return {dg, dv};
  }
};

std::optional<Tensor> swiglu(const Tensor& gate, const Tensor& value) {
  if (!untraced() || !plain(gate) || !same_place(gate, {&value}) || gate.scalar_type() != value.scalar_type() ||
      gate.sizes() != value.sizes() || gate.numel() == 0)
    return std::nullopt;
  return Swiglu::apply(gate, value);
}

struct PackedSwiglu : Function<PackedSwiglu> {
  static Tensor forward(AutogradContext* ctx, const Tensor& gv) {
    const Rows r(gv);
    const int64_t f = r.cols / 2;
    auto shape = gv.sizes().vec();
    shape.back() = f;
    Tensor out = at::empty(shape, gv.options().memory_format(at::MemoryFormat::Contiguous));
    char* const g = (char*)r.p();
    check(kat_rswiglu_fwd(g, g + f * gv.element_size(), out.data_ptr(), r.rows, f, r.ld, r.ld, f, code(gv), stream(gv)),
          "kat_rswiglu_fwd");
    ctx->save_for_backward({gv});
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list gr) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &gv = saved[0], dy = as(gr[0], gv.scalar_type());
    auto half = gv.sizes().vec();
    if (!half.empty()) half.back() /= 2;
    need(gv, {{dy, half}});
    const Rows r(gv), y(dy);
    const int64_t f = r.cols / 2, es = gv.element_size();
    Tensor d = at::empty(gv.sizes(), gv.options().memory_format(at::MemoryFormat::Contiguous));
    char *const g = (char*)r.p(), *const o = (char*)d.data_ptr();
    check(kat_rswiglu_bwd(y.p(), g, g + f * es, o, o + f * es, r.rows, f, y.ld, r.ld, r.ld, r.cols, r.cols, code(gv),
                          stream(gv)),
          "kat_rswiglu_bwd");
    return {d};
  }
};

std::optional<Tensor> swiglu_packed(const Tensor& gv) {
  if (!untraced() || !plain(gv) || gv.dim() < 1 || gv.size(-1) % 2 != 0 || gv.numel() == 0) return std::nullopt;
  return PackedSwiglu::apply(gv);
}

// the weight as the kernels take it: contiguous, fp32 or of x's dtype
bool weight_ok(const Tensor& x, const Tensor& w) {
  return same_place(x, {&w}) && x.dim() >= 1 && w.is_contiguous() && w.numel() == x.size(-1) &&
         (w.scalar_type() == x.scalar_type() || (w.scalar_type() == at::kFloat && x.scalar_type() != at::kDouble));
}

// a saved weight in a dtype the kernels take
Tensor saved_weight(const Tensor& x, const Tensor& w) {
  const at::ScalarType xt = x.scalar_type(), wide = xt == at::kDouble ? at::kDouble : at::kFloat;
  return flat(as(w, w.scalar_type() == xt ? xt : wide)).contiguous();
}

Tensor dw_like(const Tensor& x, int64_t cols) {
  return at::empty({cols}, x.options().dtype(x.scalar_type() == at::kDouble ? at::kDouble : at::kFloat));
}

struct Norm : Function<Norm> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& w, double eps) {
    const Rows r(x);
    Tensor y = at::empty(x.sizes(), x.options().memory_format(at::MemoryFormat::Contiguous));
    Tensor mean = at::empty({r.rows}, x.options().dtype(at::kFloat));
    check(kat_men_fwd(r.p(), w.data_ptr(), y.data_ptr(), mean.data_ptr<float>(), r.rows, r.cols, r.ld, r.cols,
                      (float)eps, code(x), code(w), stream(x)),
          "kat_men_fwd");
    ctx->save_for_backward({x, w, mean});
    ctx->saved_data["eps"] = eps;
    return y;
  }
  static variable_list backward(AutogradContext* ctx, variable_list gr) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &x = saved[0], dy = as(gr[0], x.scalar_type());
    const Rows r(x), g(dy);
    const Tensor w = saved_weight(x, saved[1]), mean = as(saved[2], at::kFloat).contiguous();
    need(x, {{w, {r.cols}}, {mean, {r.rows}}, {dy, x.sizes()}});
    Tensor dx = at::empty(x.sizes(), x.options().memory_format(at::MemoryFormat::Contiguous)), dw = dw_like(x, r.cols);
    const size_t wsb = kat_men_bwd_workspace_size(r.rows, r.cols, code(x));
    const Tensor ws = bytes(wsb, x);
    check(kat_men_bwd(g.p(), r.p(), w.data_ptr(), mean.data_ptr<float>(), dx.data_ptr(), dw.data_ptr(), ws.data_ptr(),
                      wsb, r.rows, r.cols, g.ld, r.ld, r.cols, (float)ctx->saved_data["eps"].toDouble(), code(x),
                      code(w), stream(x)),
          "kat_men_bwd");
    return {dx, dw, Tensor()};
  }
};

std::optional<Tensor> norm(const Tensor& x, const Tensor& w, double eps) {
  if (!untraced() || !plain(x) || x.numel() == 0 || !weight_ok(x, w)) return std::nullopt;
  return Norm::apply(x, w, eps);
}

struct AddNorm : Function<AddNorm> {
  static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& r, const Tensor& w, double eps,
                               at::ScalarType yt) {
    const Rows rx(x), rr(r);
    const auto opt = x.options().memory_format(at::MemoryFormat::Contiguous);
    Tensor h = at::empty(x.sizes(), opt), y = at::empty(x.sizes(), opt.dtype(yt));
    Tensor mean = at::empty({rx.rows}, x.options().dtype(at::kFloat));
    check(kat_add_men_fwd(rx.p(), rr.p(), w.data_ptr(), h.data_ptr(), y.data_ptr(), mean.data_ptr<float>(), rx.rows,
                          rx.cols, rx.ld, rr.ld, rx.cols, rx.cols, (float)eps, code(x), code(r), code(y), code(w),
                          stream(x)),
          "kat_add_men_fwd");
    ctx->save_for_backward({h, w, mean});
    ctx->saved_data["eps"] = eps;
    ctx->saved_data["x"] = (int64_t)x.scalar_type();
    ctx->saved_data["r"] = (int64_t)r.scalar_type();
    ctx->saved_data["y"] = (int64_t)yt;
    return {h, y};
  }
  static variable_list backward(AutogradContext* ctx, variable_list gr) {
    const auto saved = ctx->get_saved_variables();
    const auto rt = (at::ScalarType)ctx->saved_data["r"].toInt(), yt = (at::ScalarType)ctx->saved_data["y"].toInt();
    const Tensor h = as(saved[0], (at::ScalarType)ctx->saved_data["x"].toInt());
    const Tensor dy = as(gr[1], yt), dh = as(gr[0], h.scalar_type());
    const Rows rh(h), g(dy), d(dh);
    const Tensor w = saved_weight(h, saved[1]), mean = as(saved[2], at::kFloat).contiguous();
    need(h, {{w, {rh.cols}}, {mean, {rh.rows}}, {dy, h.sizes()}, {dh, h.sizes()}});
    const auto opt = h.options().memory_format(at::MemoryFormat::Contiguous);
    Tensor dx = at::empty(h.sizes(), opt), dr, dw = dw_like(h, rh.cols);
    // a same-dtype branch gets the stream's gradient itself, a narrower one its cast
    const bool want_r = ctx->needs_input_grad(1);
    if (want_r && rt != h.scalar_type()) dr = at::empty(h.sizes(), opt.dtype(rt));
    const size_t wsb = kat_men_bwd_workspace_size(rh.rows, rh.cols, code(h));
    const Tensor ws = bytes(wsb, h);
    check(kat_add_men_bwd(g.p(), d.p(), rh.p(), w.data_ptr(), mean.data_ptr<float>(), dx.data_ptr(),
                          dr.defined() ? dr.data_ptr() : nullptr, dw.data_ptr(), ws.data_ptr(), wsb, rh.rows, rh.cols,
                          g.ld, d.ld, rh.ld, rh.cols, rh.cols, (float)ctx->saved_data["eps"].toDouble(), code(h),
                          dtype_code(dr.defined() ? rt : h.scalar_type()), dtype_code(yt), code(w), stream(h)),
          "kat_add_men_bwd");
    return {dx, !want_r ? Tensor() : dr.defined() ? dr : dx, dw, Tensor(), Tensor()};
  }
};

// out: the normalised output's dtype (None: x's)
std::optional<std::tuple<Tensor, Tensor>> add_norm(const Tensor& x, const Tensor& r, const Tensor& w, double eps,
                                                   std::optional<at::ScalarType> out) {
  if (!untraced() || !plain(x) || x.numel() == 0 || !same_place(x, {&r}) || r.sizes() != x.sizes() || !weight_ok(x, w))
    return std::nullopt;
  const at::ScalarType xt = x.scalar_type(), yt = out.value_or(xt);
  auto narrow_ok = [&](at::ScalarType t) {
    return t == xt || (xt == at::kFloat && (t == at::kBFloat16 || t == at::kHalf));
  };
  if (!narrow_ok(r.scalar_type()) || !narrow_ok(yt)) return std::nullopt;
  const auto o = AddNorm::apply(x, r, w, eps, yt);
  return std::make_tuple(o[0], o[1]);
}

// ---------------------------------------------------------------------------
// attention
// ---------------------------------------------------------------------------

// One [B, H, T, D] operand: where it starts and its (b, h, t) strides.
struct View {
  char* p;
  int64_t s[3];
};
View bhtd(const Tensor& t) { return {(char*)t.data_ptr(), {t.stride(0), t.stride(1), t.stride(2)}}; }
// part i (q, k, v) of a packed [B, T, 3, H, D] tensor
View part(const Tensor& t, int i) {
  return {(char*)t.data_ptr() + i * t.stride(2) * t.element_size(), {t.stride(0), t.stride(3), t.stride(1)}};
}
// [B, T, H, D] memory
View bthd(const Tensor& t) { return {(char*)t.data_ptr(), {t.stride(0), t.stride(2), t.stride(1)}}; }

// The MFMA kernels' envelope (forward.py: _tiled_reason): calls inside it get
// no fallback warning.
bool head_dim_ok(int64_t D, int64_t es) {
  const int64_t step = 16 / es;
  return D >= step && D <= 256 && D % step == 0;
}
bool in_envelope(std::initializer_list<View> vs, int64_t T, int64_t D, int64_t es) {
  constexpr int64_t lim = 0x7fffffff, pad = 128;
  for (const View& v : vs) {
    if (reinterpret_cast<uintptr_t>(v.p) % 16) return false;
    for (int64_t s : v.s)
      if ((s * es) % 16) return false;
    if (v.s[2] < D || (T + pad) * v.s[2] * es > lim) return false;
  }
  return es != 2 || (T * D * 2 < lim && T * 8 < lim);
}
bool attn_dtype(const Tensor& t) { return plain(t) && code(t) != KAT_F64; }
bool slopes_ok(const Tensor& q, const Tensor& s, int64_t H) {
  return same_place(q, {&s}) && s.scalar_type() == at::kFloat && s.is_contiguous() && s.numel() == H;
}
// slopes of a module cast whole (bf16 / fp16, as its buffer becomes), which the
// entry points convert as the Python functions do
bool slopes_narrow(const Tensor& q, const Tensor& s, int64_t H) {
  return same_place(q, {&s}) && (s.scalar_type() == at::kBFloat16 || s.scalar_type() == at::kHalf) &&
         !s.requires_grad() && s.numel() == H;
}
Tensor slopes_of(const Tensor& s) {
  if (s.scalar_type() == at::kFloat) return s;
  at::NoGradGuard g;
  return s.to(at::kFloat).contiguous();
}

struct Dims {
  int64_t B, H, T, D;
};
void put(int64_t* dst, std::initializer_list<View> vs) {
  for (const View& v : vs)
    for (int64_t s : v.s) *dst++ = s;
}

void run_fwd(const Dims& n, const View& q, const View& k, const View& v, const View& o, const Tensor& L,
             const Tensor& slopes, double scale, double eps, const Tensor& km, bool extended, bool causal, int dt,
             void* st) {
  int64_t s[12], ls[3] = {L.stride(0), L.stride(1), L.stride(2)};
  put(s, {q, k, v, o});
  if (extended)
    check(kat_attn_fwd_masked(q.p, k.p, v.p, o.p, L.data_ptr<float>(), slopes.data_ptr<float>(),
                              km.defined() ? km.data_ptr<uint8_t>() : nullptr, n.T, n.B, n.H, n.T, n.D, s, ls,
                              (float)scale, (float)eps, causal, dt, st),
          "kat_attn_fwd_masked");
  else
    check(kat_attn_fwd(q.p, k.p, v.p, o.p, L.data_ptr<float>(), slopes.data_ptr<float>(), n.B, n.H, n.T, n.D, s, ls,
                       (float)scale, (float)eps, causal, dt, st),
          "kat_attn_fwd");
}

void run_bwd(const Dims& n, const View& q, const View& k, const View& v, const View& o, const Tensor& L,
             const View& go, const View& dq, const View& dk, const View& dv, const Tensor& slopes, double scale,
             double eps, const Tensor& km, bool extended, bool causal, const Tensor& like, void* st) {
  int64_t s[24], ls[3] = {L.stride(0), L.stride(1), L.stride(2)};
  put(s, {q, k, v, o, go, dq, dk, dv});
  const int dt = code(like);
  const size_t wsb = extended ? kat_attn_bwd_masked_workspace_size(n.B, n.H, n.T, n.D, dt, causal)
                              : kat_attn_bwd_workspace_size(n.B, n.H, n.T, n.D, dt);
  const Tensor ws = bytes(wsb, like);
  if (extended)
    check(kat_attn_bwd_masked(q.p, k.p, v.p, o.p, L.data_ptr<float>(), go.p, dq.p, dk.p, dv.p,
                              slopes.data_ptr<float>(), km.defined() ? km.data_ptr<uint8_t>() : nullptr, n.T,
                              ws.data_ptr(), wsb, n.B, n.H, n.T, n.D, s, ls, (float)scale, (float)eps, causal, dt, st),
          "kat_attn_bwd_masked");
  else
    check(kat_attn_bwd(q.p, k.p, v.p, o.p, L.data_ptr<float>(), go.p, dq.p, dk.p, dv.p, slopes.data_ptr<float>(),
                       ws.data_ptr(), wsb, n.B, n.H, n.T, n.D, s, ls, (float)scale, (float)eps, causal, dt, st),
          "kat_attn_bwd");
}

// What the backward does with operands outside the envelope (a gradient of
// odd layout, or saved tensors that hooks returned in another one): the Python
// function converts, warns and launches. The views are [B, H, T, D].
void python_bwd(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o, const Tensor& L, const Tensor& go,
                const Tensor& dq, const Tensor& dk, const Tensor& dv, const Tensor& slopes, double scale, double eps,
                const Tensor& km, bool extended, bool causal) {
  py::gil_scoped_acquire gil;
  auto unit = [](const Tensor& t) { return t.size(-1) == 1 || t.stride(-1) == 1 ? t : t.contiguous(); };
  py::object none = py::none();
  py::module_::import("fastalgebraictransformer_amd.backward")
      .attr("_attn_bwd_into")(unit(q), unit(k), unit(v), unit(o), L, unit(go), dq, dk, dv, slopes, scale, causal, eps,
                              km.defined() ? py::cast(km) : none, extended);
}

void need_dims(const Tensor& a, int64_t n) {
  if (a.dim() != n || (n == 5 && a.size(2) != 3))
    throw std::runtime_error("backward: a saved attention input has lost its dimensions");
}

// the key mask a backward unpacked (undefined: none) as the kernels read it:
// uint8, rows of T bytes
Tensor saved_mask(const Tensor& q, const Tensor& km, int64_t B, int64_t T) {
  if (!km.defined()) return km;
  if (!km.is_cuda() || km.device() != q.device() || km.layout() != at::kStrided || km.scalar_type() != at::kByte ||
      km.sizes() != at::IntArrayRef({B, T}))
    throw std::runtime_error("backward: the saved key mask must be uint8 [B, T] on the inputs' CUDA device");
  return km.contiguous();
}

// a [B, T] key mask as uint8 (nonzero = attend), a copy of the caller's
struct Mask {
  Tensor t;  // undefined: no mask
};
bool mask_ok(const Tensor& q, const std::optional<Tensor>& m, int64_t B, int64_t T) {
  return !m || (m->defined() && m->is_cuda() && m->device() == q.device() && m->layout() == at::kStrided &&
                !m->key_set().has_any(c10::DispatchKeySet{c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched,
                                                          c10::DispatchKey::FuncTorchGradWrapper}) &&
                m->dim() == 2 && m->size(0) == B && m->size(1) == T);
}
Mask mask_of(const std::optional<Tensor>& m) {
  if (!m) return {};
  at::NoGradGuard g;
  // a bool mask converts in one pass (its elements are 0 or 1)
  return {(m->scalar_type() == at::kBool ? *m : m->ne(0)).to(at::kByte).contiguous()};
}

struct Attention : Function<Attention> {
  static Tensor forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& slopes,
                        double scale, double eps, Mask km, bool extended, bool causal) {
    const Dims n{q.size(0), q.size(1), q.size(2), q.size(3)};
    Tensor o = at::empty(q.sizes(), q.options().memory_format(at::MemoryFormat::Contiguous));
    Tensor L = at::empty({n.B, n.H, n.T}, q.options().dtype(at::kFloat));
    run_fwd(n, bhtd(q), bhtd(k), bhtd(v), bhtd(o), L, slopes, scale, eps, km.t, extended, causal, code(q), stream(q));
    ctx->save_for_backward({q, k, v, o, L, slopes, km.t});
    ctx->saved_data["scale"] = scale;
    ctx->saved_data["eps"] = eps;
    ctx->saved_data["extended"] = extended;
    ctx->saved_data["causal"] = causal;
    return o;
  }
  static variable_list backward(AutogradContext* ctx, variable_list gr) {
    const auto s = ctx->get_saved_variables();
    const at::ScalarType dt = s[0].scalar_type();
    const Tensor &q = s[0], k = as(s[1], dt), v = as(s[2], dt), o = as(s[3], dt), L = as(s[4], at::kFloat);
    Tensor go = as(gr[0], dt);
    need_dims(q, 4);
    const Tensor slopes = flat(s[5]), km = saved_mask(q, s[6], q.size(0), q.size(2));
    need(q, {{k, q.sizes()}, {v, q.sizes()}, {o, q.sizes()}, {L, q.sizes().slice(0, 3)}, {slopes, {q.size(1)}},
             {go, q.sizes()}});
    const double scale = ctx->saved_data["scale"].toDouble(), eps = ctx->saved_data["eps"].toDouble();
    const bool extended = ctx->saved_data["extended"].toBool(), causal = ctx->saved_data["causal"].toBool();
    const Dims n{q.size(0), q.size(1), q.size(2), q.size(3)};
    if (go.stride(-1) != 1 && n.D != 1) go = go.contiguous();
    const auto opt = q.options().memory_format(at::MemoryFormat::Contiguous);
    Tensor dq = at::empty(q.sizes(), opt), dk = at::empty(q.sizes(), opt), dv = at::empty(q.sizes(), opt);
    auto unit = [](const Tensor& t) { return t.stride(-1) == 1; };
    if (unit(q) && unit(k) && unit(v) && unit(o) && unit(go) && slopes_ok(q, slopes, n.H) &&
        in_envelope({bhtd(q), bhtd(k), bhtd(v), bhtd(o), bhtd(go)}, n.T, n.D, q.element_size()))
      run_bwd(n, bhtd(q), bhtd(k), bhtd(v), bhtd(o), L, bhtd(go), bhtd(dq), bhtd(dk), bhtd(dv), slopes, scale, eps,
              km, extended, causal, q, stream(q));
    else
      python_bwd(q, k, v, o, L, go, dq, dk, dv, slopes, scale, eps, km, extended, causal);
    return {dq, dk, dv, Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

bool attn_ok(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& slopes) {
  return untraced() && attn_dtype(q) && same_place(q, {&k, &v}) && k.scalar_type() == q.scalar_type() &&
         v.scalar_type() == q.scalar_type() && q.dim() == 4 && k.sizes() == q.sizes() && v.sizes() == q.sizes() &&
         q.numel() > 0 && q.stride(3) == 1 && k.stride(3) == 1 && v.stride(3) == 1 &&
         head_dim_ok(q.size(3), q.element_size()) &&
         in_envelope({bhtd(q), bhtd(k), bhtd(v)}, q.size(2), q.size(3), q.element_size()) &&
         (slopes_ok(q, slopes, q.size(1)) || slopes_narrow(q, slopes, q.size(1)));
}

std::optional<Tensor> attention(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& slopes, double scale,
                                double eps) {
  if (!attn_ok(q, k, v, slopes)) return std::nullopt;
  return Attention::apply(q, k, v, slopes_of(slopes), scale, eps, Mask{}, false, true);
}

std::optional<Tensor> attention_masked(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& slopes,
                                       double scale, const std::optional<Tensor>& km, bool causal, double eps) {
  if (!attn_ok(q, k, v, slopes) || !mask_ok(q, km, q.size(0), q.size(2))) return std::nullopt;
  return Attention::apply(q, k, v, slopes_of(slopes), scale, eps, mask_of(km), true, causal);
}

struct PackedAttention : Function<PackedAttention> {
  static Tensor forward(AutogradContext* ctx, const Tensor& qkv, const Tensor& slopes, double scale, double eps,
                        Mask km) {
    const Dims n{qkv.size(0), qkv.size(3), qkv.size(1), qkv.size(4)};
    Tensor y = at::empty({n.B, n.T, n.H, n.D}, qkv.options().memory_format(at::MemoryFormat::Contiguous));
    Tensor L = at::empty({n.B, n.H, n.T}, qkv.options().dtype(at::kFloat));
    run_fwd(n, part(qkv, 0), part(qkv, 1), part(qkv, 2), bthd(y), L, slopes, scale, eps, km.t, km.t.defined(), true,
            code(qkv), stream(qkv));
    ctx->save_for_backward({qkv, y, L, slopes, km.t});
    ctx->saved_data["scale"] = scale;
    ctx->saved_data["eps"] = eps;
    return y;
  }
  static variable_list backward(AutogradContext* ctx, variable_list gr) {
    const auto s = ctx->get_saved_variables();
    const Tensor &qkv = s[0], y = as(s[1], qkv.scalar_type()), L = as(s[2], at::kFloat), slopes = flat(s[3]);
    Tensor go = as(gr[0], qkv.scalar_type());
    need_dims(qkv, 5);
    const int64_t yd[] = {qkv.size(0), qkv.size(1), qkv.size(3), qkv.size(4)}, ld[] = {yd[0], yd[2], yd[1]};
    need(qkv, {{y, yd}, {L, ld}, {slopes, {yd[2]}}, {go, yd}});
    const Tensor km = saved_mask(qkv, s[4], qkv.size(0), qkv.size(1));
    const double scale = ctx->saved_data["scale"].toDouble(), eps = ctx->saved_data["eps"].toDouble();
    const Dims n{qkv.size(0), qkv.size(3), qkv.size(1), qkv.size(4)};
    if (go.stride(-1) != 1 && n.D != 1) go = go.contiguous();
    Tensor d = at::empty(qkv.sizes(), qkv.options().memory_format(at::MemoryFormat::Contiguous));
    if (qkv.stride(-1) == 1 && y.stride(-1) == 1 && go.stride(-1) == 1 && slopes_ok(qkv, slopes, n.H) &&
        in_envelope({part(qkv, 0), part(qkv, 1), part(qkv, 2), bthd(y), bthd(go)}, n.T, n.D, qkv.element_size())) {
      run_bwd(n, part(qkv, 0), part(qkv, 1), part(qkv, 2), bthd(y), L, bthd(go), part(d, 0), part(d, 1), part(d, 2),
              slopes, scale, eps, km, km.defined(), true, qkv, stream(qkv));
    } else {
      auto p = [](const Tensor& t, int i) { return t.select(2, i).transpose(1, 2); };
      python_bwd(p(qkv, 0), p(qkv, 1), p(qkv, 2), y.transpose(1, 2), L, go.transpose(1, 2), p(d, 0), p(d, 1), p(d, 2),
                 slopes, scale, eps, km, km.defined(), true);
    }
    return {d, Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

std::optional<Tensor> attention_packed(const Tensor& qkv, const Tensor& slopes, double scale, double eps,
                                       const std::optional<Tensor>& km) {
  if (!untraced() || !attn_dtype(qkv) || qkv.dim() != 5 || qkv.size(2) != 3 || qkv.numel() == 0 ||
      qkv.stride(4) != 1 || !head_dim_ok(qkv.size(4), qkv.element_size()) ||
      !in_envelope({part(qkv, 0), part(qkv, 1), part(qkv, 2)}, qkv.size(1), qkv.size(4), qkv.element_size()) ||
      !(slopes_ok(qkv, slopes, qkv.size(3)) || slopes_narrow(qkv, slopes, qkv.size(3))) ||
      !mask_ok(qkv, km, qkv.size(0), qkv.size(1)))
    return std::nullopt;
  return PackedAttention::apply(qkv, slopes_of(slopes), scale, eps, mask_of(km));
}

// q [B, H, D] against caches [B, H, T, D]: (out, L); no gradient
std::optional<std::tuple<Tensor, Tensor>> decode(const Tensor& q, const Tensor& k, const Tensor& v,
                                                 const Tensor& slopes, double scale,
                                                 const std::optional<Tensor>& lengths, double eps) {
  if (!untraced() || !attn_dtype(q) || !same_place(q, {&k, &v}) || k.scalar_type() != q.scalar_type() ||
      v.scalar_type() != q.scalar_type() || q.dim() != 3 || k.dim() != 4 || k.sizes() != v.sizes() ||
      k.size(0) != q.size(0) || k.size(1) != q.size(1) || k.size(3) != q.size(2) || q.numel() == 0 ||
      k.numel() == 0 || q.stride(2) != 1 || k.stride(3) != 1 || v.stride(3) != 1 ||
      !(slopes_ok(q, slopes, q.size(1)) || slopes_narrow(q, slopes, q.size(1))))
    return std::nullopt;
  if (lengths && !(lengths->defined() && lengths->is_cuda() && lengths->device() == q.device() &&
                   lengths->layout() == at::kStrided && lengths->scalar_type() == at::kInt &&
                   lengths->is_contiguous() && lengths->numel() == q.size(0) &&
                   !lengths->key_set().has(c10::DispatchKey::Python)))
    return std::nullopt;
  at::NoGradGuard g;
  const Tensor sl = slopes_of(slopes);
  const int64_t B = q.size(0), H = q.size(1), D = q.size(2), T = k.size(2);
  Tensor out = at::empty({B, H, D}, q.options().memory_format(at::MemoryFormat::Contiguous));
  Tensor L = at::empty({B, H}, q.options().dtype(at::kFloat));
  const size_t wsb = kat_attn_decode_workspace_size(B, H, T, D, code(q));
  const Tensor ws = bytes(std::max<size_t>(wsb, 4), q);
  const int64_t s[10] = {q.stride(0), q.stride(1), k.stride(0), k.stride(1), k.stride(2),
                         v.stride(0), v.stride(1), v.stride(2), out.stride(0), out.stride(1)};
  check(kat_attn_decode(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), L.data_ptr<float>(),
                        sl.data_ptr<float>(), lengths ? lengths->data_ptr<int32_t>() : nullptr, ws.data_ptr(),
                        wsb, B, H, T, D, s, (float)scale, (float)eps, code(q), stream(q)),
        "kat_attn_decode");
  return std::make_tuple(out, L);
}

}  // namespace

PYBIND11_MODULE(_katops, m) {
  // the GIL is released while a call runs (as around a ctypes call)
  typedef py::call_guard<py::gil_scoped_release> nogil;
  m.def("softmax", &softmax, nogil());
  m.def("swiglu", &swiglu, nogil());
  m.def("swiglu_packed", &swiglu_packed, nogil());
  m.def("norm", &norm, nogil());
  m.def("add_norm", &add_norm, nogil());
  m.def("attention", &attention, nogil());
  m.def("attention_masked", &attention_masked, nogil());
  m.def("attention_packed", &attention_packed, nogil());
  m.def("decode", &decode, nogil());
  // the layout rules alone (any device): (in place?, rows, cols, row stride)
  // of rows2d, and whether [B, H, T, D] operands lie in the MFMA envelope
  m.def("rows2d", [](const Tensor& t) {
    const Rows r(t);
    return std::make_tuple(r.t.is_same(t), r.rows, r.cols, r.ld);
  });
  m.def("attn_layout_ok", [](const std::vector<Tensor>& ts) {
    for (const Tensor& t : ts)
      if (t.dim() != 4 || t.stride(3) != 1 || !head_dim_ok(t.size(3), t.element_size()) ||
          !in_envelope({bhtd(t)}, t.size(2), t.size(3), t.element_size()))
        return false;
    return true;
  });
}
