// Host path of the differentiable entry points: a CPython module (_ua_host) over the C ABI of libua_hip.so.
//
// On short sequences a pass is a few kernels of 5 to 30 us, and what the caller waits for is the host: building
// descriptors, tensors and autograd nodes in Python took 320 us per forward + backward (520 us through the decoder front end,
// whose views each add a node), against about 60 us here.  Every function returns None for calls it does not take (tensors off
// the GPU or of mismatched shapes and dtypes, tensor subclasses, function transforms, dispatch modes, more heads than grid
// rows); the Python operators then do the same work, or raise.
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/Exceptions.h>

#include "../../include/ua.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::Function;
using torch::autograd::variable_list;

struct UaFailure : std::runtime_error { using std::runtime_error::runtime_error; };
PyObject* g_error = nullptr;     // _lib.UaError
PyObject* g_ops = nullptr;       // module ops: owner of the note that the merge's backward leaves for the chunked backward

void check(int code, const char* what) {
  if (code < 0) throw UaFailure(std::string(what) + " failed (" + std::to_string(code) + "): " + ua_last_error());
}
size_t workspace_bytes(const ua_desc& d, int op) {
  const size_t n = ua_workspace_bytes(&d, op);
  if (n == 0) throw UaFailure(std::string("unsupported problem: ") + ua_last_error());
  return n;
}
Tensor bytes(size_t n, const Tensor& like) { return at::empty({(int64_t)n}, like.options().dtype(at::kByte)); }
ua_stream_t stream_of(const Tensor& t) { return (ua_stream_t)c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

constexpr int64_t kGridRows = 65535;     // one grid row per head (times chunk, in the chunked operator)
bool dtype_ok(const Tensor& t) { return t.scalar_type() == at::kBFloat16 || t.scalar_type() == at::kFloat; }
int dtype_code(const Tensor& t) { return t.scalar_type() == at::kBFloat16 ? UA_BF16 : UA_F32; }

// [b, h, ...] gate whose trailing dims merge into one of L positions with a uniform stride
bool gate_stride(const Tensor& t, int64_t& st) {
  if (t.dim() == 3) { st = t.stride(2); return true; }
  if (t.dim() != 4) return false;
  st = t.stride(3);
  return t.size(2) == 1 || t.stride(2) == t.size(3) * t.stride(3);
}

// How the tensors of one entry point map onto the operator.
enum Kind { UNIVERSAL = 0, DECODER = 1, GEN2 = 2 };
struct Problem {
  ua_desc d{};
  ua_rows k{}, v{}, q{};
  ua_gates g{};
  Tensor src, dest;                       // gates kept alive when they had to be copied
};
ua_rows rows5(const Tensor& t) {           // [b, h, n, c, d]
  return ua_rows{t.data_ptr(), t.stride(0), t.stride(1), 0, t.stride(2), t.stride(3), (int32_t)t.size(3)};
}
ua_rows rows_of_queries(const Tensor& t) { // [b, h, r, l, d] or [b, h, r, n, c, d]
  if (t.dim() == 5) return ua_rows{t.data_ptr(), t.stride(0), t.stride(1), t.stride(2), 0, t.stride(3), (int32_t)t.size(3)};
  return ua_rows{t.data_ptr(), t.stride(0), t.stride(1), t.stride(2), t.stride(3), t.stride(4), (int32_t)t.size(4)};
}
// rows of a tensor shaped like the entry point's queries (also O, dO and dxq)
ua_rows rows_like_queries(int kind, const Tensor& t, int h, int r) {
  switch (kind) {
    case DECODER:    // [b, s, n, d], query head j = h_index * r + r_index
      return ua_rows{t.data_ptr(), t.stride(0), t.stride(2) * r, t.stride(2), 0, t.stride(1), (int32_t)t.size(1)};
    case GEN2:       // [B, H_q, L, d], query head j = r_index * H_kv + h_index
      return ua_rows{t.data_ptr(), t.stride(0), t.stride(1), t.stride(1) * h, 0, t.stride(2), (int32_t)t.size(2)};
    default:
      return rows_of_queries(t);
  }
}
ua_rows rows_like_keys(int kind, const Tensor& t) {
  switch (kind) {
    case DECODER: return ua_rows{t.data_ptr(), t.stride(0), t.stride(2), 0, 0, t.stride(1), (int32_t)t.size(1)};
    case GEN2: return ua_rows{t.data_ptr(), t.stride(0), t.stride(1), 0, 0, t.stride(2), (int32_t)t.size(2)};
    default: return rows5(t);
  }
}
// the same for a result the library writes: rows t at t * stride_inner
ua_rows result_keys(int kind, const Tensor& t, int L) {
  ua_rows r = rows_like_keys(kind, t);
  r.inner_len = L;      // contiguous: chunk boundaries do not matter
  return r;
}
ua_rows result_queries(int kind, const Tensor& t, int h, int r, int L) {
  ua_rows x = rows_like_queries(kind, t, h, r);
  x.inner_len = L;
  return x;
}

// q, k, v, s1 (, s2) in the argument order of Problem, whatever the entry point's
bool describe(int kind, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& s1, const Tensor& s2, int flags, Problem& p) {
  if (!q.is_cuda() || !k.is_cuda() || !v.is_cuda() || !s1.is_cuda() || (s2.defined() && !s2.is_cuda())) return false;
  const auto dev = q.device();
  if (k.device() != dev || v.device() != dev || s1.device() != dev || (s2.defined() && s2.device() != dev)) return false;
  if (!dtype_ok(q) || k.scalar_type() != q.scalar_type() || v.scalar_type() != q.scalar_type()) return false;
  if (q.numel() == 0 || k.sizes() != v.sizes()) return false;
  int64_t b, h, r, L, d;
  if (kind == DECODER) {
    if (q.dim() != 4 || k.dim() != 4 || s1.dim() != 3) return false;
    b = q.size(0); L = q.size(1); d = q.size(3); h = k.size(2);
    if (k.size(0) != b || k.size(1) != L || k.size(3) != d || h == 0 || q.size(2) % h) return false;
    r = q.size(2) / h;
    if (s1.size(0) != b || s1.size(1) != L || s1.size(2) != 2 * h) return false;
  } else if (kind == GEN2) {
    if (q.dim() != 4 || k.dim() != 4) return false;
    b = q.size(0); L = q.size(2); d = q.size(3); h = k.size(1);
    if (k.size(0) != b || k.size(2) != L || k.size(3) != d || h == 0 || q.size(1) % h) return false;
    r = q.size(1) / h;
    if (s1.dim() != 3 || s2.dim() != 3) return false;
  } else {
    if ((q.dim() != 5 && q.dim() != 6) || k.dim() != 5) return false;
    b = k.size(0); h = k.size(1); L = k.size(2) * k.size(3); d = k.size(4); r = q.size(2);
    if (q.size(0) != b || q.size(1) != h || q.size(-1) != d || (q.dim() == 5 ? q.size(3) : q.size(3) * q.size(4)) != L) return false;
  }
  if (b * h * r > kGridRows || L > INT32_MAX / 2) return false;
  if (q.stride(-1) != 1 || k.stride(-1) != 1 || v.stride(-1) != 1) return false;
  p.d = ua_desc{(int32_t)b, (int32_t)h, (int32_t)r, (int32_t)L, (int32_t)d, 0, dtype_code(q), flags};
  p.q = rows_like_queries(kind, q, (int)h, (int)r);
  p.k = rows_like_keys(kind, k);
  p.v = rows_like_keys(kind, v);
  const auto gt = s1.scalar_type();
  if (kind == DECODER) {
    if (gt != q.scalar_type() && gt != at::kFloat) return false;
    char* base = (char*)s1.data_ptr();
    p.g = ua_gates{base, base + h * s1.stride(2) * s1.element_size(), s1.stride(0), s1.stride(2), s1.stride(1)};
  } else {
    if (s2.scalar_type() != gt || (gt != q.scalar_type() && gt != at::kFloat)) return false;
    if (s1.dim() < 3 || s2.dim() < 3 || s1.size(0) != b || s2.size(0) != b || s1.size(1) != h || s2.size(1) != h ||
        s1.numel() != b * h * L || s2.numel() != b * h * L) return false;
    int64_t st1, st2;
    if (!gate_stride(s1, st1) || !gate_stride(s2, st2) || st1 != st2 || s1.stride(0) != s2.stride(0) || s1.stride(1) != s2.stride(1)) {
      if (s1.dim() > 4 || s2.dim() > 4) return false;
      p.src = s1.reshape({b, h, L}).contiguous();
      p.dest = s2.reshape({b, h, L}).contiguous();
      p.g = ua_gates{p.src.data_ptr(), p.dest.data_ptr(), h * L, L, 1};
    } else {
      p.g = ua_gates{s1.data_ptr(), s2.data_ptr(), s1.stride(0), s1.stride(1), st1};
    }
  }
  if (gt == at::kFloat && q.scalar_type() != at::kFloat) p.d.flags |= UA_FLAG_GATES_F32;
  return true;
}

struct FusedResult { Tensor O, lse, state; };
FusedResult fused_forward(int kind, const Problem& p, const Tensor& q, bool keep) {
  const ua_desc& d = p.d;
  Tensor ws = bytes(workspace_bytes(d, UA_OP_FUSED_FWD), q);
  Tensor O = at::empty(q.sizes(), q.options());
  Tensor lse = at::empty({d.b, d.h, d.r, d.L}, q.options().dtype(at::kFloat));
  const ua_rows o = result_queries(kind, O, d.h, d.r, d.L);
  check(ua_fused_fwd_strided(&d, &p.k, &p.v, &p.q, &p.g, &o, lse.data_ptr<float>(), ws.data_ptr(), (size_t)ws.numel(), stream_of(q)),
        "ua_fused_fwd_strided");
  return {O, lse, keep ? ws : Tensor()};
}

// a tensor that arrives as an upstream gradient, in the dtype of the tensors and with unit feature stride
Tensor upstream(const Tensor& g, const Tensor& like) {
  Tensor x = g.scalar_type() == like.scalar_type() ? g : g.to(like.scalar_type());
  return x.stride(-1) == 1 ? x : x.contiguous();
}

// -> gradients of q, k, v, s1 (, s2)
variable_list fused_backward(int kind, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& s1, const Tensor& s2, const Tensor& O,
                             const Tensor& lse, const Tensor& g, const Tensor& state, int flags) {
  Problem p;
  TORCH_CHECK(describe(kind, q, k, v, s1, s2, flags, p), "the tensors saved by the forward changed");
  const ua_desc& d = p.d;
  c10::DeviceGuard guard(q.device());
  Tensor dO = upstream(g, q);
  Tensor ws = bytes(workspace_bytes(d, state.defined() ? UA_OP_FUSED_BWD_SCRATCH : UA_OP_FUSED_BWD), q);
  Tensor dq = at::empty(q.sizes(), q.options()), dk = at::empty(k.sizes(), k.options()), dv = at::empty(v.sizes(), v.options());
  Tensor d1 = at::empty(s1.sizes(), s1.options()), d2 = kind == DECODER ? Tensor() : at::empty(s2.sizes(), s2.options());
  ua_gates dg;
  if (kind == DECODER) {
    char* base = (char*)d1.data_ptr();
    dg = ua_gates{base, base + (int64_t)d.h * d1.element_size(), (int64_t)d.L * 2 * d.h, 1, 2 * (int64_t)d.h};
  } else {
    dg = ua_gates{d1.data_ptr(), d2.data_ptr(), (int64_t)d.h * d.L, d.L, 1};
  }
  const ua_rows o = rows_like_queries(kind, O, d.h, d.r), go = rows_like_queries(kind, dO, d.h, d.r);
  const ua_rows gq = result_queries(kind, dq, d.h, d.r, d.L), gk = result_keys(kind, dk, d.L), gv = result_keys(kind, dv, d.L);
  check(ua_fused_bwd_strided(&d, &p.k, &p.v, &p.q, &p.g, &o, lse.data_ptr<float>(), &go, &gk, &gv, &gq, &dg,
                             state.defined() ? state.data_ptr() : nullptr, ws.data_ptr(), (size_t)ws.numel(), stream_of(q)),
        "ua_fused_bwd_strided");
  return {dq, dk, dv, d1, d2};
}

[[noreturn]] void not_differentiable() {
  throw std::runtime_error("the hand-written backward passes of Universal Attention are not differentiable (the reference's are not either)");
}
// The backward as a node of its own, for callers that record a graph through it (create_graph): differentiating it raises.
struct FusedBackward : Function<FusedBackward> {
  static variable_list forward(AutogradContext*, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& s1, const std::optional<Tensor>& s2,
                               const Tensor& O, const Tensor& lse, const Tensor& g, const std::optional<Tensor>& state, int64_t kind, int64_t flags) {
    variable_list r = fused_backward((int)kind, q, k, v, s1, s2.value_or(Tensor()), O, lse, g, state.value_or(Tensor()), (int)flags);
    if (kind == DECODER) r.pop_back();
    return r;
  }
  static variable_list backward(AutogradContext*, const variable_list&) { not_differentiable(); }
};

std::optional<Tensor> maybe(const Tensor& t) { return t.defined() ? std::optional<Tensor>(t) : std::nullopt; }

struct Fused : Function<Fused> {
  static variable_list forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& s1,
                               const std::optional<Tensor>& s2, const Problem* p, int64_t kind, bool keep, int64_t flags) {
    FusedResult r = fused_forward((int)kind, *p, q, keep);
    // the forward state (packed inputs + bias tiles) stays alive until the backward unless the caller asked otherwise
    ctx->save_for_backward({q, k, v, s1, s2.value_or(Tensor()), r.O, r.lse, r.state});
    ctx->saved_data["kind"] = kind;
    ctx->saved_data["flags"] = flags;
    ctx->mark_non_differentiable({r.lse});
    ctx->set_materialize_grads(false);
    return {r.O, r.lse};
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    variable_list out(9);
    if (!grads[0].defined()) return out;
    const variable_list s = ctx->get_saved_variables();
    const int64_t kind = ctx->saved_data["kind"].toInt(), flags = ctx->saved_data["flags"].toInt();
    variable_list r;
    if (at::GradMode::is_enabled()) r = FusedBackward::apply(s[0], s[1], s[2], s[3], maybe(s[4]), s[5], s[6], grads[0], maybe(s[7]), kind, flags);
    else r = fused_backward((int)kind, s[0], s[1], s[2], s[3], s[4], s[5], s[6], grads[0], s[7], (int)flags);
    for (size_t i = 0; i < r.size(); ++i) out[i] = r[i];
    return out;
  }
};

// ---- stand-alone decay bias -------------------------------------------------------------------
bool describe_bias(const Tensor& k, const Tensor& src, const Tensor& dest, ua_desc& d, ua_rows& rows) {
  if (!k.is_cuda() || src.device() != k.device() || dest.device() != k.device() || k.dim() != 4 || k.numel() == 0) return false;
  if (!dtype_ok(k) || src.scalar_type() != k.scalar_type() || dest.scalar_type() != k.scalar_type()) return false;
  if (src.dim() != 3 || src.sizes() != dest.sizes() || src.sizes() != k.sizes().slice(0, 3) || k.stride(3) != 1) return false;
  if (k.size(0) * k.size(1) > kGridRows) return false;
  d = ua_desc{(int32_t)k.size(0), (int32_t)k.size(1), 1, (int32_t)k.size(2), (int32_t)k.size(3), 0, dtype_code(k), 0};
  rows = ua_rows{k.data_ptr(), k.stride(0), k.stride(1), 0, 0, k.stride(2), (int32_t)k.size(2)};
  return true;
}
size_t bias_bytes(const ua_desc& d, int bwd) {
  const size_t n = ua_affinity_workspace_bytes(&d, bwd);
  if (n == 0) throw UaFailure(std::string("unsupported problem: ") + ua_last_error());
  return n;
}
Tensor bias_forward(const Tensor& k, const Tensor& src, const Tensor& dest, const ua_desc& d, const ua_rows& rows) {
  const Tensor s = src.contiguous(), t = dest.contiguous();
  Tensor ws = bytes(bias_bytes(d, 0), k);
  Tensor aff = at::empty({d.b, d.h, d.L, d.L}, k.options());
  check(ua_affinity_fwd(&d, &rows, s.data_ptr(), t.data_ptr(), aff.data_ptr(), ws.data_ptr(), (size_t)ws.numel(), stream_of(k)), "ua_affinity_fwd");
  return aff;
}
variable_list bias_backward(const Tensor& k, const Tensor& src, const Tensor& dest, const Tensor& g) {
  ua_desc d;
  ua_rows rows;
  TORCH_CHECK(describe_bias(k, src, dest, d, rows), "the tensors saved by the forward changed");
  c10::DeviceGuard guard(k.device());
  const Tensor s = src.contiguous(), t = dest.contiguous();
  Tensor daff = g.to(k.scalar_type()).contiguous();
  if ((uintptr_t)daff.data_ptr() % 16) daff = daff.clone();      // a contiguous view at an odd offset of its storage
  Tensor ws = bytes(bias_bytes(d, 1), k);
  Tensor dk = at::empty(k.sizes(), k.options()), ds = at::empty(src.sizes(), src.options()), dd = at::empty(dest.sizes(), dest.options());
  check(ua_affinity_bwd(&d, &rows, s.data_ptr(), t.data_ptr(), daff.data_ptr(), dk.data_ptr(), ds.data_ptr(), dd.data_ptr(), ws.data_ptr(),
                        (size_t)ws.numel(), stream_of(k)), "ua_affinity_bwd");
  return {dk, ds, dd};
}
struct BiasBackward : Function<BiasBackward> {
  static variable_list forward(AutogradContext*, const Tensor& k, const Tensor& src, const Tensor& dest, const Tensor& g) { return bias_backward(k, src, dest, g); }
  static variable_list backward(AutogradContext*, const variable_list&) { not_differentiable(); }
};
struct Bias : Function<Bias> {
  static Tensor forward(AutogradContext* ctx, const Tensor& k, const Tensor& src, const Tensor& dest, const ua_desc* d, const ua_rows* rows) {
    ctx->save_for_backward({k, src, dest});
    ctx->set_materialize_grads(false);
    return bias_forward(k, src, dest, *d, *rows);
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    variable_list out(5);
    if (!grads[0].defined()) return out;
    const variable_list s = ctx->get_saved_variables();
    const variable_list r = at::GradMode::is_enabled() ? BiasBackward::apply(s[0], s[1], s[2], grads[0]) : bias_backward(s[0], s[1], s[2], grads[0]);
    for (size_t i = 0; i < 3; ++i)
      if (ctx->needs_input_grad(i)) out[i] = r[i];
    return out;
  }
};

// ---- chunked operator and merge ---------------------------------------------------------------
// [.., L, d, n] whose leading dims merge into one index (strides of size-1 dims do not matter)
bool chunked_strides(const Tensor& t, ua_chunked& c) {
  const int64_t nd = t.dim();
  if (nd < 4) return false;
  int64_t z = 0, run = 0;
  bool any = false;
  for (int64_t i = nd - 4; i >= 0; --i) {
    if (t.size(i) == 1) continue;
    if (!any) { z = t.stride(i); run = z * t.size(i); any = true; }
    else { if (t.stride(i) != run) return false; run *= t.size(i); }
  }
  if (!any) z = t.stride(nd - 3) * t.size(nd - 3);
  c = ua_chunked{t.data_ptr(), z, t.stride(nd - 3), t.stride(nd - 2), t.stride(nd - 1)};
  return true;
}
enum { KEEP_NONE = 0, KEEP_NORMALISERS = 1, KEEP_STATE = 2 };
struct ChunkOptions { int keep; bool recompute, skip_masked, contiguous_out; };
int64_t pack_options(const ChunkOptions& o) { return o.keep | (o.recompute ? 4 : 0) | (o.skip_masked ? 8 : 0) | (o.contiguous_out ? 16 : 0); }
ChunkOptions unpack_options(int64_t x) { return {(int)(x & 3), (x & 4) != 0, (x & 8) != 0, (x & 16) != 0}; }

bool describe_chunked(const Tensor& kc, const Tensor& vc, const Tensor& xq, const Tensor& src, const Tensor& dest, bool recompute, Problem& p) {
  if (!describe(UNIVERSAL, xq, kc, vc, src, dest, recompute ? UA_FLAG_RECOMPUTE : 0, p)) return false;
  p.d.chunk = (int32_t)kc.size(3);
  if ((int64_t)p.d.b * p.d.h * p.d.r * kc.size(2) > kGridRows) return false;
  // ua_fwd and ua_bwd take contiguous gates
  if (!(p.g.stride_t == 1 && p.g.stride_h == p.d.L && p.g.stride_b == (int64_t)p.d.h * p.d.L)) {
    p.src = src.reshape({p.d.b, p.d.h, p.d.L}).contiguous();
    p.dest = dest.reshape({p.d.b, p.d.h, p.d.L}).contiguous();
    p.g.src = p.src.data_ptr();
    p.g.dest = p.dest.data_ptr();
  }
  return true;
}
struct ChunkedResult { Tensor out, denom, state; };
ChunkedResult chunked_forward(const Problem& p, const Tensor& kc, const Tensor& xq, const ChunkOptions& o) {
  const ua_desc& d = p.d;
  const int64_t b = d.b, h = d.h, r = d.r, L = d.L, n = kc.size(2);
  Tensor ws = bytes(workspace_bytes(d, UA_OP_FWD), xq);
  Tensor out = o.contiguous_out ? at::empty({b, h, r, L, d.d, n}, xq.options())
                                : at::empty_strided({b, h, r, L, d.d, n}, {h * r * n * L * d.d, r * n * L * d.d, n * L * d.d, d.d, 1, L * d.d}, xq.options());
  Tensor denom = at::empty({b, h, r, L, n}, xq.options()), lse2;
  if (o.keep == KEEP_NORMALISERS) lse2 = at::empty({b * h * r * n * ((L + 127) / 128 * 128)}, xq.options().dtype(at::kFloat));
  ua_chunked oc;
  TORCH_INTERNAL_ASSERT(chunked_strides(out, oc));
  check(ua_fwd(&d, &p.k, &p.v, &p.q, p.g.src, p.g.dest, &oc, denom.data_ptr(), lse2.defined() ? lse2.data_ptr<float>() : nullptr, ws.data_ptr(),
               (size_t)ws.numel(), stream_of(xq)), "ua_fwd");
  return {out, denom, o.keep == KEEP_STATE ? ws : lse2};
}
// what the merge's backward left for exactly this (out, g_out, g_denom): the per-(row, chunk) term, or nothing
Tensor delta_from_merge(const Tensor& out, const Tensor& g_out, const Tensor& g_denom, int64_t L, int64_t n) {
  pybind11::gil_scoped_acquire gil;
  PyObject *a = THPVariable_Wrap(out), *b = THPVariable_Wrap(g_out), *c = THPVariable_Wrap(g_denom);
  PyObject* f = PyObject_GetAttrString(g_ops, "_delta_from_merge");
  PyObject* r = f ? PyObject_CallFunction(f, "OOOLL", a, b, c, (long long)L, (long long)n) : nullptr;
  Py_XDECREF(f); Py_DECREF(a); Py_DECREF(b); Py_DECREF(c);
  if (!r) throw python_error();
  Tensor t;
  if (r != Py_None) t = THPVariable_Unpack(r);
  Py_DECREF(r);
  return t;
}
variable_list chunked_backward(const Tensor& kc, const Tensor& vc, const Tensor& xq, const Tensor& src, const Tensor& dest, const Tensor& out,
                               const Tensor& g_out, const Tensor& g_denom, const Tensor& saved, const ChunkOptions& o) {
  const int64_t n = kc.size(2), c = kc.size(3), L = n * c;
  Problem p;
  TORCH_CHECK(describe_chunked(kc, vc, xq, src, dest, o.recompute, p), "the tensors saved by the forward changed");
  ua_desc& d = p.d;
  c10::DeviceGuard guard(xq.device());
  Tensor delta;
  if (c % 64 == 0) delta = delta_from_merge(out, g_out, g_denom, L, n);
  if (o.skip_masked || delta.defined()) d.flags |= UA_FLAG_SKIP_MASKED;
  Tensor state, lse2;
  if (saved.defined()) (saved.scalar_type() == at::kFloat ? lse2 : state) = saved;
  Tensor ws = bytes(workspace_bytes(d, state.defined() ? UA_OP_BWD_SCRATCH : UA_OP_BWD), xq);
  Tensor go = g_out.to(xq.scalar_type()), ot = out;
  ua_chunked oc, gc;
  if (!chunked_strides(ot, oc)) { ot = ot.contiguous(); chunked_strides(ot, oc); }
  if (!chunked_strides(go, gc)) { go = go.contiguous(); chunked_strides(go, gc); }
  // with the merge's delta the kernels do not read g_denom
  Tensor gd = delta.defined() ? g_denom : g_denom.to(at::kFloat).contiguous();
  Tensor dk = at::empty(kc.sizes(), kc.options()), dv = at::empty(vc.sizes(), vc.options()), dq = at::empty(xq.sizes(), xq.options());
  Tensor ds = at::empty(src.sizes(), src.options()), dd = at::empty(dest.sizes(), dest.options());
  check(ua_bwd(&d, &p.k, &p.v, &p.q, p.g.src, p.g.dest, &oc, &gc, (const float*)gd.data_ptr(), dk.data_ptr(), dv.data_ptr(), dq.data_ptr(),
               ds.data_ptr(), dd.data_ptr(), delta.defined() ? delta.data_ptr<float>() : nullptr, lse2.defined() ? lse2.data_ptr<float>() : nullptr,
               state.defined() ? state.data_ptr() : nullptr, ws.data_ptr(), (size_t)ws.numel(), stream_of(xq)), "ua_bwd");
  return {dk, dv, dq, ds, dd};
}
struct ChunkedBackward : Function<ChunkedBackward> {
  static variable_list forward(AutogradContext*, const Tensor& kc, const Tensor& vc, const Tensor& xq, const Tensor& src, const Tensor& dest,
                               const Tensor& out, const Tensor& g_out, const Tensor& g_denom, const std::optional<Tensor>& saved, int64_t opts) {
    return chunked_backward(kc, vc, xq, src, dest, out, g_out, g_denom, saved.value_or(Tensor()), unpack_options(opts));
  }
  static variable_list backward(AutogradContext*, const variable_list&) { not_differentiable(); }
};
struct Chunked : Function<Chunked> {
  static variable_list forward(AutogradContext* ctx, const Tensor& kc, const Tensor& vc, const Tensor& xq, const Tensor& src, const Tensor& dest,
                               const Problem* p, int64_t opts) {
    ChunkedResult r = chunked_forward(*p, kc, xq, unpack_options(opts));
    // `out` is the tensor the caller holds anyway: saving it costs no memory
    ctx->save_for_backward({kc, vc, xq, src, dest, r.out, r.state});
    ctx->saved_data["opts"] = opts;
    ctx->set_materialize_grads(false);
    return {r.out, r.denom};
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    variable_list res(7);
    if (!grads[0].defined() && !grads[1].defined()) return res;
    const variable_list s = ctx->get_saved_variables();
    const int64_t opts = ctx->saved_data["opts"].toInt();
    const Tensor& out = s[5];
    const Tensor g_out = grads[0].defined() ? grads[0] : at::zeros_like(out);
    const Tensor g_denom = grads[1].defined() ? grads[1] : at::zeros({out.size(0), out.size(1), out.size(2), out.size(3), out.size(5)}, out.options());
    const variable_list r = at::GradMode::is_enabled()
        ? ChunkedBackward::apply(s[0], s[1], s[2], s[3], s[4], out, g_out, g_denom, maybe(s[6]), opts)
        : chunked_backward(s[0], s[1], s[2], s[3], s[4], out, g_out, g_denom, s[6], unpack_options(opts));
    for (size_t i = 0; i < 5; ++i) res[i] = r[i];
    return res;
  }
};

bool merge_ok(const Tensor& mat, const Tensor& vec, ua_chunked& c) {
  if (!mat.is_cuda() || vec.device() != mat.device() || mat.dim() < 4 || mat.numel() == 0 || !dtype_ok(mat) || vec.scalar_type() != mat.scalar_type()) return false;
  const int64_t nd = mat.dim();
  return vec.dim() == nd - 1 && vec.sizes().slice(0, nd - 2) == mat.sizes().slice(0, nd - 2) && vec.size(nd - 2) == mat.size(nd - 1) && chunked_strides(mat, c);
}
Tensor merge_forward(const Tensor& mat, const Tensor& vec, const ua_chunked& c) {
  const int64_t nd = mat.dim(), L = mat.size(nd - 3), d = mat.size(nd - 2), n = mat.size(nd - 1), rows = vec.numel() / n;
  const Tensor v = vec.contiguous();
  Tensor res = at::empty(mat.sizes().slice(0, nd - 1), mat.options());
  check(ua_merge_fwd(dtype_code(mat), rows, (int32_t)L, (int32_t)d, (int32_t)n, &c, v.data_ptr(), res.data_ptr(), stream_of(mat)), "ua_merge_fwd");
  return res;
}
variable_list merge_backward(const Tensor& mat, const Tensor& vec, const Tensor& grad) {
  ua_chunked c;
  TORCH_CHECK(merge_ok(mat, vec, c), "the tensors saved by the forward changed");
  c10::DeviceGuard guard(mat.device());
  const int64_t nd = mat.dim(), L = mat.size(nd - 3), d = mat.size(nd - 2), n = mat.size(nd - 1), rows = vec.numel() / n, Z = rows / L;
  const Tensor v = vec.contiguous(), g = grad.to(mat.scalar_type()).contiguous();
  // chunk-major storage: the gradient is consumed chunk by chunk by the chunked backward
  std::vector<int64_t> strides(nd);
  strides[nd - 1] = L * d; strides[nd - 2] = 1; strides[nd - 3] = d;
  int64_t run = n * L * d;
  for (int64_t i = nd - 4; i >= 0; --i) { strides[i] = run; run *= mat.size(i); }
  Tensor d_mat = at::empty_strided(mat.sizes(), strides, mat.options()), d_vec = at::empty(vec.sizes(), vec.options()), delta;
  const ua_chunked dc{d_mat.data_ptr(), n * L * d, d, 1, L * d};
  // the per-(row, chunk) term is only worth keeping where a chunked backward can take it: chunks that are a multiple of 64
  const int64_t Lp = (L + 127) / 128 * 128;
  if (L % n == 0 && (L / n) % 64 == 0)
    delta = Lp == L ? at::empty({Z, n, Lp}, mat.options().dtype(at::kFloat)) : at::zeros({Z, n, Lp}, mat.options().dtype(at::kFloat));
  check(ua_merge_bwd(dtype_code(mat), rows, (int32_t)L, (int32_t)d, (int32_t)n, &c, v.data_ptr(), g.data_ptr(), &dc, d_vec.data_ptr(),
                     delta.defined() ? delta.data_ptr<float>() : nullptr, stream_of(mat)), "ua_merge_bwd");
  if (delta.defined()) {
    pybind11::gil_scoped_acquire gil;
    PyObject *a = THPVariable_Wrap(d_mat), *b = THPVariable_Wrap(d_vec), *m = THPVariable_Wrap(mat), *x = THPVariable_Wrap(delta);
    PyObject* f = PyObject_GetAttrString(g_ops, "_leave_note");
    PyObject* r = f ? PyObject_CallFunctionObjArgs(f, a, b, m, x, nullptr) : nullptr;
    Py_XDECREF(f); Py_DECREF(a); Py_DECREF(b); Py_DECREF(m); Py_DECREF(x);
    if (!r) throw python_error();
    Py_DECREF(r);
  }
  return {d_mat, d_vec};
}
struct MergeBackward : Function<MergeBackward> {
  static variable_list forward(AutogradContext*, const Tensor& mat, const Tensor& vec, const Tensor& g) { return merge_backward(mat, vec, g); }
  static variable_list backward(AutogradContext*, const variable_list&) { not_differentiable(); }
};
struct Merge : Function<Merge> {
  static Tensor forward(AutogradContext* ctx, const Tensor& mat, const Tensor& vec, const ua_chunked* c) {
    ctx->save_for_backward({mat, vec});
    ctx->set_materialize_grads(false);
    return merge_forward(mat, vec, *c);
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    variable_list out(3);
    if (!grads[0].defined()) return out;
    const variable_list s = ctx->get_saved_variables();
    const variable_list r = at::GradMode::is_enabled() ? MergeBackward::apply(s[0], s[1], grads[0]) : merge_backward(s[0], s[1], grads[0]);
    out[0] = r[0];
    out[1] = r[1];
    return out;
  }
};

// ---- module -----------------------------------------------------------------------------------
// plain tensors (or parameters), no function transform and no dispatch mode active
bool plain(PyObject* const* args, Py_ssize_t n) {
  for (Py_ssize_t i = 0; i < n; ++i)
    if (!THPVariable_CheckExact(args[i])) return false;
  return !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) && !c10::impl::TorchDispatchModeTLS::any_modes_set();
}
template <class... Ts> bool recorded(const Ts&... t) { return at::GradMode::is_enabled() && (t.requires_grad() || ...); }
struct NoGil {
  PyThreadState* s = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(s); }
};
template <class F> PyObject* guarded(F f) {
  HANDLE_TH_ERRORS
  try {
    return f();
  } catch (const UaFailure& e) {
    PyErr_SetString(g_error ? g_error : PyExc_RuntimeError, e.what());
    return nullptr;
  }
  END_HANDLE_TH_ERRORS
}
PyObject* pair(const Tensor& a, const Tensor& b) {
  PyObject* t = PyTuple_New(2);
  PyTuple_SET_ITEM(t, 0, THPVariable_Wrap(a));
  PyTuple_SET_ITEM(t, 1, THPVariable_Wrap(b));
  return t;
}

// (q, k, v, s1, s2 or None), flags, keep_state
PyObject* run_fused(int kind, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& s1, const Tensor& s2, bool prune, bool recompute, bool keep_state) {
  const int flags = (prune ? UA_FLAG_PRUNE : 0) | (recompute ? UA_FLAG_RECOMPUTE : 0);
  Problem p;
  Tensor O, lse;
  bool taken;
  {
    NoGil nogil;
    c10::DeviceGuard guard(q.device());
    taken = describe(kind, q, k, v, s1, s2, flags, p);
    if (taken) {
      const bool rec = recorded(q, k, v, s1) || (s2.defined() && recorded(s2)), keep = keep_state && !recompute && rec;
      if (!keep) p.d.flags |= UA_FLAG_FORWARD_ONLY;
      if (rec) {
        variable_list r = Fused::apply(q, k, v, s1, maybe(s2), (const Problem*)&p, (int64_t)kind, keep, (int64_t)flags);
        O = r[0]; lse = r[1];
      } else {
        FusedResult r = fused_forward(kind, p, q, false);
        O = r.O; lse = r.lse;
      }
    }
  }
  if (!taken) Py_RETURN_NONE;
  return pair(O, lse);
}
// universal(kc, vc, xq, src, dest, prune, recompute, keep_state) -> (O, lse) or None
PyObject* py_universal(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    if (n != 8 || !plain(a, 5)) Py_RETURN_NONE;
    return run_fused(UNIVERSAL, THPVariable_Unpack(a[2]), THPVariable_Unpack(a[0]), THPVariable_Unpack(a[1]), THPVariable_Unpack(a[3]), THPVariable_Unpack(a[4]),
                     PyObject_IsTrue(a[5]) == 1, PyObject_IsTrue(a[6]) == 1, PyObject_IsTrue(a[7]) == 1);
  });
}
// decoder(q, k, v, static, prune, recompute) -> (O, lse) or None
PyObject* py_decoder(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    if (n != 6 || !plain(a, 4)) Py_RETURN_NONE;
    return run_fused(DECODER, THPVariable_Unpack(a[0]), THPVariable_Unpack(a[1]), THPVariable_Unpack(a[2]), THPVariable_Unpack(a[3]), Tensor(),
                     PyObject_IsTrue(a[4]) == 1, PyObject_IsTrue(a[5]) == 1, true);
  });
}
// gen2(q, k, v, src, dest, keep_state) -> (O, lse) or None
PyObject* py_gen2(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    if (n != 6 || !plain(a, 5)) Py_RETURN_NONE;
    return run_fused(GEN2, THPVariable_Unpack(a[0]), THPVariable_Unpack(a[1]), THPVariable_Unpack(a[2]), THPVariable_Unpack(a[3]), THPVariable_Unpack(a[4]), false,
                     false, PyObject_IsTrue(a[5]) == 1);
  });
}
// bias(k, src, dest) -> aff or None
PyObject* py_bias(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    if (n != 3 || !plain(a, 3)) Py_RETURN_NONE;
    const Tensor &k = THPVariable_Unpack(a[0]), &s = THPVariable_Unpack(a[1]), &d = THPVariable_Unpack(a[2]);
    ua_desc desc;
    ua_rows rows;
    Tensor aff;
    {
      NoGil nogil;
      c10::DeviceGuard guard(k.device());
      if (describe_bias(k, s, d, desc, rows))
        aff = recorded(k, s, d) ? Bias::apply(k, s, d, (const ua_desc*)&desc, (const ua_rows*)&rows) : bias_forward(k, s, d, desc, rows);
    }
    if (!aff.defined()) Py_RETURN_NONE;
    return THPVariable_Wrap(aff);
  });
}
// chunked(kc, vc, xq, src, dest, keep (0 nothing, 1 normalisers, 2 state), recompute, skip_masked, contiguous_out) -> (out, denom) or None
PyObject* py_chunked(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    if (n != 9 || !plain(a, 5)) Py_RETURN_NONE;
    const Tensor &kc = THPVariable_Unpack(a[0]), &vc = THPVariable_Unpack(a[1]), &xq = THPVariable_Unpack(a[2]), &s = THPVariable_Unpack(a[3]), &d = THPVariable_Unpack(a[4]);
    ChunkOptions o{(int)PyLong_AsLong(a[5]), PyObject_IsTrue(a[6]) == 1, PyObject_IsTrue(a[7]) == 1, PyObject_IsTrue(a[8]) == 1};
    Tensor out, denom;
    {
      NoGil nogil;
      c10::DeviceGuard guard(kc.device());
      Problem p;
      if (describe_chunked(kc, vc, xq, s, d, o.recompute, p)) {
        if (recorded(kc, vc, xq, s, d)) {
          variable_list r = Chunked::apply(kc, vc, xq, s, d, (const Problem*)&p, pack_options(o));
          out = r[0]; denom = r[1];
        } else {
          o.keep = KEEP_NONE;
          ChunkedResult r = chunked_forward(p, kc, xq, o);
          out = r.out; denom = r.denom;
        }
      }
    }
    if (!out.defined()) Py_RETURN_NONE;
    return pair(out, denom);
  });
}
// merge(mat, vec) -> result or None
PyObject* py_merge(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    if (n != 2 || !plain(a, 2)) Py_RETURN_NONE;
    const Tensor &mat = THPVariable_Unpack(a[0]), &vec = THPVariable_Unpack(a[1]);
    Tensor res;
    {
      NoGil nogil;
      c10::DeviceGuard guard(mat.device());
      ua_chunked c;
      if (merge_ok(mat, vec, c)) res = recorded(mat, vec) ? Merge::apply(mat, vec, (const ua_chunked*)&c) : merge_forward(mat, vec, c);
    }
    if (!res.defined()) Py_RETURN_NONE;
    return THPVariable_Wrap(res);
  });
}
// init(UaError, ops)
PyObject* py_init(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 2) { PyErr_SetString(PyExc_TypeError, "init(UaError, ops)"); return nullptr; }
  Py_INCREF(a[0]); Py_INCREF(a[1]);
  g_error = a[0];
  g_ops = a[1];
  Py_RETURN_NONE;
}
PyObject* py_source_hash(PyObject*, PyObject* const*, Py_ssize_t) { return PyUnicode_FromString(UA_SOURCE_HASH); }

#define UA_METHOD(name) {#name, (PyCFunction)(void*)py_##name, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {UA_METHOD(universal), UA_METHOD(decoder), UA_METHOD(gen2), UA_METHOD(bias), UA_METHOD(chunked), UA_METHOD(merge),
                         UA_METHOD(init), UA_METHOD(source_hash), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_ua_host", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__ua_host(void) { return PyModule_Create(&module_def); }
