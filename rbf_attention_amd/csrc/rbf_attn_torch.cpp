// Native eager path of the Python wrappers (run_triton_rbf,
// run_triton_non_softmax_rbf, rbf_decode): argument preparation, allocation,
// the C-ABI calls and the autograd node, without Python between them.
//
// In Python an autograd.Function's backward runs on the autograd engine's
// device thread and has to win the GIL from the thread that waits for it.  With
// the wrappers' glue this came to 140 us of host time per forward + backward
// (20 us of it the forward), against 75-90 us of GPU work for B4 H8 N1024 or
// B32 H8 N516 (D = 64).  The results are those of the registered ops: same
// kernels, same layouts, same formula for the position term.
//
// Each entry point returns None for arguments it does not take (wrong shapes,
// types, devices, bandwidths ...); the caller then goes through the registered
// ops, whose checks raise.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <algorithm>
#include <cmath>
#include <tuple>
#include <vector>

#include <ATen/ATen.h>
#include <ATen/TensorSubclassLikeUtils.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/DeviceGuard.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/graph_task.h>
#include <torch/csrc/autograd/python_cpp_function.h>
#include <torch/csrc/autograd/python_variable.h>

#include "rbf_attn.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::Variable;
using torch::autograd::variable_list;

int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kBFloat16: return RBF_ATTN_BF16;
    case at::kHalf: return RBF_ATTN_FP16;
    case at::kFloat: return RBF_ATTN_FP32;
    default: return -1;
  }
}

int64_t padded_dim(int64_t d) { return d <= 8 ? 8 : (d + 7) / 8 * 8; }

// The C ABI's layout contract: unit last stride, 16-byte aligned base and
// strides, head dim a multiple of 8, the values in memory (no negative bit, no
// tensor of implied zeros).  Copies only when needed.
Tensor prep(const Tensor& t, int64_t dp) {
  const int64_t d = t.size(3);
  if (dp != d) return at::constant_pad_nd(t, {0, dp - d});
  if (t.is_neg() || t._is_zerotensor()) return t.clone(at::MemoryFormat::Contiguous);
  const bool base = reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
  if (base && t.is_contiguous()) return t;
  const int64_t es = t.element_size();
  const bool ok = base && t.stride(3) == 1 && t.stride(0) * es % 16 == 0 && t.stride(1) * es % 16 == 0 &&
                  t.stride(2) * es % 16 == 0;
  return ok ? t : t.clone(at::MemoryFormat::Contiguous);
}

// Descriptor of a (B, H, N, D) tensor; the stride of a dimension of size 1 is
// never used and is passed as 0 (torch gives such dimensions any stride).
rbf_attn_tensor desc(const Tensor& t) {
  auto s = [&](int i) { return t.size(i) != 1 ? t.stride(i) : 0; };
  return {t.data_ptr(), s(0), s(1), s(2)};
}

void* current_stream(const at::Device& dev) {
  return static_cast<void*>(c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(dev.index()).stream());
}

// Python objects of the ops layer, set once, at load (configure): the error class
// of failed library calls, and the launcher of calls with a fused position term
// (ops._launch_pos_bytes: entry point's name, args as bytes, term), the one place
// where such calls can be observed from Python.
PyObject* error_class = nullptr;
PyObject* pos_launcher = nullptr;

// Throws the pending Python error, kept in the exception (it may be caught on
// another thread, or after the GIL was released).  With the GIL held.
[[noreturn]] void throw_python_error() {
  python_error e;
  e.persist();
  throw e;
}

// A failed library call raises _lib.RbfAttnError(code, message).
void check_rc(int rc) {
  if (rc == 0) return;
  const pybind11::gil_scoped_acquire gil;
  TORCH_CHECK(error_class != nullptr, "librbfattn: ", rc, ": ", rbf_attn_last_error());
  if (PyObject* e = PyObject_CallFunction(error_class, "is", rc, rbf_attn_last_error())) {
    PyErr_SetObject(error_class, e);
    Py_DECREF(e);
  }
  throw_python_error();
}

struct Call {
  bool softmax, causal, token_major;
  double scale;
  int64_t num_prefix;
};

rbf_attn_args base_args(const Call& c, const Tensor& q, int64_t dp) {
  rbf_attn_args a = {};
  a.abi_version = RBF_ATTN_ABI_VERSION;
  a.variant = c.softmax ? RBF_ATTN_SOFTMAX : RBF_ATTN_NON_SOFTMAX;
  a.dtype = dtype_code(q.scalar_type());
  a.B = (int32_t)q.size(0);
  a.H = (int32_t)q.size(1);
  a.N = (int32_t)q.size(2);
  a.D = (int32_t)dp;
  a.causal = c.causal ? 1 : 0;
  a.num_prefix = (int32_t)c.num_prefix;
  a.gamma = (float)c.scale;
  return a;
}

// Position term of a call: fused (kept in pos) where the library fuses it for
// these args, else added to q and k here, each sum rounded to the element type.
void place_pos(const rbf_attn_args& a, Tensor& q, Tensor& k, Tensor& pos, int64_t dp) {
  if (!pos.defined()) return;
  if (rbf_attn_pos_supported(&a) == 1) {
    pos = prep(pos, dp);
  } else {
    q = q + pos;
    k = k + pos;
    pos = Tensor();
  }
}

void launch_pos(const char* name, const rbf_attn_args& a, const Tensor& pos) {
  const pybind11::gil_scoped_acquire gil;
  TORCH_CHECK(pos_launcher != nullptr, "rbf_attn: the position term's launcher is not set");
  PyObject* t = THPVariable_Wrap(pos);
  PyObject* r = PyObject_CallFunction(pos_launcher, "sy#N", name, reinterpret_cast<const char*>(&a), (Py_ssize_t)sizeof(a), t);
  if (r == nullptr) throw_python_error();
  Py_DECREF(r);
}

void launch(int (*plain)(const rbf_attn_args*, void*), const char* with_pos, const rbf_attn_args& a, const Tensor& pos,
            const at::Device& dev) {
  if ((int64_t)a.B * a.H * a.N == 0) return;  // nothing to compute (data pointers may be null)
  if (pos.defined()) launch_pos(with_pos, a, pos);
  else check_rc(plain(&a, current_stream(dev)));
}

Tensor unpad(const Tensor& t, int64_t d) { return t.size(3) == d ? t : t.slice(3, 0, d).contiguous(); }

// (out, L); L undefined without the normaliser.
std::tuple<Tensor, Tensor> forward(Tensor q, Tensor k, const Tensor& v, Tensor pos, const Call& c) {
  const c10::OptionalDeviceGuard guard(q.device());
  const int64_t B = q.size(0), H = q.size(1), N = q.size(2), D = q.size(3), dp = padded_dim(D);
  rbf_attn_args a = base_args(c, q, dp);
  place_pos(a, q, k, pos, dp);
  const Tensor q_ = prep(q, dp), k_ = prep(k, dp), v_ = prep(v, dp);
  const Tensor out = c.token_major && dp == D ? at::empty({B, N, H, dp}, q.options()).transpose(1, 2)
                                              : at::empty({B, H, N, dp}, q.options());
  Tensor L;
  a.q = desc(q_);
  a.k = desc(k_);
  a.v = desc(v_);
  a.o = desc(out);
  if (c.softmax) {
    L = at::empty({B, H, N}, q.options().dtype(at::kFloat));
    a.lse = L.data_ptr<float>();
  }
  launch(rbf_attn_fwd, "rbf_attn_fwd_pos", a, pos, q.device());
  return {unpad(out, D), L};
}

// dq, dk, dv.  packed: the gradient of q, k and v as one (B, N, 3, H, D) tensor
// (D a multiple of 8), of which the three returned are views.
std::tuple<Tensor, Tensor, Tensor> backward(Tensor q, Tensor k, const Tensor& v, const Tensor& out, const Tensor& L,
                                            const Tensor& dout, Tensor pos, const Call& c, const Tensor& packed = Tensor()) {
  const c10::OptionalDeviceGuard guard(q.device());
  const int64_t B = q.size(0), H = q.size(1), N = q.size(2), D = q.size(3), dp = padded_dim(D);
  rbf_attn_args a = base_args(c, q, dp);
  place_pos(a, q, k, pos, dp);
  const Tensor q_ = prep(q, dp), k_ = prep(k, dp), v_ = prep(v, dp), do_ = prep(dout, dp);
  const Tensor o_ = c.softmax ? prep(out, dp) : Tensor();
  const Tensor rows = at::empty({B, H, N}, q.options().dtype(at::kFloat));
  const auto grad = [&](int64_t i) {
    return packed.defined() ? packed.select(2, i).transpose(1, 2) : at::empty({B, H, N, dp}, q.options());
  };
  const Tensor dq = grad(0), dk = grad(1), dv = grad(2);
  a.q = desc(q_);
  a.k = desc(k_);
  a.v = desc(v_);
  a.dout = desc(do_);
  a.dq = desc(dq);
  a.dk = desc(dk);
  a.dv = desc(dv);
  if (c.softmax) {
    a.o = desc(o_);
    a.lse = L.data_ptr<float>();
    a.delta = rows.data_ptr<float>();
  } else {
    a.lse = rows.data_ptr<float>();
  }
  launch(rbf_attn_bwd, "rbf_attn_bwd_pos", a, pos, q.device());
  return {unpad(dq, D), unpad(dk, D), unpad(dv, D)};
}

// The packed (B, N, 3, H, D) tensor of which q, k and v, in this order, are the
// (B, H, N, D) views; undefined if they are not, or if anything else refers to
// their memory (a gradient that a hook kept, that autograd.grad returns, or a
// view of one): a gradient is never shared with another.
Tensor packed_of(const Tensor& q, const Tensor& k, const Tensor& v) {
  if (!q.defined() || !k.defined() || !v.defined() || q.dim() != 4 || k.sizes() != q.sizes() || v.sizes() != q.sizes() ||
      !q.is_alias_of(k) || !q.is_alias_of(v) || k.scalar_type() != q.scalar_type() || v.scalar_type() != q.scalar_type() ||
      q.use_count() != 1 || k.use_count() != 1 || v.use_count() != 1 || q.storage().use_count() != 3)
    return Tensor();
  const int64_t B = q.size(0), H = q.size(1), N = q.size(2), D = q.size(3);
  const int64_t strides[4] = {N * 3 * H * D, D, 3 * H * D, 1};
  if (q.strides() != at::IntArrayRef(strides) || k.strides() != q.strides() || v.strides() != q.strides() ||
      k.storage_offset() != q.storage_offset() + H * D || v.storage_offset() != q.storage_offset() + 2 * H * D)
    return Tensor();
  return q.as_strided({B, N, 3, H, D}, {N * 3 * H * D, 3 * H * D, H * D, D, 1}, q.storage_offset());
}

// q, k, v as (B, H, N, D) views of the model projection's (B, N, 3, H, D) output.
// Autograd of select or unbind stacks the three gradients and then copies the
// stack to this layout for the projection's backward (38 + 37 us of a 670 us
// module step at B32 N516 H8 D64); this node's backward returns the packed
// tensor itself when the attention's backward wrote the three into one (below)
// and they are referred to nowhere else, and else copies each into its place.
struct UnpackFunction : torch::autograd::Function<UnpackFunction> {
  static variable_list forward(AutogradContext* ctx, const Variable& qkv) {
    ctx->saved_data["sizes"] = qkv.sizes().vec();
    const auto view = [&](int64_t i) { return qkv.select(2, i).transpose(1, 2); };
    return {view(0), view(1), view(2)};
  }

  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    const auto first = std::find_if(grads.begin(), grads.end(), [](const Tensor& g) { return g.defined(); });
    if (first == grads.end()) return {Variable()};
    // create_graph (a gradient that has a graph of its own), or gradients of
    // another kind than the attention's (batched by vmap, subclasses)
    if (at::GradMode::is_enabled() || std::any_of(grads.begin(), grads.end(), [](const Tensor& g) {
          return g.defined() && at::isTensorSubclassLike(g);
        })) {
      std::vector<Tensor> parts;
      for (const Tensor& g : grads) parts.push_back((g.defined() ? g : at::zeros_like(*first)).transpose(1, 2));
      return {at::stack(parts, 2)};
    }
    Tensor packed = packed_of(grads[0], grads[1], grads[2]);
    if (packed.defined()) return {packed};
    packed = at::empty(ctx->saved_data["sizes"].toIntVector(), first->options());
    for (int64_t i = 0; i < 3; ++i) {
      Tensor slot = packed.select(2, i).transpose(1, 2);
      if (grads[i].defined()) slot.copy_(grads[i]);
      else slot.zero_();
    }
    return {packed};
  }
};

// Whether the gradients of q, k and v go to one UnpackFunction that will use them
// up, so that a packed tensor of the three pays: q, k and v are its outputs, this
// backward pass runs it, and no hook and no autograd.grad asks for them there (a
// dq that is kept would keep the memory of all three).
bool pack_gradients(const Tensor& q, const Tensor& k, const Tensor& v) {
  if (!q.requires_grad() || !k.requires_grad() || !v.requires_grad()) return false;
  const auto& f = q.grad_fn();
  if (!f || f != k.grad_fn() || f != v.grad_fn() || q.output_nr() != 0 || k.output_nr() != 1 || v.output_nr() != 2 ||
      dynamic_cast<torch::autograd::CppNode<UnpackFunction>*>(f.get()) == nullptr)
    return false;
  if (!f->pre_hooks().empty() || !f->tensor_pre_hooks().empty() || !f->retains_grad_hooks().empty()) return false;
  const auto* info = torch::autograd::get_current_graph_task_exec_info();
  if (info == nullptr || info->empty()) return true;  // a pass that runs every node
  const auto it = info->find(f.get());
  return it != info->end() && it->second.needed_ && !it->second.captures_;
}

bool like(const Tensor& t, const Tensor& q) {
  return t.scalar_type() == q.scalar_type() && t.device() == q.device();
}

// What the backward pass reads, as the registered backward ops check it: the
// saved tensors may have gone through a program's saved-tensor hooks, which can
// bring them back in another shape, type or place.
void check_saved(const Tensor& q, const variable_list& others, const Tensor& pos, const Tensor& L) {
  TORCH_CHECK_VALUE(q.dim() == 4 && q.size(3) <= 256, "scaled_bwd: expected (B, H, N, D) tensors, got q of shape ", q.sizes());
  TORCH_CHECK_TYPE(dtype_code(q.scalar_type()) >= 0, "scaled_bwd: unsupported dtype ", q.scalar_type());
  TORCH_CHECK(q.is_cuda(), "scaled_bwd: the RBF attention kernels run only on a ROCm GPU, tensors are on ", q.device());
  const auto check = [&](const Tensor& t, at::IntArrayRef sizes, at::ScalarType type) {
    TORCH_CHECK_VALUE(t.sizes() == sizes, "scaled_bwd: shape mismatch ", t.sizes(), " vs ", sizes);
    TORCH_CHECK_TYPE(t.scalar_type() == type, "scaled_bwd: dtype mismatch ", t.scalar_type(), " vs ", type);
    TORCH_CHECK_VALUE(t.device() == q.device(), "scaled_bwd: device mismatch ", t.device(), " vs ", q.device());
  };
  for (const Tensor& t : others) check(t, q.sizes(), q.scalar_type());
  if (L.defined()) check(L, q.sizes().slice(0, 3), at::kFloat);
  if (pos.defined()) {
    const int64_t sizes[4] = {pos.dim() == 4 && pos.size(0) == 1 ? 1 : q.size(0), q.size(1), q.size(2), q.size(3)};
    check(pos, sizes, q.scalar_type());
  }
}

struct RbfAttentionFunction : torch::autograd::Function<RbfAttentionFunction> {
  static Variable forward(AutogradContext* ctx, const Variable& q, const Variable& k, const Variable& v,
                          const std::optional<Variable>& pos, bool softmax, bool causal, double scale, int64_t num_prefix,
                          bool token_major) {
    const Call c = {softmax, causal, token_major, scale, num_prefix};
    const Tensor p = pos.has_value() ? *pos : Tensor();
    auto [out, L] = ::forward(q, k, v, p, c);
    if (softmax) ctx->save_for_backward({q, k, v, p, out, L});
    else ctx->save_for_backward({q, k, v, p});
    ctx->saved_data["softmax"] = softmax;
    ctx->saved_data["causal"] = causal;
    ctx->saved_data["scale"] = scale;
    ctx->saved_data["num_prefix"] = num_prefix;
    return out;
  }

  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    const Call c = {ctx->saved_data["softmax"].toBool(), ctx->saved_data["causal"].toBool(), false,
                    ctx->saved_data["scale"].toDouble(), ctx->saved_data["num_prefix"].toInt()};
    const variable_list s = ctx->get_saved_variables();
    const Tensor& q = s[0];
    variable_list others = {s[1], s[2], grads[0]};
    if (c.softmax) others.push_back(s[4]);
    check_saved(q, others, s[3], c.softmax ? s[5] : Tensor());
    const bool pack = q.size(3) % 8 == 0 && pack_gradients(q, s[1], s[2]);
    // As the registered backward ops: the result carries no graph of its own, and
    // the views of a packed tensor no record of their base.
    const at::AutoDispatchBelowADInplaceOrView below_autograd;
    Tensor packed;
    if (pack)
      packed = at::empty({q.size(0), q.size(2), 3, q.size(1), q.size(3)}, q.options());
    auto [dq, dk, dv] =
        ::backward(q, s[1], s[2], c.softmax ? s[4] : Tensor(), c.softmax ? s[5].contiguous() : Tensor(), grads[0], s[3], c, packed);
    Tensor dpos;
    if (s[3].defined()) {
      dpos = at::empty(dq.sizes(), dq.options());
      at::add_out(dpos, dq, dk);
      if (s[3].size(0) == 1 && dpos.size(0) != 1) dpos = dpos.sum(0, /*keepdim=*/true);
    }
    return {dq, dk, dv, dpos, Variable(), Variable(), Variable(), Variable(), Variable()};
  }
};

bool takes_dims(const Tensor& q) {
  return q.dim() == 4 && q.is_cuda() && dtype_code(q.scalar_type()) >= 0 && q.size(3) >= 1 && q.size(3) <= 256;
}
// a position term (1 or B, H, N, D) of q's type and device
bool takes_pos(const Tensor& p, const Tensor& q) {
  return p.dim() == 4 && like(p, q) && p.size(1) == q.size(1) && p.size(2) == q.size(2) && p.size(3) == q.size(3) &&
         (p.size(0) == 1 || p.size(0) == q.size(0));
}
// sizes, bandwidth and prefix within what the C ABI accepts
bool takes_scale(double scale);
bool takes_call(const Tensor& q, double scale, long long num_prefix) {
  return takes_scale(scale) && num_prefix >= 0 && num_prefix <= INT32_MAX && q.size(2) <= (1 << 30) &&
         q.size(0) <= INT32_MAX && q.size(1) <= INT32_MAX &&
         (double)q.size(0) * q.size(1) * ((q.size(2) + 31) / 32 + 4) < 2147483647.0 * 4;
}
bool takes_scale(double scale) { return std::isfinite((float)scale) && (float)scale > 0.f; }

const Tensor& unpack(PyObject* o) { return THPVariable_Unpack(o); }

// attention(q, k, v, pos | None, softmax, causal, scale, num_prefix, token_major)
PyObject* attention(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK(n == 9, "attention: 9 arguments");
  for (int i = 0; i < 3; ++i)
    if (!THPVariable_Check(args[i])) Py_RETURN_NONE;
  const Tensor &q = unpack(args[0]), &k = unpack(args[1]), &v = unpack(args[2]);
  if (!takes_dims(q) || !like(k, q) || !like(v, q) || k.sizes() != q.sizes() || v.sizes() != q.sizes()) Py_RETURN_NONE;
  std::optional<Variable> pos;
  if (args[3] != Py_None) {
    if (!THPVariable_Check(args[3])) Py_RETURN_NONE;
    if (!takes_pos(unpack(args[3]), q)) Py_RETURN_NONE;
    pos = unpack(args[3]);
  }
  const bool softmax = args[4] == Py_True, causal = args[5] == Py_True, token_major = args[8] == Py_True;
  const double scale = PyFloat_AsDouble(args[6]);
  const long long num_prefix = PyLong_AsLongLong(args[7]);
  if (PyErr_Occurred()) return nullptr;
  if (!takes_call(q, scale, num_prefix)) Py_RETURN_NONE;
  Tensor out;
  {
    const pybind11::gil_scoped_release no_gil;
    out = RbfAttentionFunction::apply(q, k, v, pos, softmax, causal, scale, (int64_t)num_prefix, token_major);
  }
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// unpack_qkv(qkv) -> (q, k, v)
PyObject* unpack_qkv(PyObject*, PyObject* o) {
  HANDLE_TH_ERRORS
  if (!THPVariable_Check(o)) Py_RETURN_NONE;
  const Tensor& qkv = unpack(o);
  if (qkv.dim() != 5 || qkv.size(2) != 3 || !qkv.is_contiguous()) Py_RETURN_NONE;
  if (qkv._fw_grad(/*level=*/0).defined()) Py_RETURN_NONE;  // forward mode: plain views have it
  const variable_list v = UnpackFunction::apply(qkv);
  PyObject* r = PyTuple_New(3);
  if (r == nullptr) return nullptr;
  for (int i = 0; i < 3; ++i) PyTuple_SET_ITEM(r, i, THPVariable_Wrap(v[i]));
  return r;
  END_HANDLE_TH_ERRORS
}

// decode(q, k_cache, v_cache, cache_lens | None, softmax, scale) -> (out, L)
PyObject* decode(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK(n == 6, "decode: 6 arguments");
  for (int i = 0; i < 3; ++i)
    if (!THPVariable_Check(args[i])) Py_RETURN_NONE;
  const Tensor &q = unpack(args[0]), &k = unpack(args[1]), &v = unpack(args[2]);
  if (!takes_dims(q) || k.dim() != 4 || v.dim() != 4 || !like(k, q) || !like(v, q) || k.sizes() != v.sizes()) Py_RETURN_NONE;
  const int64_t B = q.size(0), H = q.size(1), T = q.size(2), D = q.size(3), L = k.size(2), dp = padded_dim(D);
  if (k.size(0) != B || k.size(1) != H || k.size(3) != D || T < 1 || T > 32 || L < T || B * H == 0) Py_RETURN_NONE;
  Tensor lens;
  if (args[3] != Py_None) {
    if (!THPVariable_Check(args[3])) Py_RETURN_NONE;
    lens = unpack(args[3]);
    if (lens.dim() != 1 || lens.size(0) != B) Py_RETURN_NONE;
  }
  const bool softmax = args[4] == Py_True;
  const double scale = PyFloat_AsDouble(args[5]);
  if (PyErr_Occurred()) return nullptr;
  rbf_attn_decode_args a = {};
  a.abi_version = RBF_ATTN_ABI_VERSION;
  a.variant = softmax ? RBF_ATTN_SOFTMAX : RBF_ATTN_NON_SOFTMAX;
  a.dtype = dtype_code(q.scalar_type());
  if (!takes_scale(scale) || B > INT32_MAX || H > INT32_MAX || L > (1 << 30)) Py_RETURN_NONE;
  a.B = (int32_t)B;
  a.H = (int32_t)H;
  a.T = (int32_t)T;
  a.D = (int32_t)dp;
  a.L = (int32_t)L;
  a.gamma = (float)scale;
  a.workspace_bytes = rbf_attn_decode_workspace_size(&a);
  if (a.workspace_bytes == 0) Py_RETURN_NONE;
  Tensor out, lse;
  {
    const pybind11::gil_scoped_release no_gil;
    const at::NoGradGuard no_grad;
    const c10::OptionalDeviceGuard guard(q.device());
    const Tensor q_ = prep(q, dp), k_ = prep(k, dp), v_ = prep(v, dp);
    const auto f32 = q.options().dtype(at::kFloat);
    out = at::empty({B, H, T, dp}, q.options());
    lse = at::empty({B, H, T}, f32);
    const Tensor ws = at::empty({(int64_t)(a.workspace_bytes + 15) / 16 * 4}, f32);
    a.q = desc(q_);
    a.k = desc(k_);
    a.v = desc(v_);
    a.o = desc(out);
    if (lens.defined()) {
      lens = lens.to(q.device(), at::kInt).contiguous();
      a.lens = lens.data_ptr<int32_t>();
    }
    a.lse = softmax ? lse.data_ptr<float>() : nullptr;
    a.workspace = ws.data_ptr();
    check_rc(rbf_attn_decode(&a, current_stream(q.device())));
    out = unpad(out, D);
  }
  PyObject* o = THPVariable_Wrap(std::move(out));
  PyObject* l = THPVariable_Wrap(std::move(lse));
  PyObject* r = PyTuple_Pack(2, o, l);
  Py_XDECREF(o);
  Py_XDECREF(l);
  return r;
  END_HANDLE_TH_ERRORS
}

// configure(error class, position term's launcher)
PyObject* configure(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 2) {
    PyErr_SetString(PyExc_TypeError, "configure: 2 arguments");
    return nullptr;
  }
  Py_INCREF(args[0]);
  Py_XSETREF(error_class, args[0]);
  Py_INCREF(args[1]);
  Py_XSETREF(pos_launcher, args[1]);
  Py_RETURN_NONE;
}

// check(code): what a library call that returns this code does
PyObject* check(PyObject*, PyObject* code) {
  HANDLE_TH_ERRORS
  const long rc = PyLong_AsLong(code);
  if (PyErr_Occurred()) return nullptr;
  {
    const pybind11::gil_scoped_release no_gil;
    check_rc((int)rc);
  }
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"configure", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(configure)), METH_FASTCALL, nullptr},
    {"check", check, METH_O, nullptr},
    {"attention", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(attention)), METH_FASTCALL, nullptr},
    {"unpack_qkv", unpack_qkv, METH_O, nullptr},
    {"decode", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(decode)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_rbf_attn_torch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__rbf_attn_torch() {
  // the name that an output's grad_fn shows in Python
  static PyTypeObject node_type = {};
  torch::autograd::registerCppFunction(
      typeid(torch::autograd::CppNode<RbfAttentionFunction>),
      torch::autograd::_initFunctionPyTypeObject(node_type, "_EagerRbfAttentionBackward", nullptr, nullptr));
  return PyModule_Create(&module_def);
}
