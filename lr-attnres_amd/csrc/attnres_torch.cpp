// Host side of the drop-in's eager calls: argument checks, descriptors, output
// allocation and the autograd nodes in C++, over the C ABI of
// libattnres_hip.so.  The Python classes of attnres_ops.py do the same work and
// stay the general route: every entry here returns None (nothing launched) for
// whatever is not plain -- tensor subclasses, modes and transforms (vmap, jvp,
// tracing, dispatch and function modes), mixed dtypes, layouts that need a
// copy, non-GPU tensors, arguments the Python code refuses -- and the caller
// then takes that route, which converts, copies or raises.
//
// Why: a training read with 13 values and keys spent 340 us on the host in
// Python (27 tensors through argument loops, ctypes tables, a Python
// autograd.Function and 27 gradient views) against 49 to 240 us of kernels.
//
// Nothing of a call outlives it but the autograd node's saved tensors: the
// backward builds its descriptor from the tensors it unpacks (so saved-tensor
// hooks hold, whatever layout they give back, and in-place checks), on the
// stream current then.
#include <dlfcn.h>

#include <limits>
#include <string>
#include <vector>

#include <torch/extension.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>

#include "../../include/attnres_hip.h"
#include "../../include/attnres_phase1_bank.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// ------------------------------------------------------------------ the library

struct Lib {
#define ATTNRES_FN(name) decltype(&::name) name = nullptr;
#define ATTNRES_FNS(X)                                                                                             \
  X(attnres_last_error) X(attnres_read_forward) X(attnres_read_backward) X(attnres_read_backward_workspace_size)   \
  X(attnres_phase1_forward) X(attnres_phase1_backward_sites) X(attnres_phase1_bank_fits)                           \
  X(attnres_phase1_bank_forward) X(attnres_phase1_bank_backward) X(attnres_phase1_bank_backward_workspace_size)    \
  X(attnres_phase2_forward) X(attnres_phase2_backward) X(attnres_phase2_backward_workspace_size)                   \
  X(attnres_accum_read_forward) X(attnres_accum_read_backward) X(attnres_block_accum_forward)                      \
  X(attnres_block_accum_backward)
  ATTNRES_FNS(ATTNRES_FN)
} lib;

void bind(const std::string& path) {
  void* h = dlopen(path.c_str(), RTLD_NOW | RTLD_LOCAL);
  TORCH_CHECK(h, "attnres: cannot load ", path, ": ", dlerror());
#define ATTNRES_SYM(name)                                                      \
  lib.name = reinterpret_cast<decltype(lib.name)>(dlsym(h, #name));            \
  TORCH_CHECK(lib.name, "attnres: ", path, " has no " #name "; rebuild the library");
  ATTNRES_FNS(ATTNRES_SYM)
}

void check(int rc, const char* what) {
  if (rc != 0)
    throw std::runtime_error(std::string("attnres HIP ") + what + " failed: " + lib.attnres_last_error());
}

// ------------------------------------------------------------------ helpers

int dtype_code(at::ScalarType t) {
  return t == at::kFloat ? ATTNRES_DTYPE_F32 : t == at::kBFloat16 ? ATTNRES_DTYPE_BF16 : t == at::kHalf ? ATTNRES_DTYPE_F16 : -1;
}

// whether plain eager execution is what the caller runs in
bool plain_mode() {
  if (c10::impl::TorchDispatchModeTLS::any_modes_set() || at::impl::torch_function_mode_enabled()) return false;
  if (c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode)) return false;
  return !torch::jit::tracer::isTracing();
}

bool plain_tensor(const Tensor& t) {
  return t.defined() && t.is_cuda() && t.layout() == at::kStrided && !t.is_conj() && !t.is_neg() &&
         !t._fw_grad(0).defined();
}

// a plain tensor argument (Tensor or Parameter, no subclass); false otherwise
bool unpack(PyObject* o, Tensor* out) {
  if (!THPVariable_CheckExact(o)) return false;
  *out = THPVariable_Unpack(o);
  return plain_tensor(*out);
}
bool unpack_opt(const py::object& o, Tensor* out) { return o.is_none() || unpack(o.ptr(), out); }

bool unpack_list(const py::object& o, variable_list* out) {
  if (!PyList_Check(o.ptr()) && !PyTuple_Check(o.ptr())) return false;
  const Py_ssize_t n = PySequence_Fast_GET_SIZE(o.ptr());
  PyObject** items = PySequence_Fast_ITEMS(o.ptr());
  out->resize(n);
  for (Py_ssize_t i = 0; i < n; ++i)
    if (!unpack(items[i], &(*out)[i])) return false;
  return n > 0;
}

// elements between the rows of a [B, T, W] tensor whose tokens are uniformly strided; -1 if they are not
int64_t row_stride(const Tensor& t) {
  const auto sz = t.sizes();
  const auto st = t.strides();
  const int64_t B = sz[0], T = sz[1], W = sz[2];
  if (W > 1 && st[2] != 1) return -1;
  const int64_t r = B * T <= 1 ? W : T == 1 ? st[0] : st[1];
  if (T > 1 && B > 1 && st[0] != T * st[1]) return -1;
  return r >= W ? r : -1;
}

// [B, T, W] row tensors of one shape, dtype and device
bool same_rows(const variable_list& v, int64_t B, int64_t T, at::ScalarType dt, c10::Device dev, int64_t* strides) {
  for (size_t i = 0; i < v.size(); ++i) {
    const Tensor& t = v[i];
    if (t.dim() != 3 || t.size(0) != B || t.size(1) != T || t.size(2) != v[0].size(2)) return false;
    if (t.scalar_type() != dt || t.device() != dev) return false;
    strides[i] = row_stride(t);
    if (strides[i] < 0) return false;
  }
  return true;
}

bool dense(const Tensor& t, at::ScalarType dt, c10::Device dev, int64_t numel) {
  return t.scalar_type() == dt && t.device() == dev && t.numel() == numel && t.is_contiguous();
}

bool any_grad(const variable_list& v) {
  if (!at::GradMode::is_enabled()) return false;
  for (const Tensor& t : v)
    if (t.defined() && t.requires_grad()) return true;
  return false;
}

void* stream_of(c10::Device dev) {
  return (void*)c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(dev.index()).stream();
}

Tensor bytes(size_t n, c10::Device dev) { return at::empty({(int64_t)std::max<size_t>(n, 1)}, at::dtype(at::kByte).device(dev)); }

void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
float* fptr(const Tensor& t) { return t.defined() ? t.data_ptr<float>() : nullptr; }

// the first node of an error when gradients of these gradients are asked for
// (the backwards are not differentiable); plain gradients when no incoming one
// requires a gradient, as torch's once_differentiable returns them
variable_list once(variable_list grads, const variable_list& incoming) {
  if (!any_grad(incoming)) return grads;
  variable_list have;
  for (const Tensor& g : grads)
    if (g.defined()) have.push_back(g);
  if (have.empty()) return grads;
  auto err = std::make_shared<torch::autograd::DelayedError>(
      "trying to differentiate twice a function that was marked with @once_differentiable", (int64_t)have.size());
  variable_list in;
  for (const Tensor& g : have) in.push_back(g.detach().requires_grad_(true));
  variable_list out = (*err)(std::move(in));
  size_t k = 0;
  for (Tensor& g : grads)
    if (g.defined()) g = out[k++];
  return grads;
}

// Saved tensors as the kernels address them: a saved-tensor hook may give a tensor back in another layout.  Those that
// may be strided rows (rows(i)) are copied unless they are; the others are made dense.
template <class F>
void lay_out(variable_list* s, F rows) {
  for (size_t i = 0; i < s->size(); ++i) {
    Tensor& t = (*s)[i];
    if (t.defined() && !t.is_contiguous() && !(rows(i) && t.dim() == 3 && row_stride(t) >= 0)) t = t.contiguous();
  }
}
void copy_dense(Tensor* t) { *t = t->clone(at::MemoryFormat::Contiguous); }

struct Pointers {
  const void* p[ATTNRES_MAX_SOURCES];
  int64_t s[ATTNRES_MAX_SOURCES];
  void fill(const Tensor* t, int n) {
    for (int i = 0; i < n; ++i) {
      p[i] = t[i].data_ptr();
      s[i] = row_stride(t[i]);
    }
  }
};

template <class M>
c10::intrusive_ptr<M> meta_of(AutogradContext* ctx) {
  return c10::static_intrusive_pointer_cast<M>(ctx->saved_data["m"].toCapsule());
}

constexpr float kEps = std::numeric_limits<float>::epsilon();

// ------------------------------------------------------------------ the reads

struct ReadMeta : torch::CustomClassHolder {
  int n = 0;          // sources
  bool lr = false;
  int heads = 1, key_norm = 0, norm = 0, gate_act = 0;
  bool gate_per_token = false;
  float scale = 1.f;
  bool has[5] = {};   // query, query_dyn, gate, bias, static_keys, in this order after values and keys
};

struct ReadCall {
  attnres_read_desc d{};
  Pointers v, k;
  Tensor opt[5];
  int64_t B, T, D, R = 0;
  c10::Device dev;
  at::ScalarType dt;

  // flat: values, keys, the present optional tensors
  ReadCall(const ReadMeta& m, const Tensor* flat) : dev(flat[0].device()), dt(flat[0].scalar_type()) {
    B = flat[0].size(0), T = flat[0].size(1), D = flat[0].size(2);
    v.fill(flat, m.n);
    const Tensor* next = flat + m.n;
    if (m.lr) {
      k.fill(next, m.n);
      R = next[0].size(2);
      next += m.n;
    }
    for (int i = 0; i < 5; ++i)
      if (m.has[i]) opt[i] = *next++;
    d.n_src = m.n;
    d.dtype = d.key_dtype = dtype_code(dt);
    d.n_tok = B * T;
    d.dim = (int)D;
    d.rank = (int)R;
    d.heads = m.heads;
    d.mode = ATTNRES_MODE_SOFTMAX;
    d.key_norm = m.key_norm;
    d.normalize_output = m.norm;
    d.logit_scale = m.scale;
    d.norm_eps = kEps;
    d.values = v.p;
    d.value_row_stride = v.s;
    if (m.lr) {
      d.keys = k.p;
      d.key_row_stride = k.s;
    }
    d.query = ptr(opt[0]);
    d.query_dyn = ptr(opt[1]);
    d.query_dyn_row_stride = opt[1].defined() ? row_stride(opt[1]) : 0;
    d.gate = ptr(opt[2]);
    d.gate_per_token = m.gate_per_token;
    d.gate_act = m.gate_act;
    d.logit_bias = fptr(opt[3]);
    d.static_keys = ptr(opt[4]);
  }
};

// out, and what the backward needs: weights, 1/rms and the pre-norm output
Tensor read_forward(const ReadMeta& m, const Tensor* flat, bool save, Tensor* w, Tensor* inv, Tensor* pre) {
  ReadCall c(m, flat);
  c10::DeviceGuard guard(c.dev);
  const auto opt = flat[0].options().requires_grad(false);
  Tensor out = at::empty({c.B, c.T, c.D}, opt);
  const int64_t n = c.B * c.T;
  if (save) {
    *w = at::empty({n, m.heads, m.n}, opt.dtype(at::kFloat));
    if (m.norm) {
      *inv = at::empty({n}, opt.dtype(at::kFloat));
      *pre = at::empty({n, c.D}, opt);
    }
  }
  check(lib.attnres_read_forward(&c.d, out.data_ptr(), ptr(*pre), fptr(*w), fptr(*inv), stream_of(c.dev)), "forward");
  return out;
}

struct ReadFn : torch::autograd::Function<ReadFn> {
  static Tensor forward(AutogradContext* ctx, c10::intrusive_ptr<ReadMeta> m, at::TensorList in) {
    variable_list flat = in.vec();
    Tensor w, inv, pre;
    Tensor out = read_forward(*m, flat.data(), true, &w, &inv, &pre);
    ctx->saved_data["m"] = c10::IValue::make_capsule(m);
    flat.push_back(w);
    flat.push_back(inv);
    flat.push_back(pre);
    ctx->save_for_backward(std::move(flat));
    ctx->set_materialize_grads(false);
    return out;
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    auto m = meta_of<ReadMeta>(ctx);
    variable_list s = ctx->get_saved_variables();
    const size_t n_in = s.size() - 3;
    variable_list res(1 + n_in);
    if (!grads[0].defined()) return res;
    variable_list d;
    {
      at::NoGradGuard no_grad;
      const size_t n_rows = (m->lr ? 2 : 1) * (size_t)m->n;
      lay_out(&s, [&](size_t i) { return i < n_rows; });
      ReadCall c(*m, s.data());
      c10::DeviceGuard guard(c.dev);
      const auto opt = s[0].options().requires_grad(false);
      const Tensor go = grads[0].contiguous();
      const int64_t n = c.B * c.T;
      d.reserve(n_in);
      void *dv[ATTNRES_MAX_SOURCES], *dk[ATTNRES_MAX_SOURCES];
      for (Tensor& t : at::empty({m->n, c.B, c.T, c.D}, opt).unbind(0)) {
        dv[d.size()] = t.data_ptr();
        d.push_back(std::move(t));
      }
      if (m->lr)
        for (Tensor& t : at::empty({m->n, c.B, c.T, c.R}, opt).unbind(0)) {
          dk[d.size() - m->n] = t.data_ptr();
          d.push_back(std::move(t));
        }
      Tensor dopt[5];
      for (int i = 0; i < 5; ++i)
        if (m->has[i]) dopt[i] = at::empty(c.opt[i].sizes(), c.opt[i].options().requires_grad(false));
      attnres_read_grads g{};
      g.grad_out = go.data_ptr();
      g.out_prenorm = ptr(s[n_in + 2]);
      g.out_inv_rms = fptr(s[n_in + 1]);
      g.weights = fptr(s[n_in]);
      g.dvalues = dv;
      g.dkeys = m->lr ? dk : nullptr;
      g.dquery = ptr(dopt[0]);
      g.dquery_dyn = ptr(dopt[1]);
      g.dgate = ptr(dopt[2]);
      g.dbias = fptr(dopt[3]);
      g.dstatic_keys = ptr(dopt[4]);
      const size_t ws = lib.attnres_read_backward_workspace_size(&c.d);
      const Tensor work = bytes(ws, c.dev);
      g.workspace = work.data_ptr();
      g.workspace_bytes = ws;
      check(lib.attnres_read_backward(&c.d, &g, stream_of(c.dev)), "backward");
      for (int i = 0; i < 5; ++i)
        if (m->has[i]) d.push_back(dopt[i]);
    }
    // inputs that need no gradient get none (the kernels write all of them in one pass)
    for (size_t i = 0; i < n_in; ++i)
      if (ctx->needs_input_grad(i)) res[1 + i] = d[i];
    return once(std::move(res), grads);
  }
};

// keys None: the base read.  query [H, R/H] or [D]; query_dyn [B, T, H, R/H] or, unless by_heads, any [B, T, ...] of R
// elements a token; gate [H] or [B, T, H]
py::object attn_read(const py::object& values, const py::object& keys, const py::object& query, const py::object& query_dyn,
                const py::object& gate, const py::object& bias, const py::object& static_keys, int64_t heads,
                double scale, bool key_norm, bool normalize_output, int64_t gate_act, bool by_heads) {
  variable_list flat, ks;
  if (!plain_mode() || !unpack_list(values, &flat)) return py::none();
  const int64_t n = (int64_t)flat.size();
  if (n < 2 || n > ATTNRES_MAX_SOURCES || flat[0].dim() != 3) return py::none();
  const int64_t B = flat[0].size(0), T = flat[0].size(1), D = flat[0].size(2);
  const auto dt = flat[0].scalar_type();
  const auto dev = flat[0].device();
  int64_t st[ATTNRES_MAX_SOURCES];
  if (B * T < 1 || D < 1 || dtype_code(dt) < 0 || !same_rows(flat, B, T, dt, dev, st)) return py::none();
  auto m = c10::make_intrusive<ReadMeta>();
  m->n = (int)n;
  m->lr = !keys.is_none();
  m->heads = (int)heads;
  m->key_norm = key_norm;
  m->norm = normalize_output;
  m->scale = (float)scale;
  m->gate_act = (int)gate_act;
  int64_t R = D;
  if (m->lr) {
    if (!unpack_list(keys, &ks) || (int64_t)ks.size() != n || ks[0].dim() != 3) return py::none();
    R = ks[0].size(2);
    if (heads < 1 || heads > D || R < 1 || D % heads || R % heads || !same_rows(ks, B, T, dt, dev, st)) return py::none();
    flat.insert(flat.end(), ks.begin(), ks.end());
  }
  Tensor o[5];
  if (!unpack_opt(query, &o[0]) || !unpack_opt(query_dyn, &o[1]) || !unpack_opt(gate, &o[2]) ||
      !unpack_opt(bias, &o[3]) || !unpack_opt(static_keys, &o[4]))
    return py::none();
  if (!o[0].defined() && !o[1].defined()) return py::none();
  if (o[0].defined() && !dense(o[0], dt, dev, R)) return py::none();
  if (o[1].defined()) {
    if (!m->lr || !dense(o[1], dt, dev, B * T * R) || o[1].size(0) != B || o[1].dim() < 3 || o[1].size(1) != T)
      return py::none();
    if (by_heads && (o[1].dim() != 4 || o[1].size(2) != heads)) return py::none();
    if (o[1].dim() != 3) o[1] = o[1].reshape({B, T, R});
  }
  if (o[2].defined()) {
    if (!o[1].defined() || gate_act == ATTNRES_GATE_NONE) return py::none();
    m->gate_per_token = o[2].numel() != heads;
    if (!dense(o[2], dt, dev, m->gate_per_token ? B * T * heads : heads)) return py::none();
  }
  if (o[3].defined() && !dense(o[3], at::kFloat, dev, n)) return py::none();
  if (o[4].defined() && (!m->lr || !dense(o[4], dt, dev, n * R))) return py::none();
  for (int i = 0; i < 5; ++i)
    if (o[i].defined()) {
      m->has[i] = true;
      flat.push_back(o[i]);
    }
  if (any_grad(flat)) return py::cast(ReadFn::apply(m, at::TensorList(flat)));
  Tensor w, inv, pre;
  return py::cast(read_forward(*m, flat.data(), false, &w, &inv, &pre));
}

// ------------------------------------------------------------------ phase 1 from per-source logits

struct Phase1Fn : torch::autograd::Function<Phase1Fn> {
  static void describe(const variable_list& s, attnres_phase1_desc* d, Pointers* v, const void** lg) {
    const int n = (int)s.size() / 2;
    v->fill(s.data() + n, n);
    for (int i = 0; i < n; ++i) lg[i] = s[i].data_ptr();
    *d = attnres_phase1_desc{};
    d->n_src = n;
    d->n_q = (int)s[0].size(0);
    d->dtype = dtype_code(s[n].scalar_type());
    d->logits_dtype = dtype_code(s[0].scalar_type());
    d->n_tok = s[n].size(0) * s[n].size(1);
    d->dim = (int)s[n].size(2);
    d->norm_eps = kEps;
    d->values = v->p;
    d->value_row_stride = v->s;
    d->logit_q_stride = d->logit_s_stride = d->n_tok;
    d->source_logits = lg;
  }

  // in: the sources' logits [Q, B, T], then their values [B, T, D]; out: the sites' reads, then their lse
  static variable_list run(const variable_list& in) {
    attnres_phase1_desc d;
    Pointers v;
    const void* lg[ATTNRES_MAX_SOURCES];
    describe(in, &d, &v, lg);
    const Tensor& v0 = in[in.size() / 2];
    c10::DeviceGuard guard(v0.device());
    const auto opt = v0.options().requires_grad(false);
    const int64_t B = v0.size(0), T = v0.size(1), D = v0.size(2);
    Tensor out = at::empty({d.n_q, B, T, D}, opt), lse = at::empty({d.n_q, B, T}, opt.dtype(at::kFloat));
    check(lib.attnres_phase1_forward(&d, out.data_ptr(), nullptr, fptr(lse), nullptr, stream_of(v0.device())),
          "phase-1 forward");
    variable_list res = out.unbind(0);
    for (Tensor& t : lse.unbind(0)) res.push_back(t);
    return res;
  }

  static variable_list forward(AutogradContext* ctx, at::TensorList list) {
    variable_list in = list.vec();
    variable_list res = run(in);
    ctx->save_for_backward(std::move(in));
    ctx->set_materialize_grads(false);
    return res;
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    variable_list s = ctx->get_saved_variables();
    const int n = (int)s.size() / 2;
    variable_list res(s.size());
    {
      at::NoGradGuard no_grad;
      lay_out(&s, [&](size_t i) { return i >= (size_t)n; });
      attnres_phase1_desc d;
      Pointers v;
      const void* lg[ATTNRES_MAX_SOURCES];
      describe(s, &d, &v, lg);
      const Tensor& v0 = s[n];
      c10::DeviceGuard guard(v0.device());
      const auto opt = v0.options().requires_grad(false);
      const int Q = d.n_q;
      variable_list keep;
      keep.reserve(2 * Q);
      const void* go[ATTNRES_PHASE1_MAX_QUERIES];
      const float* gl[ATTNRES_PHASE1_MAX_QUERIES];
      for (int q = 0; q < Q; ++q) {
        keep.push_back(grads[q].defined() ? grads[q].contiguous() : at::zeros(v0.sizes(), opt));
        go[q] = keep.back().data_ptr();
      }
      for (int q = 0; q < Q; ++q) {
        gl[q] = nullptr;
        if (grads[Q + q].defined()) {
          keep.push_back(grads[Q + q].to(at::kFloat).contiguous());
          gl[q] = fptr(keep.back());
        }
      }
      void *dv[ATTNRES_MAX_SOURCES], *dl[ATTNRES_MAX_SOURCES];
      // (an allocation per source: a source that later blocks read too keeps its gradient long after the others')
      variable_list dvs(n);
      variable_list dls = at::empty({n, Q, v0.size(0), v0.size(1)}, opt.dtype(s[0].scalar_type())).unbind(0);
      for (int i = 0; i < n; ++i) {
        dvs[i] = at::empty(v0.sizes(), opt);
        dv[i] = dvs[i].data_ptr();
        dl[i] = dls[i].data_ptr();
      }
      check(lib.attnres_phase1_backward_sites(&d, go, gl, nullptr, nullptr, dv, dl, d.n_tok, stream_of(v0.device())),
            "phase-1 backward");
      for (int i = 0; i < n; ++i) {
        if (ctx->needs_input_grad(i)) res[i] = dls[i];
        if (ctx->needs_input_grad(n + i)) res[n + i] = dvs[i];
      }
    }
    return once(std::move(res), grads);
  }
};

py::object phase1_sources(const py::object& values, const py::object& logits) {
  variable_list v, in;
  if (!plain_mode() || !unpack_list(values, &v) || !unpack_list(logits, &in)) return py::none();
  const size_t n = v.size();
  if (n > ATTNRES_MAX_SOURCES || in.size() != n || v[0].dim() != 3 || in[0].dim() != 3) return py::none();
  const int64_t B = v[0].size(0), T = v[0].size(1), D = v[0].size(2), Q = in[0].size(0);
  const auto dt = v[0].scalar_type(), ldt = in[0].scalar_type();
  int64_t st[ATTNRES_MAX_SOURCES];
  if (B * T < 1 || D < 1 || D > ATTNRES_PHASE_MAX_DIM || Q < 1 || Q > ATTNRES_PHASE1_MAX_QUERIES) return py::none();
  if (dtype_code(dt) < 0 || dtype_code(ldt) < 0 || !same_rows(v, B, T, dt, v[0].device(), st)) return py::none();
  for (const Tensor& t : in)
    if (!dense(t, ldt, v[0].device(), Q * B * T) || t.dim() != 3 || t.size(0) != Q || t.size(1) != B) return py::none();
  in.insert(in.end(), v.begin(), v.end());
  variable_list res = any_grad(in) ? Phase1Fn::apply(at::TensorList(in)) : Phase1Fn::run(in);
  py::tuple outs(Q), lses(Q);
  for (int64_t q = 0; q < Q; ++q) {
    outs[q] = py::cast(res[q]);
    lses[q] = py::cast(res[Q + q]);
  }
  return py::make_tuple(outs, lses);
}

// ------------------------------------------------------------------ phase 1 from a query bank

struct BankMeta : torch::CustomClassHolder {
  int key_norm = 0;
};

struct BankFn : torch::autograd::Function<BankFn> {
  // s: queries [Q, D], values [B, T, D] ...
  static void describe(const BankMeta& m, const Tensor* s, int n, attnres_keyed_logits_desc* d, Pointers* v) {
    v->fill(s + 1, n);
    *d = attnres_keyed_logits_desc{};
    d->n_src = n;
    d->n_q = (int)s[0].size(0);
    d->dtype = dtype_code(s[1].scalar_type());
    d->n_tok = s[1].size(0) * s[1].size(1);
    d->dim = (int)s[1].size(2);
    d->key_norm = m.key_norm;
    d->norm_eps = kEps;
    d->values = v->p;
    d->value_row_stride = v->s;
    d->queries = s[0].data_ptr();
  }

  static variable_list run(const BankMeta& m, const variable_list& in, bool save, Tensor* logits, Tensor* inv) {
    attnres_keyed_logits_desc d;
    Pointers v;
    describe(m, in.data(), (int)in.size() - 1, &d, &v);
    const Tensor& v0 = in[1];
    c10::DeviceGuard guard(v0.device());
    const auto opt = v0.options().requires_grad(false);
    const int64_t B = v0.size(0), T = v0.size(1), D = v0.size(2);
    Tensor out = at::empty({d.n_q, B, T, D}, opt), lse = at::empty({d.n_q, B, T}, opt.dtype(at::kFloat));
    if (save) {
      *logits = at::empty({d.n_q, d.n_src, d.n_tok}, opt);
      if (m.key_norm) *inv = at::empty({d.n_src, d.n_tok}, opt.dtype(at::kFloat));
    }
    check(lib.attnres_phase1_bank_forward(&d, out.data_ptr(), fptr(lse), ptr(*logits), fptr(*inv),
                                          stream_of(v0.device())), "query-bank forward");
    return {out, lse};
  }

  static variable_list forward(AutogradContext* ctx, c10::intrusive_ptr<BankMeta> m, at::TensorList list) {
    variable_list in = list.vec();
    Tensor logits, inv;
    variable_list res = run(*m, in, true, &logits, &inv);
    ctx->saved_data["m"] = c10::IValue::make_capsule(m);
    in.push_back(logits);
    in.push_back(inv);
    ctx->save_for_backward(std::move(in));
    ctx->set_materialize_grads(false);
    return res;
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    auto m = meta_of<BankMeta>(ctx);
    variable_list s = ctx->get_saved_variables();
    const int n = (int)s.size() - 3;
    variable_list res(2 + n);
    if (!grads[0].defined() && !grads[1].defined()) return res;
    {
      at::NoGradGuard no_grad;
      lay_out(&s, [&](size_t i) { return i > 0 && i <= (size_t)n; });
      attnres_keyed_logits_desc d;
      Pointers v;
      describe(*m, s.data(), n, &d, &v);
      if (!lib.attnres_phase1_bank_fits(&d)) {  // (given back at another alignment)
        for (int i = 0; i <= n; ++i) copy_dense(&s[i]);
        describe(*m, s.data(), n, &d, &v);
      }
      const Tensor& v0 = s[1];
      c10::DeviceGuard guard(v0.device());
      const auto opt = v0.options().requires_grad(false);
      Tensor go = grads[0].defined() ? grads[0].contiguous()
                                     : at::zeros({d.n_q, v0.size(0), v0.size(1), v0.size(2)}, opt);
      if ((uintptr_t)go.data_ptr() % 16) go = go.clone();  // (a view into a larger gradient)
      Tensor gl;
      if (grads[1].defined()) gl = grads[1].to(at::kFloat).contiguous();
      variable_list dvs = at::empty({n, v0.size(0), v0.size(1), v0.size(2)}, opt).unbind(0);
      void* dv[ATTNRES_MAX_SOURCES];
      for (int i = 0; i < n; ++i) dv[i] = dvs[i].data_ptr();
      Tensor dq, work;
      size_t ws = 0;
      if (ctx->needs_input_grad(0)) {
        dq = at::empty(s[0].sizes(), opt);
        ws = lib.attnres_phase1_bank_backward_workspace_size(&d);
        work = bytes(ws, v0.device());
      }
      check(lib.attnres_phase1_bank_backward(&d, go.data_ptr(), fptr(gl), ptr(s[n + 1]), fptr(s[n + 2]), dv, ptr(dq),
                                             ptr(work), ws, stream_of(v0.device())), "query-bank backward");
      res[1] = dq;
      for (int i = 0; i < n; ++i)
        if (ctx->needs_input_grad(1 + i)) res[2 + i] = dvs[i];
    }
    return once(std::move(res), grads);
  }
};

py::object phase1_bank(const py::object& values, const py::object& queries, bool key_norm) {
  variable_list v;
  Tensor q;
  if (!plain_mode() || !unpack_list(values, &v) || !unpack(queries.ptr(), &q)) return py::none();
  const size_t n = v.size();
  if (n > ATTNRES_MAX_SOURCES || v[0].dim() != 3 || q.dim() != 2) return py::none();
  const int64_t B = v[0].size(0), T = v[0].size(1), D = v[0].size(2), Q = q.size(0);
  const auto dt = v[0].scalar_type();
  int64_t st[ATTNRES_MAX_SOURCES];
  if (B * T < 1 || D < 1 || Q < 1 || Q > ATTNRES_PHASE1_MAX_QUERIES || dtype_code(dt) < 0 ||
      !same_rows(v, B, T, dt, v[0].device(), st) || !dense(q, dt, v[0].device(), Q * D))
    return py::none();
  auto m = c10::make_intrusive<BankMeta>();
  m->key_norm = key_norm;
  v.insert(v.begin(), q);
  attnres_keyed_logits_desc d;
  Pointers p;
  BankFn::describe(*m, v.data(), (int)n, &d, &p);
  if (!lib.attnres_phase1_bank_fits(&d)) return py::none();
  Tensor a, b;
  variable_list res = any_grad(v) ? BankFn::apply(m, at::TensorList(v)) : BankFn::run(*m, v, false, &a, &b);
  return py::make_tuple(res[0], res[1]);
}

// ------------------------------------------------------------------ phase 2 and the accumulate-and-read

struct MergeMeta : torch::CustomClassHolder {
  int merge = 0, key_norm = 0, norm = 0, scale_key = 0;
  float scale = 1.f, bias = 0.f, vscale = 1.f;
  int64_t qrow = -1;  // row of a query bank, or the query itself
  // accumulate-and-read
  int64_t D = 0, R = 0;
  int heads = 1, acc_key_norm = 0;
  bool has_partial = false;
};

void fill_merge(const MergeMeta& m, const Tensor& pv, const Tensor& pk, const Tensor& query, const Tensor& inter,
                const Tensor& lse, int64_t D, attnres_phase2_desc* d) {
  *d = attnres_phase2_desc{};
  d->dtype = dtype_code(inter.scalar_type());
  d->n_tok = inter.size(0) * inter.size(1);
  d->dim = (int)D;
  d->rank = pk.defined() ? (int)pk.size(-1) : 0;
  d->merge = m.merge;
  d->key_norm = m.key_norm;
  d->normalize_output = m.norm;
  d->logit_scale = m.scale;
  d->norm_eps = kEps;
  d->logit_bias = m.bias;
  d->value_scale = m.vscale;
  d->scale_key = m.scale_key;
  d->partial_value = ptr(pv);
  d->partial_value_row_stride = pv.defined() ? row_stride(pv) : D;
  d->partial_key = ptr(pk);
  d->partial_key_row_stride = pk.defined() ? row_stride(pk) : 0;
  d->query = (const char*)query.data_ptr() + (m.qrow >= 0 ? m.qrow * query.size(1) * query.element_size() : 0);
  d->interblock_output = inter.data_ptr();
  d->interblock_row_stride = row_stride(inter);
  d->interblock_lse = fptr(lse);
}

struct Phase2Fn : torch::autograd::Function<Phase2Fn> {
  // in: partial value, inter, lse, query, partial key (LR)
  static Tensor run(const MergeMeta& m, const variable_list& in) {
    attnres_phase2_desc d;
    fill_merge(m, in[0], in.size() > 4 ? in[4] : Tensor(), in[3], in[1], in[2], in[0].size(2), &d);
    c10::DeviceGuard guard(in[0].device());
    Tensor out = at::empty(in[0].sizes(), in[0].options().requires_grad(false));
    check(lib.attnres_phase2_forward(&d, out.data_ptr(), stream_of(in[0].device())), "phase-2 forward");
    return out;
  }

  static Tensor forward(AutogradContext* ctx, c10::intrusive_ptr<MergeMeta> m, at::TensorList list) {
    variable_list in = list.vec();
    Tensor out = run(*m, in);
    ctx->saved_data["m"] = c10::IValue::make_capsule(m);
    ctx->save_for_backward(std::move(in));
    ctx->set_materialize_grads(false);
    return out;
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    auto m = meta_of<MergeMeta>(ctx);
    variable_list s = ctx->get_saved_variables();
    variable_list res(1 + s.size());
    if (!grads[0].defined()) return res;
    {
      at::NoGradGuard no_grad;
      const bool lr = s.size() > 4;
      lay_out(&s, [](size_t i) { return i < 2 || i == 4; });
      attnres_phase2_desc d;
      fill_merge(*m, s[0], lr ? s[4] : Tensor(), s[3], s[1], s[2], s[0].size(2), &d);
      const auto dev = s[0].device();
      c10::DeviceGuard guard(dev);
      const auto opt = s[0].options().requires_grad(false);
      const Tensor go = grads[0].contiguous();
      Tensor dp = at::empty(s[0].sizes(), opt), di = at::empty(s[1].sizes(), opt);
      Tensor dl = at::empty(s[2].sizes(), opt.dtype(at::kFloat)), dk, dq;
      if (lr) dk = at::empty(s[4].sizes(), opt);
      if (ctx->needs_input_grad(3)) dq = at::empty(s[3].sizes(), opt);
      attnres_phase2_grads g{};
      g.grad_out = go.data_ptr();
      g.dpartial_value = dp.data_ptr();
      g.dpartial_key = ptr(dk);
      g.dquery = ptr(dq);
      g.dinterblock_output = di.data_ptr();
      g.dinterblock_lse = fptr(dl);
      if (dq.defined() && m->qrow >= 0) {
        g.dquery_rows = (int)s[3].size(0);
        g.dquery_row = (int)m->qrow;
      }
      const size_t ws = lib.attnres_phase2_backward_workspace_size(&d);
      const Tensor work = bytes(ws, dev);
      g.workspace = work.data_ptr();
      g.workspace_bytes = ws;
      check(lib.attnres_phase2_backward(&d, &g, stream_of(dev)), "phase-2 backward");
      const Tensor all[5] = {dp, di, dl, dq, dk};
      for (size_t i = 0; i < s.size(); ++i)
        if (ctx->needs_input_grad(i)) res[1 + i] = all[i];
    }
    return once(std::move(res), grads);
  }
};

// query: [D] / [rank], or with query_row >= 0 a bank [rows, rank] (LR)
py::object merge_read(const py::object& partial_value, const py::object& partial_key, const py::object& query,
                  const py::object& inter, const py::object& lse, int64_t merge, bool key_norm, bool normalize_output,
                  double scale, double bias, double vscale, bool scale_key, int64_t query_row) {
  variable_list in(4);
  Tensor pk;
  if (!plain_mode() || !unpack(partial_value.ptr(), &in[0]) || !unpack(inter.ptr(), &in[1]) ||
      !unpack(lse.ptr(), &in[2]) || !unpack(query.ptr(), &in[3]) || !unpack_opt(partial_key, &pk))
    return py::none();
  if (in[0].dim() != 3) return py::none();
  const int64_t B = in[0].size(0), T = in[0].size(1), D = in[0].size(2), n = B * T;
  const auto dt = in[0].scalar_type();
  const auto dev = in[0].device();
  int64_t st[2];
  if (n < 1 || D < 1 || D > ATTNRES_PHASE_MAX_DIM || dtype_code(dt) < 0) return py::none();
  if (!same_rows({in[0], in[1]}, B, T, dt, dev, st) || !dense(in[2], at::kFloat, dev, n)) return py::none();
  int64_t W = D;
  if (pk.defined()) {
    if (pk.dim() != 3 || !same_rows({pk}, B, T, dt, dev, st)) return py::none();
    W = pk.size(2);
    in.push_back(pk);
  }
  auto m = c10::make_intrusive<MergeMeta>();
  if (query_row >= 0) {
    if (!pk.defined() || in[3].dim() != 2 || in[3].size(1) != W || query_row >= in[3].size(0) ||
        !dense(in[3], dt, dev, in[3].size(0) * W))
      return py::none();
    m->qrow = query_row;
  } else if (!dense(in[3], dt, dev, W)) {
    return py::none();
  }
  m->merge = (int)merge;
  m->key_norm = key_norm;
  m->norm = normalize_output;
  m->scale = (float)scale;
  m->bias = (float)bias;
  m->vscale = (float)vscale;
  m->scale_key = scale_key;
  return py::cast(any_grad(in) ? Phase2Fn::apply(m, at::TensorList(in)) : Phase2Fn::run(*m, in));
}

void fill_split(const MergeMeta& m, const Tensor& y, const Tensor& pv, const Tensor& pk, bool complete, float vscale,
                int64_t n, attnres_block_accum_desc* d) {
  *d = attnres_block_accum_desc{};
  d->split.dtype = dtype_code(y.scalar_type());
  d->split.n_tok = n;
  d->split.dim = (int)m.D;
  d->split.rank = (int)m.R;
  d->split.proj_cols = (int)y.size(-1);
  d->split.heads = m.heads;
  d->split.key_norm = m.acc_key_norm;
  d->split.norm_eps = kEps;
  d->split.projected = y.data_ptr();
  d->split.row_stride = y.size(-1);  // (contiguous)
  d->complete = complete;
  d->partial_value = ptr(pv);
  d->partial_key = ptr(pk);
  d->value_scale = vscale;
}

// a gradient with rows of W elements, uniformly strided as [n, W] (copied if not); *stride its row stride
Tensor grad_rows(const Tensor& g, int64_t W, int64_t* stride) {
  if (g.dim() == 3) {
    *stride = row_stride(g);
    if (*stride >= W) return g;
  }
  *stride = W;
  return g.contiguous();
}

// rows of whole 16-byte vectors, as the fused kernels read them
bool fused_rows(const Tensor& t) {
  return ((uintptr_t)t.data_ptr() | (uintptr_t)(row_stride(t) * t.element_size())) % 16 == 0;
}

struct AccumReadFn : torch::autograd::Function<AccumReadFn> {
  // in: y [B, T, P], query bank [rows, R], inter [B, T, D], lse [B, T], and the old partial value and key
  static variable_list run(const MergeMeta& m, const variable_list& in, Tensor* kinv) {
    const int64_t B = in[2].size(0), T = in[2].size(1), n = B * T;
    const auto dev = in[0].device();
    c10::DeviceGuard guard(dev);
    const auto opt = in[0].options().requires_grad(false);
    Tensor value = at::empty({B, T, m.D}, opt), key = at::empty({B, T, m.R}, opt), out = at::empty({B, T, m.D}, opt);
    if (m.acc_key_norm) *kinv = at::empty({n, m.heads}, opt.dtype(at::kFloat));
    attnres_accum_read_desc d;
    fill_split(m, in[0], m.has_partial ? in[4] : Tensor(), m.has_partial ? in[5] : Tensor(), false, 1.f, n, &d.accum);
    fill_merge(m, value, key, in[1], in[2], in[3], m.D, &d.read);
    check(lib.attnres_accum_read_forward(&d, value.data_ptr(), key.data_ptr(), fptr(*kinv), out.data_ptr(),
                                         stream_of(dev)), "accumulate-and-read forward");
    return {value, key, out};
  }

  static variable_list forward(AutogradContext* ctx, c10::intrusive_ptr<MergeMeta> m, at::TensorList list) {
    variable_list in = list.vec();
    Tensor kinv;
    variable_list res = run(*m, in, &kinv);
    ctx->saved_data["m"] = c10::IValue::make_capsule(m);
    in.push_back(kinv);
    in.push_back(res[0]);
    in.push_back(res[1]);
    ctx->save_for_backward(std::move(in));
    ctx->set_materialize_grads(false);
    return res;
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    auto m = meta_of<MergeMeta>(ctx);
    variable_list s = ctx->get_saved_variables();
    const size_t n_in = s.size() - 3;
    variable_list res(1 + n_in);
    if (!grads[0].defined() && !grads[1].defined() && !grads[2].defined()) return res;
    {
      at::NoGradGuard no_grad;
      lay_out(&s, [](size_t i) { return i == 2; });
      for (size_t i : {(size_t)0, (size_t)2, n_in + 1})  // (given back at another alignment)
        if (!fused_rows(s[i])) copy_dense(&s[i]);
      const Tensor &y = s[0], &query = s[1], &inter = s[2], &lse = s[3], &kinv = s[n_in], &value = s[n_in + 1],
                   &key = s[n_in + 2];
      const int64_t n = inter.size(0) * inter.size(1);
      const auto dev = y.device();
      c10::DeviceGuard guard(dev);
      const auto opt = y.options().requires_grad(false);
      attnres_accum_read_desc d;
      fill_split(*m, y, m->has_partial ? s[4] : Tensor(), m->has_partial ? s[5] : Tensor(), false, 1.f, n, &d.accum);
      fill_merge(*m, value, key, query, inter, lse, m->D, &d.read);
      Tensor go = grads[2].defined() ? grads[2].contiguous() : at::zeros(value.sizes(), opt);
      if (!fused_rows(go)) copy_dense(&go);
      int64_t gvs = m->D;
      Tensor gv, gk;
      if (grads[0].defined()) gv = grad_rows(grads[0], m->D, &gvs);
      if (gv.defined() && !fused_rows(gv)) {
        copy_dense(&gv);
        gvs = m->D;
      }
      if (grads[1].defined()) gk = grads[1].contiguous();
      Tensor gy = at::empty(y.sizes(), opt), di = at::empty(inter.sizes(), opt);
      Tensor dl = at::empty(lse.sizes(), opt.dtype(at::kFloat)), dq, dpk;
      if (ctx->needs_input_grad(1)) dq = at::empty(query.sizes(), opt);
      if (m->has_partial && ctx->needs_input_grad(5)) dpk = at::empty(s[5].sizes(), opt);
      attnres_phase2_grads g{};
      g.grad_out = go.data_ptr();
      g.dquery = ptr(dq);
      g.dinterblock_output = di.data_ptr();
      g.dinterblock_lse = fptr(dl);
      if (dq.defined()) {
        g.dquery_rows = (int)query.size(0);
        g.dquery_row = (int)m->qrow;
      }
      const size_t ws = lib.attnres_phase2_backward_workspace_size(&d.read);
      const Tensor work = bytes(ws, dev);
      g.workspace = work.data_ptr();
      g.workspace_bytes = ws;
      check(lib.attnres_accum_read_backward(&d, &g, ptr(gv), gvs, ptr(gk), fptr(kinv), gy.data_ptr(), ptr(dpk),
                                            stream_of(dev)), "accumulate-and-read backward");
      // the grown value's total gradient is also the old partial value's: columns [0, D) of gy
      const Tensor all[6] = {gy, dq, di, dl, m->has_partial ? gy.narrow(-1, 0, m->D) : Tensor(), dpk};
      for (size_t i = 0; i < n_in; ++i)
        if (ctx->needs_input_grad(i)) res[1 + i] = all[i];
    }
    return once(std::move(res), grads);
  }
};

bool accum_inputs(const py::object& projected, const py::object& partial_value, const py::object& partial_key, int64_t D,
                  int64_t R, int64_t heads, Tensor* y, Tensor* pv, Tensor* pk) {
  if (!unpack(projected.ptr(), y) || !unpack_opt(partial_value, pv) || !unpack_opt(partial_key, pk)) return false;
  if (y->dim() != 3 || !y->is_contiguous() || y->numel() < 1 || dtype_code(y->scalar_type()) < 0) return false;
  if (D < 1 || R < 1 || heads < 1 || R % heads || y->size(2) < D + R || pv->defined() != pk->defined()) return false;
  const int64_t n = y->size(0) * y->size(1);
  for (const Tensor* t : {pv, pk})
    if (t->defined() && (t->dim() != 3 || t->size(0) != y->size(0) || t->size(1) != y->size(1) ||
                         !dense(*t, y->scalar_type(), y->device(), n * (t == pv ? D : R))))
      return false;
  return true;
}

// the checks here decide whether the fused kernels take the rows (for the Python route: _accum_read_fits)
py::object accum_read(const py::object& projected, const py::object& partial_value, const py::object& partial_key,
                      const py::object& bank, const py::object& inter, const py::object& lse, int64_t D, int64_t R,
                      double scale, int64_t heads, bool key_norm, bool merge_key_norm, int64_t merge,
                      bool normalize_output, double bias, double vscale, bool scale_key, int64_t query_row) {
  Tensor y, pv, pk, q, it, ls;
  if (!plain_mode() || !accum_inputs(projected, partial_value, partial_key, D, R, heads, &y, &pv, &pk)) return py::none();
  if (!unpack(bank.ptr(), &q) || !unpack(inter.ptr(), &it) || !unpack(lse.ptr(), &ls)) return py::none();
  const int64_t B = y.size(0), T = y.size(1);
  const auto dt = y.scalar_type();
  const auto dev = y.device();
  const size_t es = y.element_size();
  if (es != 2 || (D != 256 && D != 512 && D != 768 && D != 1024) || R > 256) return py::none();
  int64_t st[1];
  if (!same_rows({it}, B, T, dt, dev, st) || it.size(2) != D || !dense(ls, at::kFloat, dev, B * T)) return py::none();
  if (!fused_rows(y) || !fused_rows(it) || (pv.defined() && !fused_rows(pv))) return py::none();
  if (q.dim() != 2 || q.size(1) != R || query_row < 0 || query_row >= q.size(0) || !dense(q, dt, dev, q.size(0) * R))
    return py::none();
  auto m = c10::make_intrusive<MergeMeta>();
  m->merge = (int)merge;
  m->key_norm = merge_key_norm;
  m->norm = normalize_output;
  m->scale_key = scale_key;
  m->scale = (float)scale;
  m->bias = (float)bias;
  m->vscale = (float)vscale;
  m->qrow = query_row;
  m->D = D;
  m->R = R;
  m->heads = (int)heads;
  m->acc_key_norm = key_norm;
  m->has_partial = pv.defined();
  variable_list in = {y, q, it, ls};
  if (pv.defined()) {
    in.push_back(pv);
    in.push_back(pk);
  }
  Tensor kinv;
  variable_list res = any_grad(in) ? AccumReadFn::apply(m, at::TensorList(in)) : AccumReadFn::run(*m, in, &kinv);
  return py::make_tuple(res[0], res[1], res[2]);
}

// ------------------------------------------------------------------ the block accumulation

struct AccumMeta : MergeMeta {
  bool complete = false;
};

struct AccumFn : torch::autograd::Function<AccumFn> {
  // in: y [B, T, P], old partial value and key; out: value, key.  No value norm, a host scale, an unscaled key
  static variable_list run(const AccumMeta& m, const variable_list& in, Tensor* kinv) {
    const Tensor& y = in[0];
    const int64_t B = y.size(0), T = y.size(1), n = B * T;
    c10::DeviceGuard guard(y.device());
    const auto opt = y.options().requires_grad(false);
    Tensor value = at::empty({B, T, m.D}, opt), key = at::empty({B, T, m.R}, opt);
    if (m.acc_key_norm) *kinv = at::empty({n, m.heads}, opt.dtype(at::kFloat));
    attnres_block_accum_desc d;
    fill_split(m, y, m.has_partial ? in[1] : Tensor(), m.has_partial ? in[2] : Tensor(), m.complete, m.vscale, n, &d);
    check(lib.attnres_block_accum_forward(&d, value.data_ptr(), key.data_ptr(), fptr(*kinv), nullptr,
                                          stream_of(y.device())), "block accumulation forward");
    return {value, key};
  }

  static variable_list forward(AutogradContext* ctx, c10::intrusive_ptr<AccumMeta> m, at::TensorList list) {
    variable_list in = list.vec();
    Tensor kinv;
    variable_list res = run(*m, in, &kinv);
    ctx->saved_data["m"] = c10::IValue::make_capsule(m);
    in.push_back(kinv);
    ctx->save_for_backward(std::move(in));
    ctx->set_materialize_grads(false);
    return res;
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    auto m = meta_of<AccumMeta>(ctx);
    variable_list s = ctx->get_saved_variables();
    const size_t n_in = s.size() - 1;
    variable_list res(1 + n_in);
    if (!grads[0].defined() && !grads[1].defined()) return res;
    {
      at::NoGradGuard no_grad;
      lay_out(&s, [](size_t) { return false; });
      const Tensor& y = s[0];
      const int64_t n = y.size(0) * y.size(1);
      c10::DeviceGuard guard(y.device());
      attnres_block_accum_desc d;
      fill_split(*m, y, m->has_partial ? s[1] : Tensor(), m->has_partial ? s[2] : Tensor(), m->complete, m->vscale, n, &d);
      int64_t gvs = 0;
      Tensor gv, gk;
      if (grads[0].defined()) gv = grad_rows(grads[0], m->D, &gvs);
      if (grads[1].defined()) gk = grads[1].contiguous();
      Tensor gy = at::empty(y.sizes(), y.options().requires_grad(false));
      check(lib.attnres_block_accum_backward(&d, ptr(gv), gvs, ptr(gk), fptr(s[n_in]), nullptr, gy.data_ptr(), nullptr,
                                             nullptr, nullptr, 0, stream_of(y.device())), "block accumulation backward");
      if (ctx->needs_input_grad(0)) res[1] = gy;
      if (m->has_partial) {
        // the partial value's gradient: columns [0, D) of gy, or the incoming one when nothing scales it
        if (ctx->needs_input_grad(1) && gv.defined()) res[2] = m->complete ? gy.narrow(-1, 0, m->D) : gv;
        if (ctx->needs_input_grad(2) && gk.defined()) res[3] = gk;
      }
    }
    return once(std::move(res), grads);
  }
};

py::object block_accum(const py::object& projected, const py::object& partial_value, const py::object& partial_key,
                       int64_t D, int64_t R, int64_t heads, bool key_norm, bool complete, double vscale) {
  Tensor y, pv, pk;
  if (!plain_mode() || !accum_inputs(projected, partial_value, partial_key, D, R, heads, &y, &pv, &pk)) return py::none();
  auto m = c10::make_intrusive<AccumMeta>();
  m->D = D;
  m->R = R;
  m->heads = (int)heads;
  m->acc_key_norm = key_norm;
  m->has_partial = pv.defined();
  m->complete = complete;
  m->vscale = (float)vscale;
  variable_list in = {y};
  if (pv.defined()) {
    in.push_back(pv);
    in.push_back(pk);
  }
  Tensor kinv;
  variable_list res = any_grad(in) ? AccumFn::apply(m, at::TensorList(in)) : AccumFn::run(*m, in, &kinv);
  return py::make_tuple(res[0], res[1]);
}

}  // namespace

PYBIND11_MODULE(_attnres_torch, m) {
  m.def("bind", &bind);
  m.def("read", &attn_read);
  m.def("phase1_sources", &phase1_sources);
  m.def("phase1_bank", &phase1_bank);
  m.def("phase2", &merge_read);
  m.def("accum_read", &accum_read);
  m.def("block_accum", &block_accum);
}
