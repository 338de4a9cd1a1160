// Host path of the hot calls: argument checks, allocation, launch and the autograd nodes of the first backward pass, as a
// Python extension module on top of the C ABI of libe3x.so.
//
// A small product, a message on one molecule or the gradient of some thousand harmonics takes its GPU time several times
// over in the interpreter, and autograd runs the backward pass of GPU tensors on a thread of its own, where Python is slower
// still (the gradient of 1000 harmonics 88 us a pass, 35 with the pass on the calling thread; a negation of torch's own
// 41 and 21).  A call comes here when it needs nothing of Python: plain tensors, no function transform, no forward-mode
// level, no tracing, no dispatch or function mode; every entry returns None otherwise and its caller goes on in Python,
// which also has every check that raises.  What a node saves goes through torch's saved variables (version counters, hooks);
// under create_graph its backward pass is the one written in Python, which can be differentiated.
#include <torch/extension.h>

#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPGuard.h>
#include <c10/hip/HIPStream.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/forward_grad.h>
#include <torch/csrc/autograd/python_cpp_function.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/csrc/utils/pybind.h>

#include <array>
#include <mutex>

#include "../../include/e3x.h"

namespace {
using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// ---- Python objects that nodes keep: released with the interpreter lock held, whatever thread drops the node -------------
struct PyRef {
  PyObject* p = nullptr;
  PyRef() = default;
  explicit PyRef(const py::handle& h) : p(h.ptr()) { Py_XINCREF(p); }
  PyRef(const PyRef&) = delete;
  PyRef& operator=(const PyRef&) = delete;
  ~PyRef() {
    if (p && Py_IsInitialized()) {
      py::gil_scoped_acquire gil;
      Py_DECREF(p);
    }
  }
  py::object get() const { return py::reinterpret_borrow<py::object>(p); }
};

py::dict* hooks = nullptr;  // Python functions by name: see `connect`

py::object hook(const char* name) { return (*hooks)[name]; }

// the exception classes of the Python layer
[[noreturn]] void raise(int rc) {
  const std::string msg = e3x_last_error();
  if (rc == E3X_ERR_INDEX) TORCH_CHECK_INDEX(false, msg);
  py::gil_scoped_acquire gil;
  PyErr_SetString(hook("E3xError").ptr(), msg.c_str());
  python_error err;
  err.persist();
  throw err;
}
inline void check(int rc) {
  if (rc != E3X_OK) raise(rc);
}

// a Python call whose exception crosses the autograd engine as what it is
template <class F>
auto in_python(F f) {
  py::gil_scoped_acquire gil;
  try {
    return f();
  } catch (py::error_already_set& e) {
    e.restore();
    python_error err;
    err.persist();
    throw err;
  }
}

// ---- what decides whether a call is Python's ----------------------------------------------------------------------------
bool plain_state() {
  return !c10::impl::tls_is_dispatch_key_included(at::DispatchKey::FuncTorchDynamicLayerFrontMode) &&
         !c10::impl::TorchDispatchModeTLS::any_modes_set() && at::impl::PythonTorchFunctionTLS::stack_len() == 0 &&
         !torch::jit::tracer::isTracing() && !torch::autograd::ForwardADLevel::try_get_by_idx(0);
}
// a contiguous GPU tensor without a Python class of its own, conjugation or the like
bool plain(const Tensor& t, at::ScalarType dtype) {
  return t.is_cuda() && t.scalar_type() == dtype && t.layout() == at::kStrided && t.is_contiguous() &&
         !t.key_set().has_any(at::DispatchKeySet({at::DispatchKey::Python, at::DispatchKey::Negative, at::DispatchKey::Conjugate}));
}
bool recorded(std::initializer_list<const Tensor*> ts) {
  if (at::GradMode::is_enabled())
    for (const Tensor* t : ts)
      if (t->requires_grad()) return true;
  return false;
}

inline const void* in(const Tensor& t) { return t.defined() && t.numel() ? t.data_ptr() : nullptr; }
inline void* ptr(const Tensor& t) { return t.defined() && t.numel() ? t.data_ptr() : nullptr; }
template <class T>
inline T* ptr_as(const Tensor& t) { return static_cast<T*>(ptr(t)); }
inline bool aligned(const Tensor& t) { return ((uintptr_t)t.data_ptr() & 15) == 0; }
inline void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }
Tensor rows_like(const Tensor& like, int64_t rows, int64_t width) { return at::empty({rows, width}, like.options().requires_grad(false)); }
Tensor bytes_like(const Tensor& like, size_t n) { return at::empty({(int64_t)n}, like.options().dtype(at::kByte).requires_grad(false)); }
struct OnDevice {
  c10::hip::OptionalHIPGuard guard;
  explicit OnDevice(const Tensor& t) {
    if (t.device().index() != c10::hip::current_device()) guard.set_index(t.device().index());
  }
};

// ---- autograd: a node whose operation is an object, a node type for each kind of it --------------------------------------------------------------
struct Op : torch::CustomClassHolder {
  virtual variable_list forward(const variable_list& in) = 0;
  virtual variable_list to_save(const variable_list& in) { return in; }
  // gradients of the inputs, undefined where not needed
  virtual variable_list backward(const variable_list& saved, const variable_list& g, const std::vector<bool>& need) = 0;
  // the same, differentiable: in Python
  virtual py::object backward_in_python(const variable_list& saved, const variable_list& g, const std::vector<bool>& need) = 0;
};
using OpPtr = c10::intrusive_ptr<Op>;

template <class Kind>
struct OpFn : torch::autograd::Function<OpFn<Kind>> {
  template <class... Ts>
  static variable_list forward(AutogradContext* ctx, const c10::intrusive_ptr<Kind>& op, const Ts&... ts) {
    variable_list in{ts...};
    variable_list out = op->forward(in);
    ctx->save_for_backward(op->to_save(in));
    ctx->saved_data["op"] = c10::IValue::make_capsule(OpPtr(op));
    ctx->saved_data["n"] = (int64_t)in.size();
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    auto op = c10::static_intrusive_pointer_cast<Op>(ctx->saved_data["op"].toCapsule());
    const size_t n = (size_t)ctx->saved_data["n"].toInt();
    std::vector<bool> need(n);
    for (size_t i = 0; i < n; ++i) need[i] = ctx->needs_input_grad(i);
    const variable_list saved = ctx->get_saved_variables();
    variable_list grads;
    if (!at::GradMode::is_enabled()) {
      grads = op->backward(saved, g, need);
    } else {
      grads = in_python([&] {
        variable_list out;
        for (const py::handle& h : op->backward_in_python(saved, g, need)) out.push_back(h.is_none() ? Tensor() : h.cast<Tensor>());
        return out;
      });
    }
    grads.insert(grads.begin(), Tensor());  // the operation itself
    return grads;
  }
};

// the node type under the name that the function of the Python layer has
template <class Kind>
void name_nodes(const char* name) {
  static PyTypeObject type;
  torch::autograd::_initFunctionPyTypeObject(type, name, nullptr, nullptr);
  torch::autograd::registerCppFunction(typeid(torch::autograd::CppNode<OpFn<Kind>>), &type);
}

py::list flags(const std::vector<bool>& need) {
  py::list l;
  for (bool b : need) l.append(b);
  return l;
}

// ---- spherical harmonics --------------------------------------------------------------------------------------------------
struct Harmonics : torch::CustomClassHolder {
  std::vector<int32_t> ls;
  int normalize, normalization;
  int64_t width = 0;
  Harmonics(std::vector<int32_t> l, bool n, int c) : ls(std::move(l)), normalize(n), normalization(c) {
    for (int32_t v : ls) width += 2 * v + 1;
  }
  Tensor values(const Tensor& x) const {
    Tensor out = rows_like(x, x.size(0), width);
    OnDevice on(x);
    check(e3x_sh_forward(ls.data(), (int32_t)ls.size(), normalize, normalization, in(x), ptr(out), x.size(0), E3X_F32, stream_of(x)));
    return out;
  }
  Tensor gradient(const Tensor& x, const Tensor& g) const {
    Tensor gx = rows_like(x, x.size(0), 3);
    OnDevice on(x);
    check(e3x_sh_backward(ls.data(), (int32_t)ls.size(), normalize, normalization, in(x), in(g), ptr(gx), x.size(0), E3X_F32, stream_of(x)));
    return gx;
  }
};
using HarmonicsPtr = c10::intrusive_ptr<Harmonics>;

struct HarmonicsOp : Op {
  HarmonicsPtr cfg;
  explicit HarmonicsOp(HarmonicsPtr c) : cfg(std::move(c)) {}
  variable_list forward(const variable_list& in) override { return {cfg->values(in[0])}; }
  variable_list backward(const variable_list& saved, const variable_list& g, const std::vector<bool>&) override {
    return {cfg->gradient(saved[0], g[0].contiguous())};
  }
  py::object backward_in_python(const variable_list& saved, const variable_list& g, const std::vector<bool>&) override {
    return py::make_tuple(hook("harmonics_gradient")(saved[0], g[0], py::cast(cfg->ls), (bool)cfg->normalize, cfg->normalization));
  }
};

std::optional<Tensor> harmonics(const HarmonicsPtr& cfg, const Tensor& x) {
  if (x.dim() != 2 || x.size(1) != 3 || !plain(x, at::kFloat) || !plain_state()) return std::nullopt;
  py::gil_scoped_release no_gil;
  if (!recorded({&x})) return cfg->values(x);
  return OpFn<HarmonicsOp>::apply(c10::make_intrusive<HarmonicsOp>(cfg), x)[0];
}

// ---- tensor product plans ---------------------------------------------------------------------------------------------------
struct Plan : torch::CustomClassHolder {
  e3x_plan* const h;
  const int64_t in1_dim, in2_dim, out_dim, weight_numel;
  const bool in_parts, packs, node, shared, bf16;
  std::mutex mu;
  int fused_grad_w = -1, by_destination = -1, sh[2][3] = {{-1, -1, -1}, {-1, -1, -1}};  // kernels built on first use: -1 not asked yet
  Plan(intptr_t handle, int64_t d1, int64_t d2, int64_t d3, int64_t wn, bool parts, bool pk, bool nd, bool sh_w, bool half)
      : h((e3x_plan*)handle), in1_dim(d1), in2_dim(d2), out_dim(d3), weight_numel(wn), in_parts(parts), packs(pk), node(nd), shared(sh_w), bf16(half) {}
  ~Plan() override { e3x_tp_plan_destroy(h); }  // (a node may outlive the Python object)

  // (as _Plan.forward)
  Tensor forward(Tensor x1, Tensor x2, Tensor w) const {
    const int64_t Z = x1.size(0);
    Tensor out = rows_like(x1, Z, out_dim), ws;
    size_t sizes[2] = {in_parts ? e3x_tp_forward_workspace_bytes_for(h, Z) : e3x_tp_forward_workspace_bytes(h), 0};
    const int n = in_parts ? 2 : 1;
    if (in_parts) sizes[1] = e3x_tp_forward_workspace_bytes_for(h, -1);
    size_t ws_bytes = 0;
    if (sizes[0]) {
      for (int i = 0; i < n; ++i) {
        try {
          ws = bytes_like(x1, sizes[i]);
          ws_bytes = sizes[i];
          break;
        } catch (const c10::OutOfMemoryError&) {
          if (bf16 && i + 1 == n) throw;  // (fp32: the general kernel needs none)
        }
      }
      if (packs) {
        if (!aligned(x1)) x1 = x1.clone();
        if (!aligned(x2)) x2 = x2.clone();
      }
    }
    if (node) {
      if (!aligned(x1)) x1 = x1.clone();
      if (!aligned(w)) w = w.clone();
    }
    OnDevice on(x1);
    check(e3x_tp_forward_ws(h, in(x1), in(x2), in(w), ptr(out), Z, ptr(ws), ws_bytes, stream_of(x1)));
    return out;
  }

  // (as _Plan.backward_w_uvw, shared weights)
  Tensor weight_gradient(Tensor x1, Tensor x2, Tensor g, bool bf16_values = false) const {
    Tensor gw = at::empty({weight_numel}, x1.options().requires_grad(false));
    if (!aligned(x1)) x1 = x1.clone();
    if (!aligned(x2)) x2 = x2.clone();
    if (!aligned(g)) g = g.clone();
    OnDevice on(x1);
    check((bf16_values ? e3x_tp_backward_w_uvw_bf16_values : e3x_tp_backward_w_uvw)(h, in(x1), in(x2), in(g), ptr(gw), x1.size(0), stream_of(x1)));
    return gw;
  }
  // whether the plan has a kernel that is built on first use
  bool has(int& known, int (*prepare)(e3x_plan*), bool may_fail_to_build) {
    std::lock_guard<std::mutex> lock(mu);
    if (known < 0) {
      const int rc = prepare(h);
      if (rc != E3X_ERR_INVALID && !(may_fail_to_build && rc == E3X_ERR_COMPILE)) check(rc);
      known = rc == E3X_OK;
    }
    return known;
  }
};
using PlanPtr = c10::intrusive_ptr<Plan>;

// ---- dense products with shared weights -------------------------------------------------------------------------------------
// What a FullyConnectedTensorProduct keeps with its plans: plans of the product and of its input gradients by storage type,
// and the lists that permute its weights for the latter by device, each asked of Python on first use.
struct Dense : torch::CustomClassHolder {
  enum { OUT, X1, X2 };
  std::mutex mu;
  PlanPtr plans[2][3];
  std::vector<std::array<Tensor, 2>> perms;
  PlanPtr plan(const PyRef& tp, bool bf16, int which) {
    {
      std::lock_guard<std::mutex> lock(mu);
      if (plans[bf16][which]) return plans[bf16][which];
    }
    PlanPtr p = in_python([&] { return hook("plan")(tp.get(), bf16, which).cast<PlanPtr>(); });
    std::lock_guard<std::mutex> lock(mu);
    return plans[bf16][which] = p;
  }
  Tensor permuted(const PyRef& tp, const Tensor& w, int which) {
    Tensor index;
    {
      std::lock_guard<std::mutex> lock(mu);
      const size_t d = (size_t)w.device().index();
      if (d < perms.size()) index = perms[d][which - X1];
    }
    if (!index.defined()) {
      index = in_python([&] { return hook("weight_permutation")(tp.get(), w.device(), which).cast<Tensor>(); });
      std::lock_guard<std::mutex> lock(mu);
      if ((size_t)w.device().index() >= perms.size()) perms.resize((size_t)w.device().index() + 1);
      perms[(size_t)w.device().index()][which - X1] = index;
    }
    return w.index_select(0, index);
  }
  // (as _tp_gradients)
  Tensor grad_x1(const PyRef& tp, const Tensor& x2, const Tensor& w, const Tensor& g) {
    return plan(tp, g.scalar_type() == at::kBFloat16, X1)->forward(g, x2, permuted(tp, w, X1));
  }
  Tensor grad_x2(const PyRef& tp, const Tensor& x1, const Tensor& w, const Tensor& g) {
    return plan(tp, g.scalar_type() == at::kBFloat16, X2)->forward(x1, g, permuted(tp, w, X2));
  }
  Tensor grad_w(const PyRef& tp, const Tensor& x1, const Tensor& x2, const Tensor& g) {
    PlanPtr p = plan(tp, false, OUT);
    if (g.scalar_type() == at::kFloat) return p->weight_gradient(x1, x2, g);
    return p->weight_gradient(x1.to(at::kFloat), x2.to(at::kFloat), g.to(at::kFloat), g.scalar_type() == at::kBFloat16).to(g.scalar_type());
  }
};
using DensePtr = c10::intrusive_ptr<Dense>;

struct DenseOp : Op {
  DensePtr d;
  PyRef tp;
  DenseOp(DensePtr d_, const py::handle& tp_) : d(std::move(d_)), tp(tp_) {}
  variable_list forward(const variable_list& in) override {
    return {d->plan(tp, in[0].scalar_type() == at::kBFloat16, Dense::OUT)->forward(in[0], in[1], in[2])};
  }
  variable_list backward(const variable_list& s, const variable_list& gs, const std::vector<bool>& need) override {
    const Tensor g = gs[0].contiguous();
    variable_list out(3);
    if (need[2]) out[2] = d->grad_w(tp, s[0], s[1], g);
    if (need[0]) out[0] = d->grad_x1(tp, s[1], s[2], g);
    if (need[1]) out[1] = d->grad_x2(tp, s[0], s[2], g);
    return out;
  }
  py::object backward_in_python(const variable_list& s, const variable_list& g, const std::vector<bool>& need) override {
    return hook("dense_gradients")(tp.get(), py::cast(s), g[0], flags(need));
  }
};

std::optional<Tensor> dense(const DensePtr& d, const py::object& tp, int64_t d1, int64_t d2, int64_t wn, const Tensor& x, const Tensor& y, const Tensor& w) {
  const at::ScalarType dt = x.scalar_type();
  if ((dt != at::kFloat && dt != at::kBFloat16) || x.dim() != 2 || y.dim() != 2 || x.size(0) != y.size(0) || x.size(1) != d1 || y.size(1) != d2 ||
      w.dim() != 1 || w.size(0) != wn || !plain(x, dt) || !plain(y, dt) || !plain(w, dt) || x.device() != y.device() || x.device() != w.device() || !plain_state())
    return std::nullopt;
  auto op = c10::make_intrusive<DenseOp>(d, tp);
  py::gil_scoped_release no_gil;
  if (!recorded({&x, &y, &w})) return op->forward({x, y, w})[0];
  return OpFn<DenseOp>::apply(op, x, y, w)[0];
}

// ---- message step ---------------------------------------------------------------------------------------------------------------
// tensors of a DstSortedEdges
struct Edges : torch::CustomClassHolder {
  Tensor src, dst, rowptr, perm, walk_perm, row_order, src_rows;  // walk_perm, row_order, src_rows: undefined where there is none
  int64_t num_edges, num_nodes, num_src_nodes;
  Edges(Tensor s, Tensor d, Tensor r, Tensor p, std::optional<Tensor> wp, std::optional<Tensor> ro, std::optional<Tensor> sr, int64_t E, int64_t N, int64_t NS)
      : src(std::move(s)), dst(std::move(d)), rowptr(std::move(r)), perm(std::move(p)), walk_perm(wp.value_or(Tensor())), row_order(ro.value_or(Tensor())),
        src_rows(sr.value_or(Tensor())), num_edges(E), num_nodes(N), num_src_nodes(NS) {}
};
using EdgesPtr = c10::intrusive_ptr<Edges>;
int bits(const Tensor& idx) { return (int)idx.element_size() * 8; }

struct Message : torch::CustomClassHolder {  // plans of a message step, by storage type
  std::mutex mu;
  PlanPtr plans[2], grad_x1;  // (grad_x1: fp32)
  PlanPtr plan(const PyRef& tp, bool bf16, bool transposed) {
    PlanPtr& slot = transposed ? grad_x1 : plans[bf16];
    {
      std::lock_guard<std::mutex> lock(mu);
      if (slot) return slot;
    }
    PlanPtr p = in_python([&] { return hook("plan")(tp.get(), bf16, transposed ? 1 : 0).cast<PlanPtr>(); });
    std::lock_guard<std::mutex> lock(mu);
    return slot = p;
  }
};
using MessagePtr = c10::intrusive_ptr<Message>;

// sum over edges of plan(table[src], attr, w) (as _Plan.gather_scatter), or, with `normalization` >= 0, of harmonics of edge vectors
Tensor gather_scatter(Plan& p, const Tensor& table, const Tensor& attr, const Tensor& w, const Edges& e, int normalize, int normalization) {
  Tensor out = rows_like(table, e.num_nodes, p.out_dim);
  OnDevice on(table);
  if (normalization >= 0) {
    check(e3x_tp_gather_scatter_sh(p.h, in(table), ptr_as<float>(attr), in(w), in(e.src), bits(e.src), ptr_as<int32_t>(e.rowptr), ptr_as<int32_t>(e.walk_perm),
                                   ptr_as<int32_t>(e.row_order), ptr_as<int32_t>(e.src_rows), ptr(out), e.num_edges, table.size(0), e.num_nodes, normalize,
                                   normalization, stream_of(table)));
    return out;
  }
  const size_t ws_bytes = e3x_tp_gather_scatter_workspace_bytes(p.h, table.size(0));
  Tensor ws;
  if (ws_bytes) ws = bytes_like(table, ws_bytes);
  check(e3x_tp_gather_scatter_ws(p.h, in(table), in(attr), in(w), in(e.src), bits(e.src), ptr_as<int32_t>(e.rowptr), ptr_as<int32_t>(e.walk_perm),
                                 ptr_as<int32_t>(e.row_order), ptr_as<int32_t>(e.src_rows), ptr(out), e.num_edges, table.size(0), e.num_nodes, ptr(ws), ws_bytes,
                                 stream_of(table)));
  return out;
}

struct MessageOp : Op {
  MessagePtr m;
  PyRef tp, edges;  // the Python objects
  EdgesPtr e;
  HarmonicsPtr sh;  // of the edge vectors, formed in the forward kernel; null: the attributes are given
  MessageOp(MessagePtr m_, const py::handle& tp_, const py::handle& edges_, EdgesPtr e_, HarmonicsPtr s)
      : m(std::move(m_)), tp(tp_), edges(edges_), e(std::move(e_)), sh(std::move(s)) {}
  variable_list forward(const variable_list& in) override {
    PlanPtr p = m->plan(tp, in[0].scalar_type() == at::kBFloat16, false);
    return {gather_scatter(*p, in[0], in[1], in[2], *e, sh ? sh->normalize : 0, sh ? sh->normalization : -1)};
  }
  EdgesPtr transposed() const {
    return in_python([&] { return edges.get().attr("transposed")().attr("native")().cast<EdgesPtr>(); });
  }
  variable_list backward(const variable_list& s, const variable_list& gs, const std::vector<bool>& need) override {
    const Tensor g = gs[0].contiguous();
    const Tensor &x = s[0], &w = s[2];
    const Tensor attr = sh ? sh->values(s[1]).to(x.scalar_type()) : s[1];
    const bool want_attr = need[1] && attr.size(1) > 0;
    Tensor g1, g2, gw;
    // every gradient from one pass over the weights (as _message_gradients); other cases are Python's
    bool done = false;
    if (need[0] && need[2] && w.size(1) > 0) {
      const bool bf16 = x.scalar_type() == at::kBFloat16;
      PlanPtr p = m->plan(tp, bf16, false);
      const size_t ws_bytes = e3x_tp_message_backward_workspace_bytes(p->h, e->num_edges);
      const EdgesPtr t = transposed();
      if (ws_bytes && p->has(p->by_destination, e3x_tp_plan_prepare_message_backward, true)) {
        try {
          g1 = at::empty_like(x), gw = at::empty_like(w);
          if (want_attr) g2 = at::empty_like(attr);
          Tensor ws = bytes_like(x, ws_bytes);
          OnDevice on(x);
          check(e3x_tp_message_backward(p->h, in(x), in(attr), in(w), in(g), in(e->src), bits(e->src), ptr_as<int32_t>(e->rowptr), ptr_as<int32_t>(e->walk_perm),
                                        ptr_as<int32_t>(e->row_order), ptr_as<int32_t>(e->src_rows), ptr_as<int32_t>(t->rowptr), ptr_as<int32_t>(t->walk_perm), ptr(g1),
                                        ptr(gw), ptr(g2), e->num_edges, x.size(0), e->num_nodes, ptr(ws), ws_bytes, stream_of(x)));
          done = true;
        } catch (const c10::OutOfMemoryError&) {  // the kernels on the transposed plan need the gradients but no scratch
          g1 = g2 = gw = Tensor();
        }
      }
      if (!done) {
        PlanPtr q = m->plan(tp, bf16, true);
        if (q->has(q->fused_grad_w, e3x_tp_plan_prepare_gather_scatter_grad_w, bf16)) {
          g1 = rows_like(g, t->num_nodes, q->out_dim), gw = rows_like(g, t->num_edges, q->weight_numel);
          if (want_attr) g2 = at::empty_like(attr);
          OnDevice on(x);
          check(e3x_tp_gather_scatter_grad_w(q->h, in(g), in(attr), in(w), in(x), in(e->dst), bits(e->dst), ptr_as<int32_t>(t->rowptr), ptr_as<int32_t>(t->walk_perm),
                                             ptr_as<int32_t>(t->row_order), ptr_as<int32_t>(t->src_rows), ptr(g1), ptr(gw), ptr(g2), t->num_edges, g.size(0),
                                             t->num_nodes, stream_of(x)));
          done = true;
        }
      }
    }
    if (!done) {
      in_python([&] {
        py::tuple r = hook("message_gradients")(tp.get(), edges.get(), x, attr, w, g, (bool)need[0], (bool)need[1], (bool)need[2]);
        Tensor* to[3] = {&g1, &g2, &gw};
        for (int i = 0; i < 3; ++i)
          if (!r[i].is_none()) *to[i] = r[i].cast<Tensor>();
      });
    }
    if (need[2] && !gw.defined()) gw = at::zeros_like(w);
    if (sh && g2.defined()) g2 = sh->gradient(s[1], g2.to(at::kFloat));
    return {g1, g2, gw};
  }
  py::object backward_in_python(const variable_list& s, const variable_list& g, const std::vector<bool>& need) override {
    if (sh) return hook("message_sh_gradients")(tp.get(), edges.get(), py::cast(s), g[0], flags(need), (bool)sh->normalize, sh->normalization);
    return hook("message_gradients_graph")(tp.get(), edges.get(), py::cast(s), g[0], flags(need));
  }
};

std::optional<Tensor> message(const MessagePtr& m, const py::object& tp, const py::object& edges, const EdgesPtr& e, int64_t d1, int64_t d2, int64_t wn, const Tensor& x,
                              const Tensor& attr, const Tensor& w, const std::optional<HarmonicsPtr>& sh) {
  const at::ScalarType dt = x.scalar_type();
  if ((dt != at::kFloat && dt != at::kBFloat16) || x.dim() != 2 || x.size(1) != d1 || x.size(0) != e->num_src_nodes || attr.dim() != 2 ||
      attr.size(0) != e->num_edges || attr.size(1) != (sh ? 3 : d2) || w.dim() != 2 || w.size(0) != e->num_edges || w.size(1) != wn || !plain(x, dt) ||
      !plain(attr, sh ? at::kFloat : dt) || !plain(w, dt) || x.device() != attr.device() || x.device() != w.device() || x.device() != e->rowptr.device() || !plain_state())
    return std::nullopt;
  auto op = c10::make_intrusive<MessageOp>(m, tp, edges, e, sh.value_or(HarmonicsPtr()));
  py::gil_scoped_release no_gil;
  if (sh) {  // (a set whose second input is not harmonics is refused in Python)
    PlanPtr p = m->plan(op->tp, dt == at::kBFloat16, false);
    std::lock_guard<std::mutex> lock(p->mu);
    int& known = p->sh[(*sh)->normalize][(*sh)->normalization];
    if (known < 0) {
      const int rc = e3x_tp_plan_prepare_gather_scatter_sh(p->h, (*sh)->normalize, (*sh)->normalization);
      if (rc != E3X_ERR_INVALID) check(rc);
      known = rc == E3X_OK;
    }
    if (!known) return std::nullopt;
  }
  if (!recorded({&x, &attr, &w})) return op->forward({x, attr, w})[0];
  return OpFn<MessageOp>::apply(op, x, attr, w)[0];
}

// rowptr, perm, row_order (or None), grouped, pairs of e3x_edges_build
py::tuple edges_build(const Tensor& src, const Tensor& dst, int64_t num_nodes, int64_t num_src_nodes, bool order) {
  const int64_t E = src.numel();
  const auto opt = src.options().dtype(at::kInt).requires_grad(false);
  Tensor rowptr, perm, row_order;
  int32_t grouped = 0, pairs = 0;
  {
    py::gil_scoped_release no_gil;
    OnDevice on(src);
    rowptr = at::empty({num_nodes + 1}, opt), perm = at::empty({E}, opt);
    if (order) row_order = at::empty({num_nodes}, opt);
    const size_t ws_bytes = e3x_edges_workspace_bytes(E, num_nodes);
    Tensor ws = bytes_like(src, ws_bytes);
    check(e3x_edges_build(in(src), bits(src), in(dst), bits(dst), E, num_nodes, num_src_nodes, ptr_as<int32_t>(rowptr), ptr_as<int32_t>(perm),
                          ptr_as<int32_t>(row_order), &grouped, &pairs, ptr(ws), ws_bytes, stream_of(src)));
  }
  return py::make_tuple(rowptr, perm, row_order.defined() ? py::cast(row_order) : py::none(), grouped, pairs);
}

// ---- dense layers of scalars -------------------------------------------------------------------------------------------------------
struct FcPlan : torch::CustomClassHolder {
  e3x_fc_plan* const h;
  const int64_t in_dim, out_dim;
  const size_t ws_bytes;
  FcPlan(intptr_t handle, int64_t i, int64_t o, size_t ws) : h((e3x_fc_plan*)handle), in_dim(i), out_dim(o), ws_bytes(ws) {}
  ~FcPlan() override { e3x_fc_plan_destroy(h); }
  Tensor forward(const Tensor& x, const variable_list& weights, const Tensor& z) const {
    Tensor out = rows_like(x, x.size(0), out_dim), ws = bytes_like(x, ws_bytes);
    std::vector<const void*> w_ptr;
    for (const Tensor& w : weights) w_ptr.push_back(in(w));
    OnDevice on(x);
    check(e3x_fc_forward_epilogue(h, in(x), w_ptr.data(), in(z), ptr(out), x.size(0), ptr(ws), ws_bytes, stream_of(x)));
    return out;
  }
  Tensor weight_gradient(const Tensor& x, const Tensor& g) const {
    Tensor gw = rows_like(x, in_dim, out_dim);
    OnDevice on(x);
    check(e3x_fc_backward_w(h, in(x), in(g), ptr(gw), x.size(0), stream_of(x)));
    return gw;
  }
};
using FcPlanPtr = c10::intrusive_ptr<FcPlan>;
Tensor in_16_byte_rows(const Tensor& t) {
  const Tensor c = t.contiguous();
  return aligned(c) ? c : c.clone();
}

std::optional<Tensor> fc_forward(const FcPlanPtr& p, const Tensor& x, const std::vector<Tensor>& weights) {
  if (x.dim() != 2 || x.size(1) != p->in_dim || !plain(x, at::kFloat) || !aligned(x) || !plain_state()) return std::nullopt;
  bool grad = x.requires_grad();
  for (const Tensor& w : weights) {
    if (!plain(w, at::kFloat) || w.device() != x.device()) return std::nullopt;
    grad = grad || w.requires_grad();
  }
  if (weights.empty() || weights.back().size(-1) != p->out_dim || (grad && at::GradMode::is_enabled())) return std::nullopt;
  py::gil_scoped_release no_gil;
  return p->forward(x, weights, Tensor());
}

// one layer, x @ W * s (z = false), or act(x) @ W * s of the pre-activations of the layer in front (z = true): _DenseSlot, _ActDenseFn
struct LayerOp : Op {
  FcPlanPtr fwd, bwd;
  double scale;
  PyRef layer, prev;  // prev: None without an activation in front
  LayerOp(FcPlanPtr f, FcPlanPtr b, double s, const py::handle& l, const py::handle& q) : fwd(std::move(f)), bwd(std::move(b)), scale(s), layer(l), prev(q) {}
  variable_list forward(const variable_list& in) override { return {fwd->forward(in[0], {in[1].contiguous()}, Tensor())}; }
  variable_list backward(const variable_list& s, const variable_list& gs, const std::vector<bool>& need) override {
    const Tensor g = in_16_byte_rows(gs[0]);
    variable_list out(2);
    if (need[0]) out[0] = bwd->forward(g, {s[1].t().mul(scale).contiguous()}, prev.p == Py_None ? Tensor() : s[0]);
    if (need[1]) out[1] = fwd->weight_gradient(s[0], g);
    return out;
  }
  py::object backward_in_python(const variable_list& s, const variable_list& g, const std::vector<bool>& need) override {
    return hook("layer_gradients")(layer.get(), prev.get(), py::cast(s), g[0], flags(need));
  }
};
struct ActLayerOp : LayerOp {
  using LayerOp::LayerOp;
};
template <class Kind>
Tensor run_layer(const FcPlanPtr& f, const FcPlanPtr& b, double scale, const py::object& layer, const py::object& prev, const Tensor& x, const Tensor& w) {
  auto op = c10::make_intrusive<Kind>(f, b, scale, layer, prev);
  py::gil_scoped_release no_gil;
  return recorded({&x, &w}) ? OpFn<Kind>::apply(op, x, w)[0] : op->forward({x, w})[0];
}
std::optional<Tensor> fc_layer(const FcPlanPtr& f, const FcPlanPtr& b, double scale, const py::object& layer, const py::object& prev, const Tensor& x, const Tensor& w) {
  if (x.dim() != 2 || x.size(1) != f->in_dim || !plain(x, at::kFloat) || !aligned(x) || !plain(w, at::kFloat) || w.dim() != 2 || w.size(0) != f->in_dim ||
      w.size(1) != f->out_dim || w.device() != x.device() || !plain_state())
    return std::nullopt;
  return prev.is_none() ? run_layer<LayerOp>(f, b, scale, layer, prev, x, w) : run_layer<ActLayerOp>(f, b, scale, layer, prev, x, w);
}

// ---- mixing of a convolution block (_Mix) -------------------------------------------------------------------------------------------
struct MixOp : Op {
  variable_list forward(const variable_list& t) override {
    Tensor out = at::empty_like(t[0]);
    OnDevice on(out);
    check(e3x_mix_forward(ptr_as<float>(t[0]), ptr_as<float>(t[1]), ptr_as<float>(t[2]), ptr_as<float>(t[3]), ptr_as<float>(t[4]), ptr_as<float>(out), t[0].size(0), t[0].size(1), stream_of(out)));
    return {out};
  }
  variable_list to_save(const variable_list& t) override { return {t[1], t[2], t[3], t[4]}; }
  variable_list backward(const variable_list& s, const variable_list& gs, const std::vector<bool>& need) override {
    const Tensor g = gs[0].contiguous();
    variable_list out(5);
    if (need[0]) out[0] = gs[0];
    if (need[1]) out[1] = at::empty_like(s[0]);
    if (need[2]) out[2] = at::empty_like(s[1]);
    OnDevice on(g);
    check(e3x_mix_backward(ptr_as<float>(g), ptr_as<float>(s[0]), ptr_as<float>(s[1]), ptr_as<float>(s[2]), ptr_as<float>(s[3]), ptr_as<float>(out[1]), ptr_as<float>(out[2]), s[1].size(0), s[1].size(1), stream_of(g)));
    return out;
  }
  py::object backward_in_python(const variable_list& s, const variable_list& g, const std::vector<bool>& need) override {
    return hook("mix_gradients")(py::cast(s), g[0], flags(need));
  }
};
std::optional<Tensor> mix(const Tensor& rows, const Tensor& alpha, const Tensor& conv, const Tensor& c0, const Tensor& c1) {
  if (rows.dim() != 2 || rows.sizes() != conv.sizes() || alpha.dim() != 2 || alpha.size(0) != rows.size(0) || alpha.size(1) != 1 || c0.dim() != 1 ||
      c0.size(0) != rows.size(1) || c1.sizes() != c0.sizes() || rows.numel() == 0)
    return std::nullopt;
  for (const Tensor* t : {&rows, &alpha, &conv, &c0, &c1})
    if (!plain(*t, at::kFloat) || t->device() != rows.device()) return std::nullopt;
  if (c0.requires_grad() || c1.requires_grad() || !plain_state()) return std::nullopt;
  auto op = c10::make_intrusive<MixOp>();
  py::gil_scoped_release no_gil;
  if (!recorded({&rows, &alpha, &conv})) return op->forward({rows, alpha, conv, c0, c1})[0];
  return OpFn<MixOp>::apply(op, rows, alpha, conv, c0, c1)[0];
}

// ---- lin2 and alpha of a convolution block as one node (_Lin2Alpha) -----------------------------------------------------------------
struct Lin2AlphaOp : Op {
  DensePtr lin2, reads, head;
  PyRef lin2_tp, reads_tp, head_tp, alpha_tp;
  int64_t k;  // leading scalars
  bool in_place;
  Lin2AlphaOp(DensePtr l, DensePtr r, DensePtr h, const py::handle& lt, const py::handle& rt, const py::handle& ht, const py::handle& at_, int64_t k_, bool ip)
      : lin2(std::move(l)), reads(std::move(r)), head(std::move(h)), lin2_tp(lt), reads_tp(rt), head_tp(ht), alpha_tp(at_), k(k_), in_place(ip) {}
  Tensor scalars(const Tensor& f) const { return in_place ? f : f.narrow(1, 0, k).contiguous(); }
  Tensor kept;  // the scalars of the forward pass where they are a copy: handed to to_save, not kept
  variable_list forward(const variable_list& in) override {
    kept = scalars(in[0]);
    return {lin2->plan(lin2_tp, false, Dense::OUT)->forward(in[0], in[1], in[2]), reads->plan(reads_tp, false, Dense::OUT)->forward(kept, in[1], in[3])};
  }
  variable_list to_save(const variable_list& in) override {
    Tensor s = in_place ? in[0] : std::move(kept);
    kept = Tensor();
    return {in[0], in[1], in[2], in[3], s};
  }
  variable_list backward(const variable_list& s, const variable_list& gs, const std::vector<bool>& need) override {
    const Tensor g_conv = gs[0].contiguous(), g_alpha = gs[1].contiguous();
    variable_list out(4);
    if (need[2]) out[2] = lin2->grad_w(lin2_tp, s[0], s[1], g_conv);
    if (need[3]) out[3] = reads->grad_w(reads_tp, s[4], s[1], g_alpha);
    if (need[0]) {
      out[0] = lin2->grad_x1(lin2_tp, s[1], s[2], g_conv);
      out[0].narrow(1, 0, k).add_(head->grad_x1(head_tp, s[1], s[3], g_alpha));
    }
    return out;
  }
  py::object backward_in_python(const variable_list& s, const variable_list& g, const std::vector<bool>& need) override {
    return hook("lin2_alpha_gradients")(lin2_tp.get(), head_tp.get(), py::cast(s), g[0], g[1], flags(need));
  }
};
std::optional<std::pair<Tensor, Tensor>> lin2_alpha(const DensePtr& l, const DensePtr& r, const DensePtr& h, const py::object& lt, const py::object& rt, const py::object& ht,
                                                    const py::object& at_, int64_t k, bool in_place, const Tensor& f, const Tensor& attr, const Tensor& w2, const Tensor& wa) {
  for (const Tensor* t : {&f, &attr, &w2, &wa})
    if (!plain(*t, at::kFloat) || t->device() != f.device()) return std::nullopt;
  if (f.dim() != 2 || attr.dim() != 2 || attr.size(0) != f.size(0) || attr.requires_grad() || !plain_state()) return std::nullopt;
  auto op = c10::make_intrusive<Lin2AlphaOp>(l, r, h, lt, rt, ht, at_, k, in_place);
  py::gil_scoped_release no_gil;
  variable_list out = OpFn<Lin2AlphaOp>::apply(op, f, attr, w2, wa);
  return std::make_pair(out[0], out[1]);
}

template <class F>
auto wrapped(F* f) { return torch::wrap_pybind_function(f); }
}  // namespace

PYBIND11_MODULE(_e3x_host, m) {
  py::class_<Harmonics, HarmonicsPtr>(m, "Harmonics").def(py::init<std::vector<int32_t>, bool, int>());
  py::class_<Plan, PlanPtr>(m, "Plan").def(py::init<intptr_t, int64_t, int64_t, int64_t, int64_t, bool, bool, bool, bool, bool>());
  py::class_<Dense, DensePtr>(m, "Dense").def(py::init<>());
  py::class_<Message, MessagePtr>(m, "Message").def(py::init<>());
  py::class_<Edges, EdgesPtr>(m, "Edges")
      .def(py::init<Tensor, Tensor, Tensor, Tensor, std::optional<Tensor>, std::optional<Tensor>, std::optional<Tensor>, int64_t, int64_t, int64_t>());
  py::class_<FcPlan, FcPlanPtr>(m, "FcPlan").def(py::init<intptr_t, int64_t, int64_t, size_t>());
  // the Python functions that nodes call: differentiable backward passes, plans on first use
  m.def("connect", [](const py::dict& d) {
    if (!hooks) hooks = new py::dict();  // (lives as long as the process)
    for (const auto& item : d) (*hooks)[item.first] = item.second;
  });
  name_nodes<HarmonicsOp>("_SphericalHarmonicsFnBackward");
  name_nodes<DenseOp>("_TpSlotBackward");
  name_nodes<MessageOp>("_MessageSlotBackward");
  name_nodes<LayerOp>("_DenseSlotBackward");
  name_nodes<ActLayerOp>("_ActDenseFnBackward");
  name_nodes<MixOp>("_MixBackward");
  name_nodes<Lin2AlphaOp>("_Lin2AlphaBackward");
  m.def("harmonics", wrapped(harmonics));
  m.def("dense", wrapped(dense));
  m.def("message", wrapped(message));
  m.def("edges_build", wrapped(edges_build));
  m.def("fc_forward", wrapped(fc_forward));
  m.def("fc_layer", wrapped(fc_layer));
  m.def("mix", wrapped(mix));
  m.def("lin2_alpha", wrapped(lin2_alpha));
}
