// torch_binding.cpp — the differentiable ops of the torch front-end as C++ autograd functions over
// the C ABI (include/msda.h), for the calls that need nothing from Python.
//
// A training step of one op took 65-158 us on the host (Python's autograd.Function, its argument
// handling and 18-argument ctypes calls, in both directions) around 15-60 us of kernels. Each entry
// point here first looks whether the call is an ordinary one: plain GPU tensors of the expected
// types, shapes and layouts, no functorch transform, forward-mode tangent, dispatch or function mode,
// and no tracing. It returns None otherwise, and the caller takes the Python path, which converts,
// checks and reports errors; so nothing is refused or accepted here that is not there.
//
// The kernel library is not linked: bind() receives the addresses of its functions from the loaded
// library (rfdetr_jax_amd/_native.py).
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/extension.h>

#include <array>
#include <optional>
#include <vector>

#include "msda.h"

namespace {

namespace py = pybind11;
using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

struct Library {
  decltype(&msda_fwd) fwd;
  decltype(&msda_fwd_sampler) fwd_sampler;
  decltype(&msda_bwd) bwd;
  decltype(&msda_bwd_sampler) bwd_sampler;
  decltype(&msda_bwd_workspace_size) bwd_workspace_size;
  decltype(&msda_fused_fwd) fused_fwd;
  decltype(&msda_fused_bwd) fused_bwd;
  decltype(&msda_fused_bwd_workspace_size) fused_bwd_workspace_size;
  decltype(&msda_grid_sample_fwd) grid_sample_fwd;
  decltype(&msda_grid_sample_bwd) grid_sample_bwd;
  decltype(&msda_value_proj_fwd) value_proj_fwd;
  decltype(&msda_value_proj_bwd) value_proj_bwd;
  decltype(&msda_value_proj_bwd_workspace_size) value_proj_bwd_workspace_size;
  decltype(&msda_attention_fwd) attention_fwd;
  decltype(&msda_attention_bwd) attention_bwd;
};

Library lib;
PyObject* check_status = nullptr;    // _native.check: raises MsdaError for a status other than 0
PyTypeObject* parameter_type = nullptr;

void bind(const py::dict& address, const py::object& check, const py::object& parameter) {
  auto get = [&](const char* name, auto& fn) { fn = reinterpret_cast<std::decay_t<decltype(fn)>>(address[name].cast<uintptr_t>()); };
  get("msda_fwd", lib.fwd);
  get("msda_fwd_sampler", lib.fwd_sampler);
  get("msda_bwd", lib.bwd);
  get("msda_bwd_sampler", lib.bwd_sampler);
  get("msda_bwd_workspace_size", lib.bwd_workspace_size);
  get("msda_fused_fwd", lib.fused_fwd);
  get("msda_fused_bwd", lib.fused_bwd);
  get("msda_fused_bwd_workspace_size", lib.fused_bwd_workspace_size);
  get("msda_grid_sample_fwd", lib.grid_sample_fwd);
  get("msda_grid_sample_bwd", lib.grid_sample_bwd);
  get("msda_value_proj_fwd", lib.value_proj_fwd);
  get("msda_value_proj_bwd", lib.value_proj_bwd);
  get("msda_value_proj_bwd_workspace_size", lib.value_proj_bwd_workspace_size);
  get("msda_attention_fwd", lib.attention_fwd);
  get("msda_attention_bwd", lib.attention_bwd);
  check_status = py::object(check).release().ptr();
  parameter_type = reinterpret_cast<PyTypeObject*>(py::object(parameter).release().ptr());
}

// Raises the Python exception of a failed call (its message is this thread's msda_last_error), from
// a Python caller or from an autograd thread, which does not hold the interpreter lock.
void check(int64_t status) {
  if (status >= 0) return;
  py::gil_scoped_acquire lock;
  PyObject* r = PyObject_CallFunction(check_status, "L", static_cast<long long>(status));
  if (r != nullptr) {
    Py_DECREF(r);
    throw std::runtime_error("msda call failed");
  }
  python_error e;
  e.persist();
  throw e;
}

// One library call on the tensor's device and current stream, without the interpreter lock (a full
// launch queue blocks).
template <typename F>
void launch(const Tensor& t, F&& f) {
  int rc;
  {
    std::optional<py::gil_scoped_release> unlocked;
    if (PyGILState_Check() != 0) unlocked.emplace();
    const c10::DeviceGuard guard(t.device());
    rc = f(static_cast<void*>(c10::hip::getCurrentHIPStream(t.device().index()).stream()));
  }
  check(rc);
}

// ---- what makes a call an ordinary one --------------------------------------------------------

bool ordinary_state() {
  const auto& tls = c10::impl::tls_local_dispatch_key_set();
  return lib.fwd != nullptr && !c10::impl::TorchDispatchModeTLS::any_modes_set() && at::impl::PythonTorchFunctionTLS::stack_len() == 0 &&
         !tls.included_.has(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) && !tls.included_.has(c10::DispatchKey::Functionalize) &&
         !torch::jit::tracer::isTracing();
}

// A plain GPU tensor (torch.Tensor or nn.Parameter themselves, no subclass) with elements; null otherwise.
const Tensor* plain(const py::handle& h) {
  PyTypeObject* type = Py_TYPE(h.ptr());
  if (!THPVariable_CheckTypeExact(type) && type != parameter_type) return nullptr;
  const Tensor& t = THPVariable_Unpack(h.ptr());
  static const c10::DispatchKeySet wrapped({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::FuncTorchBatched,
                                            c10::DispatchKey::Functionalize, c10::DispatchKey::Batched});
  if (!t.defined() || !t.is_cuda() || t.layout() != c10::kStrided || t.is_neg() || t.key_set().has_any(wrapped) || t.numel() == 0 ||
      t._fw_grad(0).defined())
    return nullptr;
  return &t;
}

bool f32(const Tensor& t) { return t.scalar_type() == at::kFloat; }
bool value_type(const Tensor& t) { return t.scalar_type() == at::kFloat || t.scalar_type() == at::kBFloat16; }
int code(const Tensor& t) { return t.scalar_type() == at::kBFloat16 ? MSDA_DTYPE_BF16 : MSDA_DTYPE_F32; }

// (H, W) pairs of Python ints, and the levels' first rows
struct Levels {
  std::vector<int32_t> shapes, starts;
  int64_t positions = 0;
};

bool levels_of(const py::handle& h, Levels& out) {
  if (!PyTuple_CheckExact(h.ptr()) && !PyList_CheckExact(h.ptr())) return false;
  for (const py::handle& pair : py::reinterpret_borrow<py::sequence>(h)) {
    if ((!PyTuple_CheckExact(pair.ptr()) && !PyList_CheckExact(pair.ptr())) || PySequence_Size(pair.ptr()) != 2) return false;
    out.starts.push_back(static_cast<int32_t>(out.positions));
    int64_t cells = 1;
    for (const py::handle& x : py::reinterpret_borrow<py::sequence>(pair)) {
      if (!PyLong_CheckExact(x.ptr())) return false;
      const int64_t n = PyLong_AsLongLong(x.ptr());
      if (n < 1 || n > (1 << 20)) {
        PyErr_Clear();
        return false;
      }
      out.shapes.push_back(static_cast<int32_t>(n));
      cells *= n;
    }
    out.positions += cells;
    if (out.positions >= (int64_t{1} << 31)) return false;
  }
  return !out.starts.empty();
}

struct Dims {  // of the deformable attention, as the C ABI takes them
  int batch, heads, head_dim, queries, levels, points;
  int64_t positions;
  std::vector<int32_t> shapes, starts;
};

// value [B * H, S, D], samples [B, Q, H, L, P, 2], weights [B, Q, H, L * P], contiguous
bool dims_of(const Tensor& value, const Tensor& samples, const Tensor& weights, Levels&& lv, Dims& d) {
  if (value.dim() != 3 || samples.dim() != 6 || weights.dim() != 4 || !value_type(value) || !f32(samples) || !f32(weights)) return false;
  if (!value.is_contiguous() || !samples.is_contiguous() || !weights.is_contiguous()) return false;
  if (samples.device() != value.device() || weights.device() != value.device()) return false;
  const auto s = samples.sizes();
  for (int64_t n : s)
    if (n >= (int64_t{1} << 31)) return false;
  if (s[5] != 2 || s[3] != static_cast<int64_t>(lv.starts.size()) || value.size(0) != s[0] * s[2] || value.size(1) != lv.positions ||
      value.size(2) >= (int64_t{1} << 31))
    return false;
  if (weights.size(0) != s[0] || weights.size(1) != s[1] || weights.size(2) != s[2] || weights.size(3) != s[3] * s[4]) return false;
  d = Dims{static_cast<int>(s[0]), static_cast<int>(s[2]), static_cast<int>(value.size(2)), static_cast<int>(s[1]),
           static_cast<int>(s[3]), static_cast<int>(s[4]), lv.positions, std::move(lv.shapes), std::move(lv.starts)};
  return true;
}

// at least `bytes`, in whole 16-byte rows
Tensor workspace(int64_t bytes, const Tensor& like) {
  return at::empty({std::max<int64_t>(1, (bytes + 15) / 16), 4}, like.options().dtype(at::kInt));
}

void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
float* fptr(const Tensor& t) { return static_cast<float*>(ptr(t)); }
Tensor like_if(bool wanted, const Tensor& t) { return wanted ? at::empty_like(t, t.options(), at::MemoryFormat::Contiguous) : Tensor(); }

// the cotangent of an output, in the type and layout that the kernels read
Tensor cotangent(const Tensor& g, at::ScalarType type) { return g.to(type).contiguous(); }

// A saved tensor in the type and layout that the kernels read. Hooks on saved tensors (offloading,
// compression) hand back tensors of their own making: the values may come in another layout or type,
// and anything else that the kernels would read past is refused (saved_as).
Tensor restored(const Tensor& t, at::ScalarType type) {
  TORCH_CHECK(t.defined() && t.is_cuda(), "a saved tensor came back on another device than the GPU; the HIP kernels need GPU tensors");
  return t.scalar_type() == type && t.is_contiguous() ? t : t.to(type).contiguous();
}

void saved_as(bool expected) { TORCH_CHECK_VALUE(expected, "saved tensors came back with other shapes, or on other devices, than they were saved"); }

// ---- the deformable-attention core ------------------------------------------------------------

struct Core : torch::autograd::Function<Core> {
  static Tensor forward(AutogradContext* ctx, const Tensor& value, const Tensor& loc, const Tensor& attn, const Dims& d, int64_t sampler) {
    Tensor out = at::empty({d.batch, d.queries, int64_t{d.heads} * d.head_dim}, loc.options());
    launch(value, [&](void* st) {
      return sampler == 0 ? lib.fwd(ptr(value), code(value), fptr(loc), fptr(attn), ptr(out), MSDA_DTYPE_F32, d.batch, d.heads, d.head_dim,
                                    d.queries, d.levels, d.points, d.shapes.data(), d.starts.data(), d.positions, st)
                          : lib.fwd_sampler(ptr(value), code(value), fptr(loc), fptr(attn), ptr(out), MSDA_DTYPE_F32, static_cast<int>(sampler),
                                            d.batch, d.heads, d.head_dim, d.queries, d.levels, d.points, d.shapes.data(), d.starts.data(),
                                            d.positions, st);
    });
    ctx->save_for_backward({value, loc, attn});
    ctx->saved_data["shapes"] = shapes_and_type(d, value);
    ctx->saved_data["sampler"] = sampler;
    return out;
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const int64_t sampler = ctx->saved_data["sampler"].toInt();
    Levels lv;
    Dims d;
    const Tensor value = restored(saved[0], shapes_of(ctx, lv)), loc = restored(saved[1], at::kFloat), attn = restored(saved[2], at::kFloat);
    const Tensor g = cotangent(grads[0], at::kFloat);
    saved_as(dims_of(value, loc, attn, std::move(lv), d) && g.device() == value.device() &&
             g.sizes().equals({d.batch, d.queries, int64_t{d.heads} * d.head_dim}));
    Tensor gv = like_if(ctx->needs_input_grad(0), value), gl = like_if(ctx->needs_input_grad(1), loc), ga = like_if(ctx->needs_input_grad(2), attn);
    Tensor ws;
    int64_t bytes = 0;
    if (gv.defined()) {
      bytes = lib.bwd_workspace_size(d.batch, d.heads, d.head_dim, d.queries, d.levels, d.points, d.shapes.data(), d.starts.data(), d.positions);
      check(bytes);
      ws = workspace(bytes, value);
    }
    launch(value, [&](void* st) {
      return sampler == 0 ? lib.bwd(ptr(value), code(value), fptr(loc), fptr(attn), ptr(g), MSDA_DTYPE_F32, ptr(gv), fptr(gl), fptr(ga), d.batch,
                                    d.heads, d.head_dim, d.queries, d.levels, d.points, d.shapes.data(), d.starts.data(), d.positions, ptr(ws),
                                    bytes, st)
                          : lib.bwd_sampler(ptr(value), code(value), fptr(loc), fptr(attn), ptr(g), MSDA_DTYPE_F32, ptr(gv), fptr(gl), fptr(ga),
                                            static_cast<int>(sampler), d.batch, d.heads, d.head_dim, d.queries, d.levels, d.points,
                                            d.shapes.data(), d.starts.data(), d.positions, ptr(ws), bytes, st);
    });
    return {gv, gl, ga, Tensor(), Tensor()};
  }

  // the level shapes and the value type of a call, kept for its backward
  static std::vector<int64_t> shapes_and_type(const Dims& d, const Tensor& value) {
    std::vector<int64_t> kept(d.shapes.begin(), d.shapes.end());
    kept.push_back(static_cast<int64_t>(value.scalar_type()));
    return kept;
  }

  static at::ScalarType shapes_of(AutogradContext* ctx, Levels& lv) {
    const auto kept = ctx->saved_data["shapes"].toIntVector();
    for (size_t i = 0; i + 1 < kept.size(); i += 2) {
      lv.shapes.push_back(static_cast<int32_t>(kept[i]));
      lv.shapes.push_back(static_cast<int32_t>(kept[i + 1]));
      lv.starts.push_back(static_cast<int32_t>(lv.positions));
      lv.positions += kept[i] * kept[i + 1];
    }
    return static_cast<at::ScalarType>(kept.back());
  }
};

py::object core(const py::handle& value, const py::handle& shapes, const py::handle& loc, const py::handle& attn, int64_t sampler) {
  const Tensor *v, *l, *a;
  Levels lv;
  Dims d;
  if (!ordinary_state() || (v = plain(value)) == nullptr || (l = plain(loc)) == nullptr || (a = plain(attn)) == nullptr ||
      !levels_of(shapes, lv) || !dims_of(*v, *l, *a, std::move(lv), d))
    return py::none();
  return py::cast(Core::apply(*v, *l, *a, d, sampler));
}

// ---- the core with the MSDeformAttn prologue --------------------------------------------------

struct Fused : torch::autograd::Function<Fused> {
  static Tensor forward(AutogradContext* ctx, const Tensor& value, const Tensor& ref, const Tensor& off, const Tensor& logits, const Dims& d) {
    Tensor out = at::empty({d.batch, d.queries, int64_t{d.heads} * d.head_dim}, off.options());
    launch(value, [&](void* st) {
      return lib.fused_fwd(ptr(value), code(value), fptr(ref), static_cast<int>(ref.size(3)), fptr(off), fptr(logits), ptr(out), MSDA_DTYPE_F32,
                           d.batch, d.heads, d.head_dim, d.queries, d.levels, d.points, d.shapes.data(), d.starts.data(), d.positions, st);
    });
    ctx->save_for_backward({value, ref, off, logits});
    ctx->saved_data["shapes"] = Core::shapes_and_type(d, value);
    return out;
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    Levels lv;
    Dims d;
    const Tensor value = restored(saved[0], Core::shapes_of(ctx, lv)), ref = restored(saved[1], at::kFloat);
    const Tensor off = restored(saved[2], at::kFloat), logits = restored(saved[3], at::kFloat);
    const Tensor g = cotangent(grads[0], at::kFloat);
    saved_as(dims_of(value, off, logits, std::move(lv), d) && ref_matches(ref, value, d) && g.device() == value.device() &&
             g.sizes().equals({d.batch, d.queries, int64_t{d.heads} * d.head_dim}));
    const int ref_dim = static_cast<int>(ref.size(3));
    Tensor gv = like_if(ctx->needs_input_grad(0), value), gr = like_if(ctx->needs_input_grad(1), ref);
    Tensor go = like_if(ctx->needs_input_grad(2), off), gl = like_if(ctx->needs_input_grad(3), logits);
    const int64_t bytes = lib.fused_bwd_workspace_size(d.batch, d.heads, d.head_dim, d.queries, d.levels, d.points, ref_dim, d.shapes.data(),
                                                       d.starts.data(), d.positions);
    check(bytes);
    const Tensor ws = workspace(bytes, value);
    launch(value, [&](void* st) {
      return lib.fused_bwd(ptr(value), code(value), fptr(ref), ref_dim, fptr(off), fptr(logits), ptr(g), MSDA_DTYPE_F32, ptr(gv), fptr(go),
                           fptr(gl), fptr(gr), d.batch, d.heads, d.head_dim, d.queries, d.levels, d.points, d.shapes.data(), d.starts.data(),
                           d.positions, ptr(ws), bytes, st);
    });
    return {gv, gr, go, gl, Tensor()};
  }

  // reference points [B, Q, L, 2 | 4], contiguous
  static bool ref_matches(const Tensor& ref, const Tensor& value, const Dims& d) {
    return ref.dim() == 4 && f32(ref) && ref.is_contiguous() && ref.device() == value.device() && ref.size(0) == d.batch &&
           ref.size(1) == d.queries && ref.size(2) == d.levels && (ref.size(3) == 2 || ref.size(3) == 4);
  }
};

py::object fused(const py::handle& value, const py::handle& shapes, const py::handle& ref, const py::handle& off, const py::handle& logits) {
  const Tensor *v, *r, *o, *l;
  Levels lv;
  Dims d;
  if (!ordinary_state() || (v = plain(value)) == nullptr || (r = plain(ref)) == nullptr || (o = plain(off)) == nullptr ||
      (l = plain(logits)) == nullptr || !levels_of(shapes, lv) || !dims_of(*v, *o, *l, std::move(lv), d))
    return py::none();
  if (!Fused::ref_matches(*r, *v, d)) return py::none();
  return py::cast(Fused::apply(*v, *r, *o, *l, d));
}

// ---- value projection -------------------------------------------------------------------------

struct ValueProj : torch::autograd::Function<ValueProj> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& w, const std::optional<Tensor>& bias,
                        const std::optional<Tensor>& mask, int64_t heads) {
    const int64_t b = x.size(0), s = x.size(1), d = w.size(0) / heads;
    Tensor out = at::empty({b * heads, s, d}, x.options());
    launch(x, [&](void* st) {
      return lib.value_proj_fwd(ptr(x), code(x), fptr(w), bias ? fptr(*bias) : nullptr, mask ? static_cast<const uint8_t*>(ptr(*mask)) : nullptr,
                                ptr(out), static_cast<int>(b), static_cast<int>(s), static_cast<int>(x.size(2)), static_cast<int>(heads),
                                static_cast<int>(d), st);
    });
    ctx->save_for_backward({x, w, mask ? *mask : Tensor()});
    ctx->saved_data["heads"] = heads;
    ctx->saved_data["bias"] = bias.has_value();
    return out;
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor x = restored(saved[0], grads[0].scalar_type()), w = restored(saved[1], at::kFloat);
    const Tensor mask = saved[2].defined() ? restored(saved[2], at::kBool) : Tensor();
    const int64_t heads = ctx->saved_data["heads"].toInt();
    saved_as(x.dim() == 3 && w.dim() == 2 && w.size(1) == x.size(2) && w.size(0) % heads == 0 && w.device() == x.device() &&
             grads[0].device() == x.device() && grads[0].sizes().equals({x.size(0) * heads, x.size(1), w.size(0) / heads}) &&
             (!mask.defined() || (mask.device() == x.device() && mask.sizes().equals({x.size(0), x.size(1)}))));
    const int b = static_cast<int>(x.size(0)), s = static_cast<int>(x.size(1)), k = static_cast<int>(x.size(2)), h = static_cast<int>(heads);
    const int d = static_cast<int>(w.size(0) / heads);
    const Tensor g = cotangent(grads[0], x.scalar_type());
    const bool want_b = ctx->saved_data["bias"].toBool() && ctx->needs_input_grad(2);
    Tensor gx = like_if(ctx->needs_input_grad(0), x), gw = like_if(ctx->needs_input_grad(1), w);
    Tensor gb = want_b ? at::empty({w.size(0)}, w.options()) : Tensor(), ws;
    int64_t bytes = 0;
    if (gw.defined() || gb.defined()) {
      bytes = lib.value_proj_bwd_workspace_size(b, s, k, h, d);
      check(bytes);
      ws = workspace(bytes, x);
    }
    launch(x, [&](void* st) {
      return lib.value_proj_bwd(ptr(x), code(x), fptr(w), static_cast<const uint8_t*>(ptr(mask)), ptr(g), ptr(gx), fptr(gw), fptr(gb), b, s, k, h,
                                d, ptr(ws), bytes, st);
    });
    return {gx, gw, gb, Tensor(), Tensor()};
  }
};

py::object value_proj(const py::handle& x, const py::handle& weight, const py::handle& bias, int64_t heads, const py::handle& mask) {
  const Tensor *a, *w, *bt = nullptr, *mt = nullptr;
  if (!ordinary_state() || (a = plain(x)) == nullptr || (w = plain(weight)) == nullptr || (!bias.is_none() && (bt = plain(bias)) == nullptr) ||
      (!mask.is_none() && (mt = plain(mask)) == nullptr))
    return py::none();
  if (a->dim() != 3 || !value_type(*a) || !a->is_contiguous() || w->dim() != 2 || !f32(*w) || !w->is_contiguous() || w->device() != a->device() ||
      w->size(1) != a->size(2) || heads < 1 || w->size(0) % heads != 0)
    return py::none();
  for (int64_t n : {a->size(0), a->size(1), a->size(2), w->size(0)})
    if (n >= (int64_t{1} << 31)) return py::none();
  if (bt != nullptr && (bt->dim() != 1 || bt->size(0) != w->size(0) || !f32(*bt) || !bt->is_contiguous() || bt->device() != a->device()))
    return py::none();
  if (mt != nullptr && (mt->dim() != 2 || mt->size(0) != a->size(0) || mt->size(1) != a->size(1) || mt->scalar_type() != at::kBool ||
                        !mt->is_contiguous() || mt->device() != a->device()))
    return py::none();
  return py::cast(ValueProj::apply(*a, *w, bt != nullptr ? std::optional<Tensor>(*bt) : std::nullopt,
                                   mt != nullptr ? std::optional<Tensor>(*mt) : std::nullopt, heads));
}

// ---- grid sampling ----------------------------------------------------------------------------

struct GridSample : torch::autograd::Function<GridSample> {
  static Tensor forward(AutogradContext* ctx, const Tensor& in, const Tensor& grid, int64_t kind, int64_t padding, int64_t mode) {
    Tensor out = at::empty({in.size(0), in.size(1), grid.size(1)}, in.options());
    launch(in, [&](void* st) {
      return lib.grid_sample_fwd(ptr(in), code(in), fptr(grid), static_cast<int>(kind), ptr(out), static_cast<int>(in.size(0)),
                                 static_cast<int>(in.size(1)), static_cast<int>(in.size(2)), static_cast<int>(in.size(3)),
                                 static_cast<int>(grid.size(1)), static_cast<int>(padding), static_cast<int>(mode), st);
    });
    ctx->save_for_backward({in, grid});
    ctx->saved_data["modes"] = std::vector<int64_t>{kind, padding, mode};
    return out;
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor in = restored(saved[0], grads[0].scalar_type()), grid = restored(saved[1], at::kFloat);
    saved_as(in.dim() == 4 && grid.dim() == 3 && grid.size(0) == in.size(0) && grid.size(2) == 2 && grid.device() == in.device() &&
             grads[0].device() == in.device() && grads[0].sizes().equals({in.size(0), in.size(1), grid.size(1)}));
    const auto modes = ctx->saved_data["modes"].toIntVector();
    const Tensor g = cotangent(grads[0], in.scalar_type());
    Tensor gi = like_if(ctx->needs_input_grad(0), in), gg = like_if(ctx->needs_input_grad(1), grid);
    launch(in, [&](void* st) {
      return lib.grid_sample_bwd(ptr(in), code(in), fptr(grid), static_cast<int>(modes[0]), ptr(g), ptr(gi), fptr(gg), static_cast<int>(in.size(0)),
                                 static_cast<int>(in.size(1)), static_cast<int>(in.size(2)), static_cast<int>(in.size(3)),
                                 static_cast<int>(grid.size(1)), static_cast<int>(modes[1]), static_cast<int>(modes[2]), st);
    });
    return {gi, gg, Tensor(), Tensor(), Tensor()};
  }
};

// coords [N, P, 2] or [N, Hg, Wg, 2] -> [N, C, P] or [N, C, Hg, Wg]
py::object grid_sample(const py::handle& inputs, const py::handle& coords, int64_t kind, int64_t padding, int64_t mode) {
  const Tensor *in, *c;
  if (!ordinary_state() || (in = plain(inputs)) == nullptr || (c = plain(coords)) == nullptr) return py::none();
  if (in->dim() != 4 || !value_type(*in) || !in->is_contiguous() || (c->dim() != 3 && c->dim() != 4) || c->size(-1) != 2 ||
      c->size(0) != in->size(0) || !f32(*c) || !c->is_contiguous() || c->device() != in->device())
    return py::none();
  for (int64_t n : {in->size(0), in->size(1), in->size(2), in->size(3), c->numel()})
    if (n >= (int64_t{1} << 31)) return py::none();
  if (c->dim() == 3) return py::cast(GridSample::apply(*in, *c, kind, padding, mode));
  const Tensor out = GridSample::apply(*in, c->reshape({c->size(0), -1, 2}), kind, padding, mode);
  return py::cast(out.reshape({in->size(0), in->size(1), c->size(1), c->size(2)}));
}

// ---- self-attention, without mask and dropout -------------------------------------------------

struct Layout {
  int batch, groups, heads, len, dim;
  bool rows;  // [B, G * P, H * D] rows, else [Z, H, L, D]
  void strides(const Tensor& t, int64_t* out) const {  // (batch, group, head, row)
    out[0] = t.stride(0);
    out[1] = rows ? len * t.stride(1) : 0;
    out[2] = rows ? dim : t.stride(1);
    out[3] = rows ? t.stride(1) : t.stride(2);
  }
};

struct Attention : torch::autograd::Function<Attention> {
  static Tensor forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v, const Layout& lay) {
    Tensor out = at::empty(q.sizes(), q.options());
    Tensor stats = at::empty({int64_t{lay.batch} * lay.groups * lay.heads * lay.len * 4}, q.options().dtype(at::kFloat));
    int64_t st[16];
    const Tensor* t[4] = {&q, &k, &v, &out};
    for (int i = 0; i < 4; ++i) lay.strides(*t[i], st + 4 * i);
    launch(q, [&](void* stream) {
      return lib.attention_fwd(ptr(q), ptr(k), ptr(v), code(q), ptr(out), fptr(stats), lay.batch, lay.groups, lay.heads, lay.len, lay.dim, st,
                               nullptr, stream);
    });
    ctx->save_for_backward({q, k, v, out, stats});
    ctx->saved_data["layout"] = std::vector<int64_t>{lay.batch, lay.groups, lay.heads, lay.len, lay.dim, lay.rows ? 1 : 0};
    return out;
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const auto channels = [&](const Tensor& t) {  // any row strides
      return t.defined() && t.is_cuda() && t.scalar_type() == grads[0].scalar_type() && t.dim() != 0 && t.stride(-1) == 1
                 ? t
                 : restored(t, grads[0].scalar_type());
    };
    const Tensor q = channels(saved[0]), k = channels(saved[1]), v = channels(saved[2]), out = channels(saved[3]);
    const Tensor stats = restored(saved[4], at::kFloat);
    const auto n = ctx->saved_data["layout"].toIntVector();
    const Layout lay{static_cast<int>(n[0]), static_cast<int>(n[1]), static_cast<int>(n[2]), static_cast<int>(n[3]), static_cast<int>(n[4]), n[5] != 0};
    for (const Tensor* t : {&q, &k, &v, &out}) saved_as(t->sizes() == grads[0].sizes() && t->device() == q.device());
    saved_as(grads[0].device() == q.device() && stats.device() == q.device() &&
             stats.numel() == int64_t{lay.batch} * lay.groups * lay.heads * lay.len * 4);
    Tensor g = grads[0];
    if (g.stride(-1) != 1) g = g.contiguous();
    Tensor gq = like_if(ctx->needs_input_grad(0), q), gk = like_if(ctx->needs_input_grad(1), k), gv = like_if(ctx->needs_input_grad(2), v);
    int64_t st[32] = {};
    const Tensor* t[8] = {&q, &k, &v, &out, &g, &gq, &gk, &gv};
    for (int i = 0; i < 8; ++i)
      if (t[i]->defined()) lay.strides(*t[i], st + 4 * i);
    launch(q, [&](void* stream) {
      return lib.attention_bwd(ptr(q), ptr(k), ptr(v), ptr(out), fptr(stats), ptr(g), code(q), ptr(gq), ptr(gk), ptr(gv), lay.batch, lay.groups,
                               lay.heads, lay.len, lay.dim, st, nullptr, stream);
    });
    return {gq, gk, gv, Tensor()};
  }
};

// q, k, v of one shape: [B, Q, C] rows in `groups` groups and `heads` heads, or [B, H, L, D] (heads 0)
py::object attention(const py::handle& q, const py::handle& k, const py::handle& v, int64_t heads, int64_t groups) {
  const Tensor *a, *b, *c;
  if (!ordinary_state() || (a = plain(q)) == nullptr || (b = plain(k)) == nullptr || (c = plain(v)) == nullptr) return py::none();
  const bool rows = heads != 0;
  if (a->dim() != (rows ? 3 : 4) || !value_type(*a)) return py::none();
  for (const Tensor* t : {a, b, c})
    if (t->sizes() != a->sizes() || t->scalar_type() != a->scalar_type() || t->device() != a->device() || t->stride(-1) != 1) return py::none();
  for (int64_t n : a->sizes())
    if (n >= (int64_t{1} << 31)) return py::none();
  if (rows && (heads < 1 || groups < 1 || a->size(2) % heads != 0 || a->size(1) % groups != 0)) return py::none();
  auto n = [](int64_t x) { return static_cast<int>(x); };
  const Layout lay = rows ? Layout{n(a->size(0)), n(groups), n(heads), n(a->size(1) / groups), n(a->size(2) / heads), true}
                          : Layout{n(a->size(0)), 1, n(a->size(1)), n(a->size(2)), n(a->size(3)), false};
  return py::cast(Attention::apply(*a, *b, *c, lay));
}

}  // namespace

PYBIND11_MODULE(_torch_binding, m) {
  m.doc() = "The differentiable ops over the C ABI, for ordinary calls (None: not one).";
  py::register_exception_translator([](std::exception_ptr p) {
    try {
      if (p) std::rethrow_exception(p);
    } catch (python_error& e) {  // its Python exception, as it was raised
      e.restore();
    }
  });
  m.def("bind", &bind);
  m.def("workspace", &workspace);
  m.def("core", &core);
  m.def("fused", &fused);
  m.def("value_proj", &value_proj);
  m.def("grid_sample", &grid_sample);
  m.def("attention", &attention);
}
