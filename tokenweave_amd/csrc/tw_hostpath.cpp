// tokenweave_amd._hostpath — the ops as plain Python calls, without torch's dispatcher.
//
// A decode-size kernel takes 3 - 5 us; torch.ops needs 1 - 1.5 us to match a schema and box its
// arguments, a ctypes call with its checks in Python 5 us, a call site like
// fused_allreduce_layernorm (assertions, two slices, a module call) another 5.  The functions
// here take the Python objects as they are, check them in C++ and enqueue the kernel: 0.3 us on
// top of the launch itself (2.3 us).
//
// A call is made directly only where the dispatcher would do nothing but call the same
// function: plain torch.Tensors or Parameters, no autograd through the data, no dispatch or
// function mode, no tracing, no profiler.  Otherwise, and whenever an argument fails a check,
// the function says so (False / NotImplemented) before it has enqueued anything, and the
// Python caller takes its ordinary route, which raises the error or does the bookkeeping.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/grad_mode.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/record_function.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <vector>

#include "tw_torch_ops.h"

namespace {

using at::Tensor;

// Interned attribute names and torch.nn's global hook tables, looked up once.
PyObject *s_parameters, *s_weight, *s_bias, *s_epsilon, *s_var_override, *s_forward, *s_compiled, *s_multicast,
    *s_signal_pads, *s_call, *s_hooks[4], *s_tp_rank, *s_skip_bias, *s_input_parallel, *s_residual, *s_out;
PyObject* g_global_hooks[4];

bool direct_allowed() {
  const auto included = c10::impl::tls_local_dispatch_key_set().included_;
  return (included - c10::default_included_set).empty() && !at::impl::torch_function_mode_enabled() &&
         !at::hasCallbacks() && !torch::jit::tracer::isTracing();
}

// The keys of a strided tensor whose storage on the GPU holds its values.  With any other key (a lazy
// sign or conjugation, a tensor of zeros without storage, a nested, sparse or wrapped one) the
// dispatcher has work to do before the op may read it.
const c10::DispatchKeySet g_own_data({c10::DispatchKey::Dense, c10::DispatchKey::AutogradFunctionality,
                                      c10::DispatchKey::ADInplaceOrView, c10::DispatchKey::AutocastCUDA});

// The tensor behind a plain torch.Tensor on the GPU; `data`: one the op reads or writes as data (a weight
// is taken by its values alone, as `.data` is).
const Tensor* plain(PyObject* o, bool data = true) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || (t.key_set() - g_own_data).highestFunctionalityKey() != c10::DispatchKey::Undefined)
    return nullptr;
  if (data && t.requires_grad() && at::GradMode::is_enabled()) return nullptr;
  return &t;
}

bool as_int(PyObject* o, int64_t* v) {
  if (!PyLong_CheckExact(o)) return false;
  int overflow = 0;
  *v = PyLong_AsLongLongAndOverflow(o, &overflow);
  return overflow == 0;
}

bool as_cap(PyObject* o, int64_t* v) {  // None: no cap
  *v = 0;
  return o == Py_None || as_int(o, v);
}

bool int_attribute(PyObject* o, PyObject* name, int64_t* v) {
  PyObject* value = PyObject_GetAttr(o, name);
  if (!value) PyErr_Clear();  // the ordinary route raises it
  const bool got = value && as_int(value, v);
  Py_XDECREF(value);
  return got;
}

bool as_double(PyObject* o, double* v) {
  if (!PyFloat_CheckExact(o)) return false;
  *v = PyFloat_AS_DOUBLE(o);
  return true;
}

Tensor& mut(const Tensor* t) { return const_cast<Tensor&>(*t); }

// Runs `f` without the GIL; false when it refused its arguments.
template <typename F>
bool enqueue(F&& f) {
  bool ok = true;
  Py_BEGIN_ALLOW_THREADS;
  try {
    f();
  } catch (...) {
    ok = false;  // the ordinary route words the error
  }
  Py_END_ALLOW_THREADS;
  return ok;
}

// A new contiguous tensor on the device of `x` (0.5 us less than through the dispatcher).
Tensor empty_on(const Tensor& x, at::IntArrayRef sizes, at::ScalarType dtype) {
  return Tensor(at::detail::empty_cuda(sizes, dtype, x.device(), std::nullopt));
}

PyObject* yes_no(bool ok) { return PyBool_FromLong(ok); }

PyObject* not_handled() {
  Py_INCREF(Py_NotImplemented);
  return Py_NotImplemented;
}

PyObject* pair(PyObject* a, PyObject* b) {  // new references to both
  PyObject* t = PyTuple_New(2);
  if (!t) return nullptr;
  Py_INCREF(a);
  Py_INCREF(b);
  PyTuple_SET_ITEM(t, 0, a);
  PyTuple_SET_ITEM(t, 1, b);
  return t;
}

// ---------------------------------------------------------------------------
// ops
// ---------------------------------------------------------------------------
template <void (*OP)(Tensor&, Tensor&, Tensor&, double)>
PyObject* norm3(PyObject*, PyObject* const* a, Py_ssize_t n) {
  double eps;
  if (n != 4 || !direct_allowed()) Py_RETURN_FALSE;
  const Tensor *x = plain(a[0]), *y = plain(a[1]), *w = plain(a[2]);
  if (!x || !y || !w || !as_double(a[3], &eps)) Py_RETURN_FALSE;
  return yes_no(enqueue([&] { OP(mut(x), mut(y), mut(w), eps); }));
}

PyObject* fused_add_rms_norm_cta(PyObject*, PyObject* const* a, Py_ssize_t n) {
  double eps;
  int64_t cap;
  if (n != 5 || !direct_allowed()) Py_RETURN_FALSE;
  const Tensor *x = plain(a[0]), *r = plain(a[1]), *w = plain(a[2]);
  if (!x || !r || !w || !as_cap(a[3], &cap) || !as_double(a[4], &eps)) Py_RETURN_FALSE;
  return yes_no(enqueue([&] { tw_torch::fused_add_rms_norm_cta(mut(x), mut(r), mut(w), cap, eps); }));
}

// (input, residual, weight, mcptr, signal_pads, rank, world_size, MAX_CTAS, epsilon); the signal pads are
// for peers, of which there are none: an integer, as the registered op wants it
template <bool ALL_GATHER>
PyObject* fused_rs_ln(PyObject*, PyObject* const* a, Py_ssize_t n) {
  double eps;
  int64_t mcptr, pads, rank, ws, cap;
  if (n != 9 || !direct_allowed()) Py_RETURN_FALSE;
  const Tensor *x = plain(a[0]), *r = plain(a[1]), *w = plain(a[2]);
  if (!x || !r || !w || !as_int(a[3], &mcptr) || !as_int(a[4], &pads) || !as_int(a[5], &rank) || !as_int(a[6], &ws) ||
      !as_cap(a[7], &cap) || !as_double(a[8], &eps) || x->dim() < 1 || x->size(-1) == 0)
    Py_RETURN_FALSE;
  const int64_t rows = x->numel() / x->size(-1);
  return yes_no(enqueue([&] { tw_torch::fused_rs_ln_rows(ALL_GATHER, *x, *r, *w, 0, rows, mcptr, rank, ws, cap, eps); }));
}

PyObject* rms_norm_static_fp8_quant(PyObject*, PyObject* const* a, Py_ssize_t n) {
  double eps;
  if (n != 5 || !direct_allowed()) Py_RETURN_FALSE;
  const Tensor *o = plain(a[0]), *x = plain(a[1]), *w = plain(a[2]), *s = plain(a[3]);
  if (!o || !x || !w || !s || !as_double(a[4], &eps)) Py_RETURN_FALSE;
  return yes_no(enqueue([&] { tw_torch::rms_norm_static_fp8_quant(mut(o), mut(x), mut(w), mut(s), eps); }));
}

PyObject* fused_add_rms_norm_static_fp8_quant(PyObject*, PyObject* const* a, Py_ssize_t n) {
  double eps;
  if (n != 6 || !direct_allowed()) Py_RETURN_FALSE;
  const Tensor *o = plain(a[0]), *x = plain(a[1]), *r = plain(a[2]), *w = plain(a[3]), *s = plain(a[4]);
  if (!o || !x || !r || !w || !s || !as_double(a[5], &eps)) Py_RETURN_FALSE;
  return yes_no(
      enqueue([&] { tw_torch::fused_add_rms_norm_static_fp8_quant(mut(o), mut(x), mut(r), mut(w), mut(s), eps); }));
}

// (result, input, weight, scales, epsilon, scale_ub | None, residual | None)
PyObject* rms_norm_dynamic_per_token_quant_out(PyObject*, PyObject* const* a, Py_ssize_t n) {
  double eps;
  if (n != 7 || !direct_allowed()) Py_RETURN_FALSE;
  const Tensor *o = plain(a[0]), *x = plain(a[1]), *w = plain(a[2]), *s = plain(a[3]);
  const Tensor* ub = a[5] == Py_None ? nullptr : plain(a[5]);
  const Tensor* r = a[6] == Py_None ? nullptr : plain(a[6]);
  if (!o || !x || !w || !s || !as_double(a[4], &eps) || (!ub && a[5] != Py_None) || (!r && a[6] != Py_None))
    Py_RETURN_FALSE;
  return yes_no(enqueue([&] {
    tw_torch::rms_norm_dynamic_per_token_quant(mut(o), *x, *w, mut(s), eps, ub ? std::optional<Tensor>(*ub) : std::nullopt,
                                               r ? std::optional<Tensor>(*r) : std::nullopt);
  }));
}

// (input, weight, epsilon, quant_dtype, scale_ub | None, residual | None) -> (output, scales)
PyObject* rms_norm_dynamic_per_token_quant(PyObject*, PyObject* const* a, Py_ssize_t n) {
  double eps;
  if (n != 6 || !direct_allowed()) return not_handled();
  const Tensor *x = plain(a[0]), *w = plain(a[1]);
  const Tensor* ub = a[4] == Py_None ? nullptr : plain(a[4]);
  const Tensor* r = a[5] == Py_None ? nullptr : plain(a[5]);
  if (!x || !w || !as_double(a[2], &eps) || !THPDtype_Check(a[3]) || (!ub && a[4] != Py_None) ||
      (!r && a[5] != Py_None) || !x->is_cuda() || x->dim() < 1 || x->size(-1) == 0 || !x->is_contiguous())
    return not_handled();
  const at::ScalarType kind = reinterpret_cast<THPDtype*>(a[3])->scalar_type;
  Tensor out, scales;
  if (!enqueue([&] {
        out = empty_on(*x, x->sizes(), kind);
        scales = empty_on(*x, {x->numel() / x->size(-1), 1}, at::kFloat);
        tw_torch::rms_norm_dynamic_per_token_quant(out, *x, *w, scales, eps,
                                                   ub ? std::optional<Tensor>(*ub) : std::nullopt,
                                                   r ? std::optional<Tensor>(*r) : std::nullopt);
      }))
    return not_handled();
  PyObject* po = THPVariable_Wrap(out);
  PyObject* ps = po ? THPVariable_Wrap(scales) : nullptr;
  PyObject* t = ps ? pair(po, ps) : nullptr;
  Py_XDECREF(po);
  Py_XDECREF(ps);
  return t;
}

// (out, a, b, max_cus | None, bias | None)
PyObject* gemm_bf16_nt(PyObject*, PyObject* const* a, Py_ssize_t n) {
  int64_t cus;
  if (n != 5 || !direct_allowed()) Py_RETURN_FALSE;
  const Tensor *o = plain(a[0]), *x = plain(a[1]), *w = plain(a[2], false);
  const Tensor* bias = a[4] == Py_None ? nullptr : plain(a[4], false);
  if (!o || !x || !w || !as_cap(a[3], &cus) || (!bias && a[4] != Py_None)) Py_RETURN_FALSE;
  return yes_no(enqueue([&] { tw_torch::gemm_bf16_nt(*o, *x, *w, cus, bias); }));
}

// The tensors of a list or tuple; `nulls`: None stands for "no tensor".
bool tensor_list(PyObject* seq, bool nulls, std::vector<const Tensor*>* out) {
  if (!PyList_CheckExact(seq) && !PyTuple_CheckExact(seq)) return false;
  const Py_ssize_t n = PySequence_Fast_GET_SIZE(seq);
  out->reserve(n);
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject* o = PySequence_Fast_GET_ITEM(seq, i);
    const Tensor* t = nulls && o == Py_None ? nullptr : plain(o, false);
    if (!t && !(nulls && o == Py_None)) return false;
    out->push_back(t);
  }
  return true;
}

// (outs, a, b, max_cus | None, biases | None).  Runs with the GIL: nobody may change the lists
// while their tensors are in use.
PyObject* gemm_bf16_nt_partials(PyObject*, PyObject* const* a, Py_ssize_t n) {
  int64_t cus;
  std::vector<const Tensor*> o, x, w, bias;
  if (n != 5 || !direct_allowed() || !as_cap(a[3], &cus) || !tensor_list(a[0], false, &o) ||
      !tensor_list(a[1], false, &x) || !tensor_list(a[2], false, &w) ||
      (a[4] != Py_None && !tensor_list(a[4], true, &bias)))
    Py_RETURN_FALSE;
  bool ok = true;
  try {
    tw_torch::gemm_bf16_nt_partials(o, x, w, cus, bias);
  } catch (...) {
    ok = false;
  }
  return yes_no(ok);
}

// ---------------------------------------------------------------------------
// layers.  An nn.Module whose __call__ would do more than call the class's forward (hooks, a
// compiled or replaced forward) is not handled here.
// ---------------------------------------------------------------------------
PyObject* instance_dict(PyObject* module) {
  PyObject** d = _PyObject_GetDictPtr(module);
  return d && *d && PyDict_CheckExact(*d) ? *d : nullptr;
}

bool plain_module(PyObject* dict) {
  for (int i = 0; i < 4; ++i) {
    PyObject* h = PyDict_GetItem(dict, s_hooks[i]);
    if (!h || !PyDict_Check(h) || PyDict_GET_SIZE(h) || PyDict_GET_SIZE(g_global_hooks[i])) return false;
  }
  PyObject* compiled = PyDict_GetItem(dict, s_compiled);
  return (!compiled || compiled == Py_None) && !PyDict_GetItem(dict, s_forward);
}

// The norm's class and torch.nn.Module with the functions that a call of a norm runs, as the package
// defined them.
PyTypeObject *g_norm, *g_module_class;
PyObject *g_norm_forward, *g_norm_call, *g_module_call;

// (RMSNorm, torch.nn.Module), once when the class is defined.
PyObject* remember_rms_norm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 2 || !PyType_Check(a[0]) || !PyType_Check(a[1])) Py_RETURN_FALSE;
  for (Py_ssize_t i = 0; i < n; ++i) Py_INCREF(a[i]);
  g_norm = (PyTypeObject*)a[0];
  g_module_class = (PyTypeObject*)a[1];
  Py_XINCREF(g_norm_forward = _PyType_Lookup(g_norm, s_forward));
  Py_XINCREF(g_norm_call = _PyType_Lookup(g_norm, s_call));
  Py_XINCREF(g_module_call = _PyType_Lookup(g_module_class, s_call));
  return yes_no(g_norm_forward && g_norm_call && g_module_call);
}

// Whether calling this object runs the package's RMSNorm: neither a subclass nor a class whose forward
// or __call__ somebody has replaced (`plain_module` looks at the instance).  Looked up by type in 35 ns
// where the reads in Python took 170.
PyObject* runs_rms_norm(PyObject*, PyObject* o) {
  return yes_no(g_norm && Py_TYPE(o) == g_norm && _PyType_Lookup(g_norm, s_forward) == g_norm_forward &&
                _PyType_Lookup(g_norm, s_call) == g_norm_call && _PyType_Lookup(g_module_class, s_call) == g_module_call);
}

// A parameter, or what the class keeps as a plain tensor attribute in its place.
const Tensor* module_tensor(PyObject* dict, PyObject* name) {
  PyObject* params = PyDict_GetItem(dict, s_parameters);
  PyObject* p = params && PyDict_Check(params) ? PyDict_GetItem(params, name) : nullptr;
  if (!p) p = PyDict_GetItem(dict, name);
  return p && p != Py_None ? plain(p, false) : nullptr;
}

// (Callers copy what module_tensor returns before they release the GIL: the module may be given
// another weight meanwhile.)

// The weight and epsilon of an RMSNorm that normalises over its whole hidden size.
const Tensor* norm_layer(PyObject* dict, double* eps) {
  PyObject* e = PyDict_GetItem(dict, s_epsilon);
  if (!e || !as_double(e, eps) || PyDict_GetItem(dict, s_var_override) != Py_None) return nullptr;
  return module_tensor(dict, s_weight);
}

// (layer, x, residual | None, out | None, MAX_CTAS | None) -> what RMSNorm.forward returns
PyObject* rms_norm_forward(PyObject*, PyObject* const* a, Py_ssize_t n) {
  double eps;
  int64_t cap;
  if (n != 5 || !direct_allowed()) return not_handled();
  PyObject* dict = instance_dict(a[0]);
  const Tensor* wp = dict ? norm_layer(dict, &eps) : nullptr;
  const Tensor* x = plain(a[1]);
  if (!wp || !x || !as_cap(a[4], &cap)) return not_handled();
  Tensor w = *wp;
  if (a[2] != Py_None) {
    const Tensor* r = plain(a[2]);
    if (!r) return not_handled();
    const bool capped = a[4] != Py_None;
    if (!enqueue([&] {
          if (capped) tw_torch::fused_add_rms_norm_cta(mut(x), mut(r), w, cap, eps);
          else tw_torch::fused_add_rms_norm(mut(x), mut(r), w, eps);
        }))
      return not_handled();
    return pair(a[1], a[2]);
  }
  if (a[3] != Py_None) {
    const Tensor* o = plain(a[3]);
    if (!o || !enqueue([&] { tw_torch::rms_norm_inplace(mut(o), mut(x), w, eps); })) return not_handled();
    Py_INCREF(a[1]);
    return a[1];
  }
  if (!x->is_cuda() || !x->is_contiguous()) return not_handled();
  Tensor out;
  if (!enqueue([&] {
        out = empty_on(*x, x->sizes(), x->scalar_type());
        tw_torch::rms_norm(out, mut(x), w, eps);
      }))
    return not_handled();
  return THPVariable_Wrap(out);
}

// (layer, args, kwargs): RMSNorm.__call__ with up to three positional arguments (x, residual,
// out), or x and one of the two others by name.
PyObject* rms_norm_call(PyObject* self, PyObject* const* a, Py_ssize_t n) {
  if (n != 3 || !PyTuple_CheckExact(a[1]) || !PyDict_CheckExact(a[2])) return not_handled();
  const Py_ssize_t given = PyTuple_GET_SIZE(a[1]);
  if (given < 1 || given > 3) return not_handled();
  PyObject* f[5] = {a[0], PyTuple_GET_ITEM(a[1], 0), Py_None, Py_None, Py_None};
  for (Py_ssize_t i = 1; i < given; ++i) f[i + 1] = PyTuple_GET_ITEM(a[1], i);
  if (PyDict_GET_SIZE(a[2])) {
    PyObject *r = PyDict_GetItem(a[2], s_residual), *o = PyDict_GetItem(a[2], s_out);
    if (given != 1 || PyDict_GET_SIZE(a[2]) != (r ? 1 : 0) + (o ? 1 : 0)) return not_handled();
    if (r) f[2] = r;
    if (o) f[3] = o;
  }
  PyObject* dict = instance_dict(a[0]);
  if (!dict || !plain_module(dict)) return not_handled();
  return rms_norm_forward(self, f, 5);
}

// (layer, hidden_states, residual, handle, per_rank, rank, world_size, MAX_CTAS, offset, row_range | None)
PyObject* fused_allreduce_layernorm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  double eps;
  int64_t per_rank, rank, ws, cap, offset, start, end;
  if (n != 10 || !direct_allowed()) Py_RETURN_FALSE;
  PyObject* dict = instance_dict(a[0]);
  if (!dict || !plain_module(dict)) Py_RETURN_FALSE;
  const Tensor* w = norm_layer(dict, &eps);
  const Tensor *x = plain(a[1]), *r = plain(a[2]);
  if (!w || !x || !r || !as_int(a[4], &per_rank) || !as_int(a[5], &rank) || !as_int(a[6], &ws) || !as_int(a[7], &cap) ||
      !as_int(a[8], &offset) || x->dim() != 2 || x->sizes() != r->sizes())
    Py_RETURN_FALSE;
  const int64_t T = x->size(0), H = x->size(1);
  if (a[9] == Py_None) {
    if (per_rank * ws != T) Py_RETURN_FALSE;
    start = rank * per_rank;
    end = start + per_rank;
  } else {
    if (!PyTuple_CheckExact(a[9]) || PyTuple_GET_SIZE(a[9]) != 2 || !as_int(PyTuple_GET_ITEM(a[9], 0), &start) ||
        !as_int(PyTuple_GET_ITEM(a[9], 1), &end))
      Py_RETURN_FALSE;
  }
  if (rank < 0 || rank >= ws || start < 0 || start >= end || end > T) Py_RETURN_FALSE;
  // copied before the handle is asked, which may run Python code
  const Tensor weight = *w;
  int64_t mcptr, pads;
  if (!int_attribute(a[3], s_multicast, &mcptr) || !int_attribute(a[3], s_signal_pads, &pads)) Py_RETURN_FALSE;
  const int64_t rows = end - start;
  return yes_no(enqueue([&] {
    tw_torch::fused_rs_ln_rows(true, *x, *r, weight, start, rows, mcptr + offset + start * H * 2, rank, ws,
                               std::min(cap, rows), eps);
  }));
}

// (layer, input, output, gemm_cus | None): RowParallelLinear.forward(is_tokenweave=True) up to
// its result.  (The caller has checked the type of the layer and of its linear method.)
PyObject* row_parallel_inplace(PyObject*, PyObject* const* a, Py_ssize_t n) {
  int64_t cus, tp_rank;
  if (n != 4 || !direct_allowed() || !as_cap(a[3], &cus)) Py_RETURN_FALSE;
  PyObject* dict = instance_dict(a[0]);
  if (!dict || PyDict_GetItem(dict, s_input_parallel) != Py_True) Py_RETURN_FALSE;
  PyObject *skip = PyDict_GetItem(dict, s_skip_bias), *rank = PyDict_GetItem(dict, s_tp_rank);
  PyObject* params = PyDict_GetItem(dict, s_parameters);
  if (!skip || !rank || !params || !PyDict_Check(params) || !as_int(rank, &tp_rank)) Py_RETURN_FALSE;
  const Tensor *w = module_tensor(dict, s_weight), *x = plain(a[1]), *o = plain(a[2]);
  if (!w || !x || !o) Py_RETURN_FALSE;
  const Tensor* bias = nullptr;
  if (tp_rank == 0 && skip == Py_False) {  // only rank 0 adds the bias
    PyObject* b = PyDict_GetItem(params, s_bias);
    if (!b || (b != Py_None && !(bias = plain(b, false)))) Py_RETURN_FALSE;
  } else if (skip != Py_True && skip != Py_False) {
    Py_RETURN_FALSE;
  }
  const Tensor weight = *w, bias_held = bias ? *bias : Tensor();
  return yes_no(enqueue([&] { tw_torch::gemm_bf16_nt(*o, *x, weight, cus, bias ? &bias_held : nullptr); }));
}

// What Python calls.  Some tensors throw when they are asked for a size (nested ones have none), and
// no C++ exception may leave through C frames: it would end the process.  Nothing is enqueued
// then, so the answer is that the call was not made: NotImplemented where a call has a RESULT,
// False where it only says whether it was made.
typedef PyObject* (*Fast)(PyObject*, PyObject* const*, Py_ssize_t);
template <Fast FN, bool RESULT>
PyObject* entry(PyObject* self, PyObject* const* a, Py_ssize_t n) noexcept {
  try {
    return FN(self, a, n);
  } catch (...) {
    return RESULT ? not_handled() : yes_no(false);
  }
}

#define TW_ENTRY(name, fn, result) {name, (PyCFunction)(void (*)(void))(entry<fn, result>), METH_FASTCALL, nullptr}
#define TW_FAST(name, fn) TW_ENTRY(name, (fn), false)
#define TW_FAST_RESULT(name, fn) TW_ENTRY(name, (fn), true)
PyMethodDef g_methods[] = {
    TW_FAST("rms_norm", norm3<tw_torch::rms_norm>),
    TW_FAST("fused_add_rms_norm", norm3<tw_torch::fused_add_rms_norm>),
    TW_FAST("rms_norm_inplace", norm3<tw_torch::rms_norm_inplace>),
    TW_FAST("fused_add_rms_norm_cta", fused_add_rms_norm_cta),
    TW_FAST("fused_rs_ln_ag_cta", fused_rs_ln<true>),
    TW_FAST("fused_rs_ln_cta", fused_rs_ln<false>),
    TW_FAST("rms_norm_static_fp8_quant", rms_norm_static_fp8_quant),
    TW_FAST("fused_add_rms_norm_static_fp8_quant", fused_add_rms_norm_static_fp8_quant),
    TW_FAST("rms_norm_dynamic_per_token_quant_out", rms_norm_dynamic_per_token_quant_out),
    TW_FAST_RESULT("rms_norm_dynamic_per_token_quant", rms_norm_dynamic_per_token_quant),
    TW_FAST("gemm_bf16_nt", gemm_bf16_nt),
    TW_FAST("gemm_bf16_nt_partials", gemm_bf16_nt_partials),
    TW_FAST_RESULT("rms_norm_forward", rms_norm_forward),
    TW_FAST_RESULT("rms_norm_call", rms_norm_call),
    TW_FAST("fused_allreduce_layernorm", fused_allreduce_layernorm),
    TW_FAST("row_parallel_inplace", row_parallel_inplace),
    TW_FAST("remember_rms_norm", remember_rms_norm),
    {"runs_rms_norm", runs_rms_norm, METH_O, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_hostpath", "direct calls of the ops (see tw_hostpath.cpp)", -1, g_methods};

bool init_names() {
  const struct { PyObject** at; const char* name; } names[] = {
      {&s_parameters, "_parameters"}, {&s_weight, "weight"}, {&s_bias, "bias"}, {&s_epsilon, "variance_epsilon"},
      {&s_var_override, "variance_size_override"}, {&s_forward, "forward"}, {&s_call, "__call__"}, {&s_compiled, "_compiled_call_impl"},
      {&s_multicast, "multicast_ptr"}, {&s_signal_pads, "signal_pad_ptrs_dev"}, {&s_hooks[0], "_forward_hooks"},
      {&s_hooks[1], "_forward_pre_hooks"}, {&s_hooks[2], "_backward_hooks"}, {&s_hooks[3], "_backward_pre_hooks"}, {&s_tp_rank, "tp_rank"},
      {&s_skip_bias, "skip_bias_add"}, {&s_input_parallel, "input_is_parallel"},
      {&s_residual, "residual"}, {&s_out, "out"}};
  for (const auto& n : names)
    if (!(*n.at = PyUnicode_InternFromString(n.name))) return false;
  PyObject* m = PyImport_ImportModule("torch.nn.modules.module");
  if (!m) return false;
  static const char* const tables[] = {"_global_forward_hooks", "_global_forward_pre_hooks", "_global_backward_hooks",
                                       "_global_backward_pre_hooks"};
  for (int i = 0; i < 4; ++i) {
    g_global_hooks[i] = PyObject_GetAttrString(m, tables[i]);
    if (!g_global_hooks[i] || !PyDict_Check(g_global_hooks[i])) return false;
  }
  Py_DECREF(m);
  return true;
}

}  // namespace

PyMODINIT_FUNC PyInit__hostpath(void) {
  if (!init_names()) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_ImportError, "torch.nn.Module keeps its hooks elsewhere");
    return nullptr;
  }
  return PyModule_Create(&g_module);
}
