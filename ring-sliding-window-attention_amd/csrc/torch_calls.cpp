// The plain attention call (one band over one sequence or pack, no ring) from Python to the launches
// without Python in between: checks, output allocation, parameter block, launch, and the autograd node.
//
// Small calls are bounded by the host.  With the same steps in Python (ring_swa/sliding_window.py,
// ops/band_attn.py) one forward took 20 us for a kernel of 12, and forward + backward of 1024 tokens, 4
// heads, 143 us for 45 us of kernels: building the parameter block through ctypes, the Python autograd
// function, and the hand-over of the interpreter lock to the autograd thread.  Here they take 10.5 and 72.
//
// band_attn() only takes what it can answer: plain tensors on one GPU, in the layout and types the
// kernels take, with no tracing, transform or mode active that has to see the call.  For everything
// else it returns None and the Python route runs, which refuses or handles it.
#include <Python.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/empty_like.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <cmath>
#include <cstdlib>
#include <optional>

#include "../../include/rswa.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// Entry points of the library that ring_swa._lib opened (bind)
struct {
  int (*fwd)(const rswa_attn_params*, void*) = nullptr;
  int (*bwd)(const rswa_attn_params*, void*) = nullptr;
  uint64_t (*bwd_bytes)(const rswa_attn_params*) = nullptr;
  PyObject* raise = nullptr;         // raises what a non-zero status means
  PyObject* python_bwd = nullptr;    // backward in Python, for the environment's switches and what has to be refused
} lib;

// With the interpreter lock only: Python changes the environment under it, and a getenv beside such a change
// may read the array that it has just freed.
bool env_switches() {
  TORCH_INTERNAL_ASSERT(PyGILState_Check());
  for (const char* name : {"RSWA_ADDRESSING", "RSWA_DKDV_FORM", "RSWA_DS_HANDOFF"}) {
    const char* v = std::getenv(name);
    if (v && *v) return true;
  }
  return false;
}

// Is anything active in this thread that has to see the operations of the call?
bool observed() {
  const auto tls = c10::impl::tls_local_dispatch_key_set();
  return tls.included_.has_any(c10::DispatchKeySet({c10::DispatchKey::Python, c10::DispatchKey::PythonTLSSnapshot,
                                                    c10::DispatchKey::FuncTorchDynamicLayerFrontMode,
                                                    c10::DispatchKey::FuncTorchDynamicLayerBackMode,
                                                    c10::DispatchKey::Functionalize})) ||
         c10::impl::TorchDispatchModeTLS::any_modes_set() || at::impl::torch_function_mode_enabled() ||
         torch::jit::tracer::isTracing();
}

// A dense tensor on the GPU and nothing else: no subclass, wrapper, lazy conjugate or tangent
bool plain(const Tensor& t) {
  static const c10::DispatchKeySet known =
      c10::DispatchKeySet({c10::DispatchKey::CUDA, c10::DispatchKey::AutogradCUDA, c10::DispatchKey::AutocastCUDA,
                           c10::DispatchKey::ADInplaceOrView});
  return t.defined() && t.is_cuda() && t.layout() == at::kStrided && (t.key_set().raw_repr() & ~known.raw_repr()) == 0 &&
         !t._fw_grad(0).defined();
}

// Queries, keys and values that the kernels take as they are?
bool fits(const Tensor& q, const Tensor& k, const Tensor& v, bool packed) {
  const int nd = packed ? 3 : 4;
  if (!plain(q) || !plain(k) || !plain(v)) return false;
  const auto type = q.scalar_type();
  if ((type != at::kBFloat16 && type != at::kHalf) || k.scalar_type() != type || v.scalar_type() != type) return false;
  if (q.dim() != nd || k.dim() != nd || v.dim() != nd || k.sizes() != v.sizes()) return false;
  if (q.device() != k.device() || q.device() != v.device()) return false;
  if (q.numel() == 0 || k.numel() == 0) return false;
  for (int d = 0; d < nd - 2; d++)
    if (q.size(d) != k.size(d) || q.size(d) >= (1 << 28)) return false;
  if (q.size(-1) != k.size(-1) || q.size(-2) % k.size(-2) != 0 || q.size(-2) >= (1 << 28)) return false;
  return q.stride(-1) == 1 && k.stride(-1) == 1 && v.stride(-1) == 1;
}

// ... and another tensor of q's type, shape and device
bool like(const Tensor& t, const Tensor& q) {
  return plain(t) && t.scalar_type() == q.scalar_type() && t.sizes() == q.sizes() && t.device() == q.device() &&
         t.stride(-1) == 1;
}

bool lse_of(const Tensor& t, const Tensor& q, bool packed) {
  if (!plain(t) || t.scalar_type() != at::kFloat || t.device() != q.device()) return false;
  return packed ? t.sizes().equals({q.size(1), q.size(0)}) : t.sizes().equals({q.size(0), q.size(2), q.size(1)});
}

struct Call {
  bool packed = false;
  int32_t window = 0, num_sink = 0;
  float scale = 0;
  Tensor cu;  // cu_seqlens of a pack; undefined: dense
};

void strides3(int64_t* dst, const Tensor& t, bool packed) {
  if (packed) {
    dst[0] = 0;
    dst[1] = t.stride(0);
    dst[2] = t.stride(1);
  } else {
    for (int i = 0; i < 3; i++) dst[i] = t.stride(i);
  }
}

// (as ring_swa/ops/band_attn.py:_params; causal, bottom-right aligned, one key range)
rswa_attn_params params(const Call& c, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& out,
                        const Tensor& lse) {
  rswa_attn_params p{};
  p.dtype = q.scalar_type() == at::kBFloat16 ? RSWA_BF16 : RSWA_F16;
  p.head_dim = (int32_t)q.size(-1);
  p.heads_q = (int32_t)q.size(-2);
  p.heads_kv = (int32_t)k.size(-2);
  if (c.packed) {
    p.batch = (int32_t)c.cu.numel() - 1;
    p.total_q = p.total_k = q.size(0);
    p.seqlen_q = p.seqlen_k = (int32_t)q.size(0);
    p.cu_seqlens_q = p.cu_seqlens_k = (const int32_t*)c.cu.data_ptr();
  } else {
    p.batch = (int32_t)q.size(0);
    p.seqlen_q = p.seqlen_k = (int32_t)q.size(1);
  }
  p.softmax_scale = c.scale;
  p.window_left = c.window;
  p.causal = 1;
  p.num_sink = c.num_sink;
  p.q = q.data_ptr();
  p.k = k.data_ptr();
  p.v = v.data_ptr();
  strides3(p.q_stride, q, c.packed);
  strides3(p.k_stride, k, c.packed);
  strides3(p.v_stride, v, c.packed);
  p.out = out.data_ptr();
  strides3(p.out_stride, out, c.packed);
  p.lse = (float*)lse.data_ptr();
  strides3(p.lse_stride, lse, c.packed);
  return p;
}

void* stream_of(const Tensor& t) {
  return (void*)c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.get_device()).stream();
}

// 0, or the library's status with nothing launched
int forward(const Call& c, const Tensor& q, const Tensor& k, const Tensor& v, Tensor& out, Tensor& lse) {
  c10::DeviceGuard guard(q.device());
  out = at::empty(q.sizes(), q.options());
  const auto f32 = q.options().dtype(at::kFloat);
  lse = c.packed ? at::empty({q.size(1), q.size(0)}, f32) : at::empty({q.size(0), q.size(2), q.size(1)}, f32);
  const rswa_attn_params p = params(c, q, k, v, out, lse);
  void* const stream = stream_of(q);
  pybind11::gil_scoped_release others_run;  // (a launch waits where the queue is full)
  return lib.fwd(&p, stream);
}

[[noreturn]] void throw_python() {
  python_error err;
  err.persist();
  throw std::move(err);
}

struct Refused {};  // by the library, ahead of any launch: the Python route says why

struct BandNode : torch::autograd::Function<BandNode> {
  static Tensor forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v, const Call& c) {
    Tensor out, lse;
    if (::forward(c, q, k, v, out, lse) != RSWA_OK) throw Refused{};
    ctx->save_for_backward({q, k, v, out, lse});
    if (c.packed) ctx->saved_data["cu"] = c.cu;
    ctx->saved_data["mask"] = c10::IValue(c10::List<int64_t>({c.packed, c.window, c.num_sink}));
    ctx->saved_data["scale"] = (double)c.scale;
    return out;
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list saved = ctx->get_saved_variables();
    const Tensor &q = saved[0], &k = saved[1], &v = saved[2], &out = saved[3], &lse = saved[4];
    const auto mask = ctx->saved_data["mask"].toIntList();
    const Call c{mask.get(0) != 0, (int32_t)mask.get(1), (int32_t)mask.get(2),
                 (float)ctx->saved_data["scale"].toDouble(),
                 mask.get(0) != 0 ? ctx->saved_data["cu"].toTensor() : Tensor()};
    Tensor dout = grads[0];
    if (dout.stride(-1) != 1) dout = dout.contiguous();
    const Tensor dq = at::empty_like(q), dk = at::empty_like(k), dv = at::empty_like(v);
    // (hooks of saved tensors may give back others: what does not fit is for the Python route to refuse)
    const bool as_saved = fits(q, k, v, c.packed) && like(out, q) && like(dout, q) && lse_of(lse, q, c.packed) &&
                          (!c.packed || c.cu.device() == q.device());
    const bool switched = [] {  // (the thread that waits for the engine has let go of the lock: no cost to be seen)
      pybind11::gil_scoped_acquire gil;
      return env_switches();
    }();
    if (!as_saved || switched) {
      pybind11::gil_scoped_acquire gil;
      PyObject* r = PyObject_CallFunction(
          lib.python_bwd, "NNNNNNNNNdiNi", THPVariable_Wrap(q), THPVariable_Wrap(k), THPVariable_Wrap(v),
          THPVariable_Wrap(out), THPVariable_Wrap(lse), THPVariable_Wrap(dout), THPVariable_Wrap(dq),
          THPVariable_Wrap(dk), THPVariable_Wrap(dv), (double)c.scale, (int)c.window, THPVariable_Wrap(c.cu),
          (int)c.num_sink);
      if (!r) throw_python();
      Py_DECREF(r);
    } else {
      c10::DeviceGuard guard(q.device());
      rswa_attn_params p = params(c, q, k, v, out, lse);
      p.dout = dout.data_ptr();
      p.dq = dq.data_ptr();
      p.dk = dk.data_ptr();
      p.dv = dv.data_ptr();
      strides3(p.dout_stride, dout, c.packed);
      strides3(p.dq_stride, dq, c.packed);
      strides3(p.dk_stride, dk, c.packed);
      strides3(p.dv_stride, dv, c.packed);
      const Tensor ws = at::empty({(int64_t)lib.bwd_bytes(&p)}, q.options().dtype(at::kByte));
      p.workspace = ws.data_ptr();
      p.workspace_bytes = (uint64_t)ws.numel();
      const int rc = lib.bwd(&p, stream_of(q));
      if (rc != RSWA_OK) {
        pybind11::gil_scoped_acquire gil;
        PyObject* r = PyObject_CallFunction(lib.raise, "i", rc);
        Py_XDECREF(r);
        if (!r) throw_python();
      }
    }
    return {dq, dk, dv, Tensor()};
  }
};

// band_attn(q, k, v, window, softmax_scale or None, cu_seqlens or None, num_sink) -> out or None
PyObject* band_attn(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 7 || !lib.fwd) Py_RETURN_NONE;
  for (int i = 0; i < 3; i++)
    if (!THPVariable_CheckExact(args[i])) Py_RETURN_NONE;
  const Tensor &q = THPVariable_Unpack(args[0]), &k = THPVariable_Unpack(args[1]), &v = THPVariable_Unpack(args[2]);
  Call c;
  c.packed = args[5] != Py_None;
  if (c.packed) {
    if (!THPVariable_CheckExact(args[5])) Py_RETURN_NONE;
    const Tensor& cu = c.cu = THPVariable_Unpack(args[5]);
    if (!plain(cu) || cu.scalar_type() != at::kInt || cu.dim() != 1 || !cu.is_contiguous() || cu.numel() < 2)
      Py_RETURN_NONE;
  }
  if (!fits(q, k, v, c.packed) || (c.packed && q.device() != c.cu.device()) || observed() || env_switches()) Py_RETURN_NONE;
  if (!PyLong_CheckExact(args[3]) || !PyLong_CheckExact(args[6])) Py_RETURN_NONE;
  int over = 0;
  const long long window = PyLong_AsLongLongAndOverflow(args[3], &over);
  if (over || window != (int32_t)window) Py_RETURN_NONE;
  const long long num_sink = PyLong_AsLongLongAndOverflow(args[6], &over);
  if (over || num_sink != (int32_t)num_sink) Py_RETURN_NONE;
  c.window = (int32_t)window;
  c.num_sink = (int32_t)num_sink;
  if (args[4] == Py_None) c.scale = (float)std::pow((double)q.size(-1), -0.5);
  else if (PyFloat_CheckExact(args[4])) c.scale = (float)PyFloat_AS_DOUBLE(args[4]);
  else Py_RETURN_NONE;
  Tensor out;
  if (c10::GradMode::is_enabled() && (q.requires_grad() || k.requires_grad() || v.requires_grad())) {
    try {
      out = BandNode::apply(q, k, v, c);
    } catch (const Refused&) {
      Py_RETURN_NONE;
    }
  } else {
    Tensor lse;
    if (forward(c, q, k, v, out, lse) != RSWA_OK) Py_RETURN_NONE;
  }
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// bind(rswa_attn_fwd, rswa_attn_bwd, rswa_attn_bwd_workspace_bytes, raise, python_bwd): addresses and callables
PyObject* bind(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 5) {
    PyErr_SetString(PyExc_TypeError, "bind takes three addresses and two callables");
    return nullptr;
  }
  void* at[3];
  for (int i = 0; i < 3; i++) {
    at[i] = PyLong_AsVoidPtr(args[i]);
    if (PyErr_Occurred()) return nullptr;
  }
  lib.bwd = reinterpret_cast<decltype(lib.bwd)>(at[1]);
  lib.bwd_bytes = reinterpret_cast<decltype(lib.bwd_bytes)>(at[2]);
  Py_INCREF(args[3]);
  Py_INCREF(args[4]);
  lib.raise = args[3];
  lib.python_bwd = args[4];
  lib.fwd = reinterpret_cast<decltype(lib.fwd)>(at[0]);
  Py_RETURN_NONE;
}

// The PyTorch whose headers this was compiled with (ring_swa._lib.torch_build): their inlined accessors read
// tensors at its layout, so that another must not be handed any
PyObject* torch_build(PyObject*, PyObject*) { return PyUnicode_FromString(RSWA_TORCH_BUILD); }

PyObject* params_bytes(PyObject*, PyObject*) { return PyLong_FromSize_t(sizeof(rswa_attn_params)); }

PyMethodDef methods[] = {
    {"band_attn", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(&band_attn)), METH_FASTCALL, nullptr},
    {"bind", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(&bind)), METH_FASTCALL, nullptr},
    {"params_bytes", &params_bytes, METH_NOARGS, nullptr},
    {"torch_build", &torch_build, METH_NOARGS, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "rswa_torch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_rswa_torch() { return PyModule_Create(&module); }
