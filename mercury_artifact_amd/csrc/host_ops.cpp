// Host side of the operators: argument checks, output and workspace allocation, stream lookup and the call into
// libmercury_hip.so, without a trip through the Python interpreter for each of them (about 40 strides, sizes and pointers
// per block call: 18 us of host time through ctypes and 30 with the operator's dispatcher, 6.5 and 7.5 here, where the
// kernels of a small block take 10).
//
// Every function takes the same arguments as the Python function of its name and does the whole call when the arguments
// are what the kernels take as they are; for anything else -- another type or layout, a device that is not the current one,
// a wrong shape, a tensor subclass -- it returns None without having done anything, and the Python function goes on to
// convert or to report.  The entry points of the library are handed over by address (bind), so that there is one place
// that decides which library is loaded.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/record_function.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/PythonTorchFunctionTLS.h>

#include "../../include/mercury_hip.h"

namespace {

struct Entry {
  decltype(&mhip_attn_fwd_block) fwd = nullptr;
  decltype(&mhip_attn_fwd_blocks) fwd_many = nullptr;
  decltype(&mhip_attn_fwd_group) fwd_group = nullptr;
  decltype(&mhip_attn_fwd_chain) fwd_chain = nullptr;
  decltype(&mhip_attn_bwd_workspace_bytes) bwd_bytes = nullptr;
  decltype(&mhip_attn_bwd_block) bwd = nullptr;
  decltype(&mhip_attn_bwd_chunk) chunk = nullptr;
  decltype(&mhip_attn_bwd_chunks) bwd_many = nullptr;
  decltype(&mhip_attn_bwd_take) bwd_take = nullptr;
  decltype(&mhip_lse_merge) merge = nullptr;
  decltype(&mhip_lse_merge_many) many = nullptr;
  decltype(&mhip_pack_reduce) pack = nullptr;
  decltype(&mhip_unpack) unpack = nullptr;
  decltype(&mhip_quantize_e4m3) quantize = nullptr;
  decltype(&mhip_error_string) error_string = nullptr;
} entry;
bool bound = false;

using at::Tensor;

// A device tensor that needs nothing of the dispatcher: exactly torch.Tensor, strided, no wrapper of a transform, no
// names (which the operators' schemas refuse).
const Tensor* plain(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const Tensor& t = THPVariable_Unpack(o);
  const auto keys = t.key_set();
  if (!t.is_cuda() || t.layout() != at::kStrided || keys.has(c10::DispatchKey::Python) ||
      keys.has(c10::DispatchKey::Functionalize) || keys.has(c10::DispatchKey::FuncTorchBatched) ||
      keys.has(c10::DispatchKey::FuncTorchGradWrapper) || keys.has(c10::DispatchKey::Negative) ||
      keys.has(c10::DispatchKey::Conjugate) || keys.has(c10::DispatchKey::ZeroTensor) || keys.has(c10::DispatchKey::Named))
    return nullptr;
  return &t;
}

// None counts as absent: returns false only for something that is neither None nor a plain tensor on `like`'s device.
bool optional(PyObject* o, const Tensor& like, const Tensor*& t) {
  t = nullptr;
  if (o == Py_None) return true;
  t = plain(o);
  return t && t->device() == like.device();
}

struct Args {                 // tensors of one call, all on one device
  PyObject* const* a;
  bool ok = true;
  const Tensor* first = nullptr;
  const Tensor& tensor(int i) {
    static const Tensor none;
    const Tensor* t = plain(a[i]);
    if (!t || (first && t->device() != first->device())) { ok = false; return none; }
    if (!first) first = t;
    return *t;
  }
};

// The tensor's current stream if its device is the current one.  A call for another device is left to the Python function,
// which changes the device for its duration (c10::hip's guards do not take the device of a tensor, whose type is "cuda").
struct OnDevice {
  bool current;
  hipStream_t stream = nullptr;
  explicit OnDevice(const Tensor& t) : current(c10::hip::current_device() == t.device().index()) {
    if (current) stream = c10::hip::getCurrentHIPStream(t.device().index()).stream();
  }
};

// Runs f while other Python threads may run, as every torch operator and every call through ctypes does: an allocation may
// wait for the device, and a launch waits while the queue is full.
template <class F>
int without_gil(F&& f) {
  struct Released {
    PyThreadState* state = PyEval_SaveThread();
    ~Released() { PyEval_RestoreThread(state); }
  } released;
  return f();
}

bool shape4(const Tensor& t, int64_t a, int64_t b, int64_t c, int64_t d) {
  return t.dim() == 4 && t.size(0) == a && t.size(1) == b && t.size(2) == c && t.size(3) == d;
}
bool shape3(const Tensor& t, int64_t a, int64_t b, int64_t c) {
  return t.dim() == 3 && t.size(0) == a && t.size(1) == b && t.size(2) == c;
}
bool same_layout(const Tensor& a, const Tensor& b) { return a.strides() == b.strides(); }
bool rows16(const Tensor& t) {            // 16-byte aligned bf16 rows with a contiguous last dimension
  return t.scalar_type() == at::kBFloat16 && t.stride(3) == 1 && t.stride(0) % 8 == 0 && t.stride(1) % 8 == 0 &&
         t.stride(2) % 8 == 0;
}
bool fits(std::initializer_list<int64_t> sizes) {
  for (int64_t s : sizes)
    if (s > INT32_MAX) return false;
  return true;
}
void* data(const Tensor* t) { return t ? t->data_ptr() : nullptr; }
float* floats(const Tensor* t) { return t ? static_cast<float*>(t->data_ptr()) : nullptr; }

PyObject* give(const Tensor& t) { return THPVariable_Wrap(t); }
PyObject* give2(const Tensor& a, const Tensor& b) {
  PyObject* r = PyTuple_New(2);
  if (!r) return nullptr;
  PyTuple_SET_ITEM(r, 0, give(a));
  PyTuple_SET_ITEM(r, 1, give(b));
  return r;
}
#define SLOW do { Py_RETURN_NONE; } while (0)

// What a code other than MHIP_OK means for the call: None for arguments the library refused before it launched anything
// (the Python function converts them or reports them); an error for anything else -- a kernel may have run, and a second
// call would add to its sums.
PyObject* refused(int code, const char* what) {
  switch (code) {
    case MHIP_EINVAL: case MHIP_EDTYPE: case MHIP_EHEADDIM: case MHIP_EALIGN: case MHIP_EUNSUPPORTED: case MHIP_ETOOLARGE:
      Py_RETURN_NONE;
    default:
      return PyErr_Format(PyExc_RuntimeError, "%s: %s (code %d)", what, entry.error_string(code), code);
  }
}
#define ENTER(n) if (nargs != (n) || !bound) SLOW

// Whether the torch operator of the name would do nothing but call its kernel: no mode, transform, trace or profiler is
// active and none of the tensors asks for a gradient.
PyObject* undispatched(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  bool yes = bound && !c10::impl::TorchDispatchModeTLS::any_modes_set() && !at::impl::torch_function_mode_enabled() &&
             !(at::isRecordFunctionEnabled() && at::hasCallbacks());
  if (yes) {
    using K = c10::DispatchKey;
    const auto in = c10::impl::tls_local_dispatch_key_set().included_;
    yes = !in.has_any(c10::DispatchKeySet({K::Python, K::Functionalize, K::FuncTorchDynamicLayerFrontMode,
                                           K::FuncTorchDynamicLayerBackMode, K::Tracer, K::PreDispatch}));
  }
  const bool grad = c10::GradMode::is_enabled();
  for (Py_ssize_t i = 0; yes && i < nargs; ++i) {
    if (a[i] == Py_None) continue;
    const Tensor* t = plain(a[i]);
    yes = t && !(grad && t->requires_grad());
  }
  return PyBool_FromLong(yes);
}

// Says that the tensors have been written to, as an operator does for the arguments it mutates: autograd compares the
// count with what it saved.
PyObject* written(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  for (Py_ssize_t i = 0; i < nargs; ++i) {
    if (!THPVariable_Check(a[i])) continue;
    const Tensor& t = THPVariable_Unpack(a[i]);
    if (t.defined() && !t.is_inference()) t.unsafeGetTensorImpl()->bump_version();
  }
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

// (chunk): whether the kernels take the rows of a chunk (2, B, Sc, Hkv, D) as they are -- contiguous last dimension, 16-byte
// aligned, the rows of one head within the reach of their 32-bit offsets (2 GiB; 1 GiB below 128 columns).
PyObject* rows_fit(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 1 || !THPVariable_Check(a[0])) SLOW;
  const Tensor& t = THPVariable_Unpack(a[0]);
  const int64_t size = t.element_size(), unit = 16 / size, last = t.dim() - 1;
  bool fit = last >= 3 && t.stride(last) == 1 && reinterpret_cast<uintptr_t>(t.const_data_ptr()) % 16 == 0;
  for (int64_t i = 0; fit && i < last; ++i) fit = t.stride(i) % unit == 0;
  fit = fit && t.size(2) * t.stride(2) * size < int64_t(1) << (t.size(last) == 128 ? 31 : 30);
  return PyBool_FromLong(fit);
  END_HANDLE_TH_ERRORS
}

// (t, *others): whether no other tensor has elements between the first and the last of t's.
PyObject* apart(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  auto extent = [](const Tensor& t) {
    const char* first = static_cast<const char*>(t.const_data_ptr());
    int64_t last = 0;
    for (int64_t i = 0; i < t.dim(); ++i) last += (t.size(i) - 1) * t.stride(i);
    return std::make_pair(first, t.numel() ? first + (last + 1) * t.element_size() : first);
  };
  for (Py_ssize_t i = 0; i < nargs; ++i)
    if (!THPVariable_Check(a[i])) SLOW;
  if (nargs < 1) SLOW;
  const auto mine = extent(THPVariable_Unpack(a[0]));
  for (Py_ssize_t i = 1; i < nargs; ++i) {
    const auto other = extent(THPVariable_Unpack(a[i]));
    if (other.first < mine.second && mine.first < other.second) Py_RETURN_FALSE;
  }
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

// (q, k, v, softmax_scale, causal, q_descale, k_descale, v_descale, out, lse)
PyObject* fwd_block(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  ENTER(10);
  Args in{a};
  const Tensor &q = in.tensor(0), &k = in.tensor(1), &v = in.tensor(2);
  if (!in.ok || q.dim() != 4 || k.dim() != 4) SLOW;
  const int64_t B = q.size(0), Sq = q.size(1), Hq = q.size(2), D = q.size(3), Sc = k.size(1), Hkv = k.size(2);
  const auto type = q.scalar_type();
  if ((type != at::kBFloat16 && type != at::kFloat8_e4m3fn) || k.scalar_type() != type || v.scalar_type() != type ||
      !shape4(k, B, Sc, Hkv, D) || !shape4(v, B, Sc, Hkv, D) || Hkv == 0 || Hq % Hkv || q.stride(3) != 1 || k.stride(3) != 1 ||
      v.stride(3) != 1 || !fits({B, Sq, Sc, Hq}))
    SLOW;
  const double scale = PyFloat_AsDouble(a[3]);
  if (scale == -1.0 && PyErr_Occurred()) { PyErr_Clear(); SLOW; }
  const int causal = PyObject_IsTrue(a[4]);
  if (causal < 0) { PyErr_Clear(); SLOW; }
  const Tensor* descale[3];
  for (int i = 0; i < 3; ++i) {
    if (!optional(a[5 + i], q, descale[i])) SLOW;
    if (descale[i] && (descale[i]->numel() != 1 || descale[i]->scalar_type() != at::kFloat)) SLOW;
  }
  const Tensor *out_given, *lse_given;
  if (!optional(a[8], q, out_given) || !optional(a[9], q, lse_given)) SLOW;
  if (out_given && (!shape4(*out_given, B, Sq, Hq, D) || out_given->scalar_type() != at::kBFloat16 || out_given->stride(3) != 1)) SLOW;
  if (lse_given && (!shape3(*lse_given, B, Hq, Sq) || lse_given->scalar_type() != at::kFloat || !lse_given->is_contiguous())) SLOW;
  OnDevice on(q);
  if (!on.current) SLOW;
  Tensor out, lse;
  const int code = without_gil([&] {
    out = out_given ? *out_given : at::empty({B, Sq, Hq, D}, q.options().dtype(at::kBFloat16).requires_grad(false));
    lse = lse_given ? *lse_given : at::empty({B, Hq, Sq}, q.options().dtype(at::kFloat).requires_grad(false));
    return entry.fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), floats(&lse),
                     B, Sq, Sc, Hq, Hkv, D, q.stride(0), q.stride(1), q.stride(2), k.stride(0), k.stride(1),
                     k.stride(2), v.stride(0), v.stride(1), v.stride(2), out.stride(0), out.stride(1), out.stride(2),
                     (float)scale, causal ? MHIP_MASK_CAUSAL : MHIP_MASK_NONE,
                     type == at::kBFloat16 ? MHIP_BF16 : MHIP_E4M3, floats(descale[0]), floats(descale[1]),
                     floats(descale[2]), on.stream);
  });
  if (code != MHIP_OK) return refused(code, "mhip_attn_fwd_block");
  return give2(out, lse);
  END_HANDLE_TH_ERRORS
}

// (q, blocks): how many of a step's blocks to launch together
PyObject* fwd_group(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  ENTER(2);
  const Tensor* q = plain(a[0]);
  const long blocks = PyLong_AsLong(a[1]);
  if (blocks == -1 && PyErr_Occurred()) { PyErr_Clear(); SLOW; }
  if (!q || q->dim() != 4 || q->size(2) == 0 || !fits({q->size(0), q->size(1), q->size(2), blocks})) SLOW;
  const int n = entry.fwd_group(q->size(0), q->size(1), q->size(2), blocks);
  if (n < 1) SLOW;
  return PyLong_FromLong(n);
  END_HANDLE_TH_ERRORS
}

// (q, chunk, n): how many of n chunks to put into one result
PyObject* fwd_chain(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  ENTER(3);
  const Tensor *q = plain(a[0]), *c = plain(a[1]);
  const long n = PyLong_AsLong(a[2]);
  if (n == -1 && PyErr_Occurred()) { PyErr_Clear(); SLOW; }
  if (!q || !c || q->dim() != 4 || c->dim() != 5 || q->size(2) == 0 ||
      !fits({q->size(0), q->size(1), q->size(2), q->size(3), c->size(2), n}))
    SLOW;
  const auto type = q->scalar_type();
  if (type != at::kBFloat16 && type != at::kFloat8_e4m3fn) SLOW;
  const int per = entry.fwd_chain(q->size(0), q->size(1), c->size(2), q->size(2), q->size(3), n > MHIP_MAX_GROUP ? MHIP_MAX_GROUP : n,
                                  type == at::kBFloat16 ? MHIP_BF16 : MHIP_E4M3);
  if (per < 1) SLOW;
  return PyLong_FromLong(per);
  END_HANDLE_TH_ERRORS
}

// (q, chunks, per, softmax_scale, causal, q_descale, k_descale, v_descale, outs, lses, first): the blocks of q against every
// (2, B, Sc, Hkv, D) tensor of the list in one launch, a result per `per` of them, into outs[first:] and lses[first:] -> True
PyObject* fwd_blocks(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  ENTER(11);
  if (!PyList_CheckExact(a[1])) SLOW;
  const Py_ssize_t n = PyList_GET_SIZE(a[1]);
  if (n < 1 || n > MHIP_MAX_GROUP) SLOW;
  const Tensor *q = plain(a[0]), *c0 = plain(PyList_GET_ITEM(a[1], 0)), *outs = plain(a[8]), *lses = plain(a[9]);
  if (!q || !c0 || !outs || !lses || q->dim() != 4 || c0->dim() != 5) SLOW;
  const int64_t B = q->size(0), Sq = q->size(1), Hq = q->size(2), D = q->size(3), Sc = c0->size(2), Hkv = c0->size(3);
  const auto type = q->scalar_type();
  if ((type != at::kBFloat16 && type != at::kFloat8_e4m3fn) || Hkv == 0 || Hq % Hkv || q->stride(3) != 1 || c0->stride(4) != 1 ||
      !fits({B, Sq, Sc, Hq}) || outs->device() != q->device() || lses->device() != q->device())
    SLOW;
  const void *ks[MHIP_MAX_GROUP], *vs[MHIP_MAX_GROUP];
  for (Py_ssize_t i = 0; i < n; ++i) {
    const Tensor* c = plain(PyList_GET_ITEM(a[1], i));
    if (!c || c->device() != q->device() || c->scalar_type() != type || c->dim() != 5 || c->size(0) != 2 || c->size(1) != B ||
        c->size(2) != Sc || c->size(3) != Hkv || c->size(4) != D || c->strides() != c0->strides())
      SLOW;
    ks[i] = c->data_ptr();
    vs[i] = static_cast<const char*>(ks[i]) + c->stride(0) * c->element_size();
  }
  const double scale = PyFloat_AsDouble(a[3]);
  if (scale == -1.0 && PyErr_Occurred()) { PyErr_Clear(); SLOW; }
  const int causal = PyObject_IsTrue(a[4]);
  const long first = PyLong_AsLong(a[10]), per = PyLong_AsLong(a[2]);
  if (causal < 0 || ((first == -1 || per == -1) && PyErr_Occurred())) { PyErr_Clear(); SLOW; }
  if (per < 1 || per > MHIP_MAX_GROUP) SLOW;
  const Py_ssize_t results = (n + per - 1) / per;
  const Tensor* descale[3];
  for (int i = 0; i < 3; ++i) {
    if (!optional(a[5 + i], *q, descale[i])) SLOW;
    if (descale[i] && (descale[i]->numel() != 1 || descale[i]->scalar_type() != at::kFloat)) SLOW;
  }
  if (outs->dim() != 5 || lses->dim() != 4 || first < 0 || first + results > outs->size(0) || first + results > lses->size(0) ||
      outs->sizes().slice(1) != q->sizes() || lses->size(1) != B || lses->size(2) != Hq || lses->size(3) != Sq ||
      outs->scalar_type() != at::kBFloat16 || lses->scalar_type() != at::kFloat || outs->stride(4) != 1 || !lses->is_contiguous())
    SLOW;
  OnDevice on(*q);
  if (!on.current) SLOW;
  const int code = without_gil([&] {
    return entry.fwd_many(q->data_ptr(), ks, vs, (int)n, (int)per, static_cast<char*>(outs->data_ptr()) + 2 * first * outs->stride(0),
                          outs->stride(0), floats(lses) + first * lses->stride(0), B, Sq, Sc, Hq, Hkv, D,
                          q->stride(0), q->stride(1), q->stride(2), c0->stride(1), c0->stride(2), c0->stride(3),
                          c0->stride(1), c0->stride(2), c0->stride(3), outs->stride(1), outs->stride(2), outs->stride(3),
                          (float)scale, causal ? MHIP_MASK_CAUSAL : MHIP_MASK_NONE,
                          type == at::kBFloat16 ? MHIP_BF16 : MHIP_E4M3, floats(descale[0]), floats(descale[1]),
                          floats(descale[2]), on.stream);
  });
  if (code != MHIP_OK) return refused(code, "mhip_attn_fwd_blocks");
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

// The two placeholders a forward operator returns besides: an empty tensor and two int64 (no dropout, never written).
PyObject* no_dropout(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  ENTER(1);
  const Tensor* q = plain(a[0]);
  if (!q) SLOW;
  return give2(at::empty({0}, q->options().dtype(at::kBFloat16).requires_grad(false)),
               at::empty({2}, q->options().dtype(at::kLong).requires_grad(false)));
  END_HANDLE_TH_ERRORS
}

Tensor bwd_workspace(const Tensor& q, int64_t Sc, int64_t Hkv) {
  return at::empty({entry.bwd_bytes(q.size(0), q.size(1), Sc, q.size(2), Hkv, q.size(3))},
                   q.options().dtype(at::kByte).requires_grad(false));
}

// (dout, q, k, v, out, softmax_lse, dq, dk, dv, softmax_scale, causal, deterministic, dq_acc) -> softmax_d
PyObject* bwd_block(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  ENTER(13);
  Args in{a};
  const Tensor &dout = in.tensor(0), &q = in.tensor(1), &k = in.tensor(2), &v = in.tensor(3), &out = in.tensor(4),
               &lse = in.tensor(5), &dq = in.tensor(6), &dk = in.tensor(7), &dv = in.tensor(8);
  if (!in.ok || q.dim() != 4 || k.dim() != 4) SLOW;
  const int64_t B = q.size(0), Sq = q.size(1), Hq = q.size(2), D = q.size(3), Sc = k.size(1), Hkv = k.size(2);
  for (const Tensor* t : {&dout, &q, &out, &dq})
    if (!shape4(*t, B, Sq, Hq, D) || !rows16(*t)) SLOW;
  for (const Tensor* t : {&k, &v, &dk, &dv})
    if (!shape4(*t, B, Sc, Hkv, D) || !rows16(*t)) SLOW;
  if (Hkv == 0 || Hq % Hkv || !same_layout(q, dout) || !same_layout(k, v) || !same_layout(dk, dv) ||
      !shape3(lse, B, Hq, Sq) || lse.scalar_type() != at::kFloat || !lse.is_contiguous() || !fits({B, Sq, Sc, Hq}))
    SLOW;
  const double scale = PyFloat_AsDouble(a[9]);
  if (scale == -1.0 && PyErr_Occurred()) { PyErr_Clear(); SLOW; }
  const int causal = PyObject_IsTrue(a[10]), deterministic = PyObject_IsTrue(a[11]);
  if (causal < 0 || deterministic < 0) { PyErr_Clear(); SLOW; }
  const Tensor* acc;
  if (!optional(a[12], q, acc)) SLOW;
  if (acc && (acc->sizes() != q.sizes() || acc->scalar_type() != at::kFloat || !acc->is_contiguous())) SLOW;
  OnDevice on(q);
  if (!on.current) SLOW;
  Tensor ws;
  const int code = without_gil([&] {
    ws = bwd_workspace(q, Sc, Hkv);
    return entry.bwd(dout.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), floats(&lse),
                     dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), floats(acc), B, Sq, Sc, Hq, Hkv, D,
                     q.stride(0), q.stride(1), q.stride(2), k.stride(0), k.stride(1), k.stride(2),
                     dk.stride(0), dk.stride(1), dk.stride(2), dq.stride(0), dq.stride(1), dq.stride(2),
                     out.stride(0), out.stride(1), out.stride(2), (float)scale,
                     causal ? MHIP_MASK_CAUSAL : MHIP_MASK_NONE, deterministic, ws.data_ptr(), on.stream);
  });
  if (code != MHIP_OK) return refused(code, "mhip_attn_bwd_block");
  // the workspace is (-delta | lse in base 2 | delta), each in a slot rounded up to 4 elements
  const int64_t rows = B * Hq * Sq, slot = (rows + 3) & ~int64_t(3);
  return give(ws.view(at::kFloat).narrow(0, 2 * slot, rows).view({B, Hq, Sq}));
  END_HANDLE_TH_ERRORS
}

// (dout, q, k, v, out, softmax_lse, dq, dq_acc, first, last, dkv, dkv32, softmax_scale, workspace) -> workspace
PyObject* bwd_chunk(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  ENTER(14);
  Args in{a};
  const Tensor &dout = in.tensor(0), &q = in.tensor(1), &k = in.tensor(2), &v = in.tensor(3), &out = in.tensor(4),
               &lse = in.tensor(5);
  if (!in.ok || q.dim() != 4 || k.dim() != 4) SLOW;
  const int64_t B = q.size(0), Sq = q.size(1), Hq = q.size(2), D = q.size(3), Sc = k.size(1), Hkv = k.size(2);
  const Tensor *dq, *acc, *dkv, *dkv32;
  if (!optional(a[6], q, dq) || !optional(a[7], q, acc) || !optional(a[10], q, dkv) || !optional(a[11], q, dkv32)) SLOW;
  for (const Tensor* t : {&dout, &q, &out, dq})
    if (t && (!shape4(*t, B, Sq, Hq, D) || !rows16(*t))) SLOW;
  for (const Tensor* t : {&k, &v})
    if (!shape4(*t, B, Sc, Hkv, D) || !rows16(*t)) SLOW;
  if (Hkv == 0 || Hq % Hkv || !same_layout(q, dout) || !same_layout(k, v) || !shape3(lse, B, Hq, Sq) ||
      lse.scalar_type() != at::kFloat || !lse.is_contiguous() || !fits({B, Sq, Sc, Hq}))
    SLOW;
  if (acc && (acc->sizes() != q.sizes() || acc->scalar_type() != at::kFloat || !acc->is_contiguous())) SLOW;
  const bool pair_shape_ok = [&] {
    for (const Tensor* t : {dkv, dkv32})
      if (t && !(t->dim() == 5 && t->size(0) == 2 && t->sizes().slice(1) == k.sizes())) return false;
    return true;
  }();
  if (!pair_shape_ok || (dkv32 && (dkv32->scalar_type() != at::kFloat || !dkv32->is_contiguous()))) SLOW;
  if (dkv && (dkv->scalar_type() != at::kBFloat16 || dkv->stride(4) != 1 || dkv->stride(0) % 8 || dkv->stride(1) % 8 ||
              dkv->stride(2) % 8 || dkv->stride(3) % 8))
    SLOW;
  const int first = PyObject_IsTrue(a[8]), last = PyObject_IsTrue(a[9]);
  const double scale = PyFloat_AsDouble(a[12]);
  if (first < 0 || last < 0 || (scale == -1.0 && PyErr_Occurred())) { PyErr_Clear(); SLOW; }
  const Tensor* kept;
  if (!optional(a[13], q, kept)) SLOW;
  if (kept && (kept->scalar_type() != at::kByte || !kept->is_contiguous() ||
               kept->numel() != entry.bwd_bytes(B, Sq, Sc, Hq, Hkv, D)))
    SLOW;
  OnDevice on(q);
  if (!on.current) SLOW;
  Tensor ws;
  auto second16 = [](const Tensor* t) { return t ? static_cast<void*>(static_cast<char*>(t->data_ptr()) + 2 * t->stride(0)) : nullptr; };
  const int code = without_gil([&] {
    ws = kept ? *kept : bwd_workspace(q, Sc, Hkv);
    return entry.chunk(dout.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), floats(&lse),
                       data(dq), floats(acc), first, last, kept != nullptr, data(dkv), second16(dkv),
                       floats(dkv32), dkv32 ? floats(dkv32) + dkv32->stride(0) : nullptr, B, Sq, Sc, Hq, Hkv, D,
                       q.stride(0), q.stride(1), q.stride(2), k.stride(0), k.stride(1), k.stride(2),
                       dkv ? dkv->stride(1) : 0, dkv ? dkv->stride(2) : 0, dkv ? dkv->stride(3) : 0,
                       dq ? dq->stride(0) : 0, dq ? dq->stride(1) : 0, dq ? dq->stride(2) : 0,
                       out.stride(0), out.stride(1), out.stride(2), (float)scale, MHIP_MASK_NONE, ws.data_ptr(),
                       on.stream);
  });
  if (code != MHIP_OK) return refused(code, "mhip_attn_bwd_chunk");
  return give(ws);
  END_HANDLE_TH_ERRORS
}

// (q, chunk, chunks): how many of a step's chunks to launch together
PyObject* bwd_group(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  ENTER(3);
  const Tensor *q = plain(a[0]), *c = plain(a[1]);
  const long n = PyLong_AsLong(a[2]);
  if (n == -1 && PyErr_Occurred()) { PyErr_Clear(); SLOW; }
  if (!q || !c || q->dim() != 4 || c->dim() != 5 || c->size(3) == 0 || q->size(2) % c->size(3) ||
      !fits({q->size(0), q->size(1), q->size(2), q->size(3), c->size(2), n}))
    SLOW;
  const int most = entry.bwd_take(q->size(0), q->size(1), c->size(2), q->size(2), c->size(3), q->size(3), n);
  if (most < 1) SLOW;
  return PyLong_FromLong(most);
  END_HANDLE_TH_ERRORS
}

// (dout, q, chunks, out, softmax_lse, dq, dq_acc, first, last, dkvs, dkv32s, softmax_scale, workspace) -> workspace: bwd_chunk
// over the (2, B, Sc, Hkv, D) tensors of a list in one launch; dkvs and dkv32s are lists of as many tensors or Nones
PyObject* bwd_chunks(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  ENTER(13);
  for (int i : {2, 9, 10})
    if (!PyList_CheckExact(a[i]) || PyList_GET_SIZE(a[i]) != PyList_GET_SIZE(a[2])) SLOW;
  const Py_ssize_t n = PyList_GET_SIZE(a[2]);
  if (n < 1 || n > MHIP_MAX_GROUP) SLOW;
  const Tensor *dout = plain(a[0]), *q = plain(a[1]), *c0 = plain(PyList_GET_ITEM(a[2], 0)), *out = plain(a[3]), *lse = plain(a[4]);
  if (!dout || !q || !c0 || !out || !lse || q->dim() != 4 || c0->dim() != 5) SLOW;
  const int64_t B = q->size(0), Sq = q->size(1), Hq = q->size(2), D = q->size(3), Sc = c0->size(2), Hkv = c0->size(3);
  const Tensor *dq, *acc, *kept;
  if (!optional(a[5], *q, dq) || !optional(a[6], *q, acc) || !optional(a[12], *q, kept)) SLOW;
  for (const Tensor* t : {dout, q, out, dq})
    if (t && (!shape4(*t, B, Sq, Hq, D) || !rows16(*t) || t->device() != q->device())) SLOW;
  if (Hkv == 0 || Hq % Hkv || !same_layout(*q, *dout) || lse->device() != q->device() || !shape3(*lse, B, Hq, Sq) ||
      lse->scalar_type() != at::kFloat || !lse->is_contiguous() || !fits({B, Sq, Sc, Hq}))
    SLOW;
  if (acc && (acc->sizes() != q->sizes() || acc->scalar_type() != at::kFloat || !acc->is_contiguous())) SLOW;
  auto rows = [](const Tensor& t) {
    return t.scalar_type() == at::kBFloat16 && t.stride(4) == 1 && t.stride(0) % 8 == 0 && t.stride(1) % 8 == 0 && t.stride(2) % 8 == 0 &&
           t.stride(3) % 8 == 0;
  };
  const void *ks[MHIP_MAX_GROUP], *vs[MHIP_MAX_GROUP];
  void *dks[MHIP_MAX_GROUP], *dvs[MHIP_MAX_GROUP];
  float *dk32s[MHIP_MAX_GROUP], *dv32s[MHIP_MAX_GROUP];
  const Tensor* g0 = nullptr;                     // the bf16 gradients have one layout
  for (Py_ssize_t i = 0; i < n; ++i) {
    const Tensor *c = plain(PyList_GET_ITEM(a[2], i)), *g, *g32;
    if (!c || c->device() != q->device() || c->dim() != 5 || c->size(0) != 2 || c->size(1) != B || c->size(2) != Sc ||
        c->size(3) != Hkv || c->size(4) != D || !rows(*c) || c->strides() != c0->strides() ||
        !optional(PyList_GET_ITEM(a[9], i), *q, g) || !optional(PyList_GET_ITEM(a[10], i), *q, g32))
      SLOW;
    if (g && (g->sizes() != c0->sizes() || !rows(*g) || (g0 && g->strides() != g0->strides()))) SLOW;
    if (g32 && (g32->sizes() != c0->sizes() || g32->scalar_type() != at::kFloat || !g32->is_contiguous())) SLOW;
    if (g && !g0) g0 = g;
    ks[i] = c->data_ptr();
    vs[i] = static_cast<const char*>(ks[i]) + 2 * c->stride(0);
    dks[i] = data(g);
    dvs[i] = g ? static_cast<char*>(dks[i]) + 2 * g->stride(0) : nullptr;
    dk32s[i] = floats(g32);
    dv32s[i] = g32 ? dk32s[i] + g32->stride(0) : nullptr;
  }
  const int first = PyObject_IsTrue(a[7]), last = PyObject_IsTrue(a[8]);
  const double scale = PyFloat_AsDouble(a[11]);
  if (first < 0 || last < 0 || (scale == -1.0 && PyErr_Occurred())) { PyErr_Clear(); SLOW; }
  if (kept && (kept->scalar_type() != at::kByte || !kept->is_contiguous() ||
               kept->numel() != entry.bwd_bytes(B, Sq, Sc, Hq, Hkv, D)))
    SLOW;
  OnDevice on(*q);
  if (!on.current) SLOW;
  Tensor ws;
  const int code = without_gil([&] {
    ws = kept ? *kept : bwd_workspace(*q, Sc, Hkv);
    return entry.bwd_many(dout->data_ptr(), q->data_ptr(), ks, vs, (int)n, out->data_ptr(), floats(lse), data(dq), floats(acc), first,
                          last, kept != nullptr, dks, dvs, dk32s, dv32s, B, Sq, Sc, Hq, Hkv, D,
                          q->stride(0), q->stride(1), q->stride(2), c0->stride(1), c0->stride(2), c0->stride(3),
                          g0 ? g0->stride(1) : 0, g0 ? g0->stride(2) : 0, g0 ? g0->stride(3) : 0,
                          dq ? dq->stride(0) : 0, dq ? dq->stride(1) : 0, dq ? dq->stride(2) : 0,
                          out->stride(0), out->stride(1), out->stride(2), (float)scale, ws.data_ptr(), on.stream);
  });
  if (code != MHIP_OK) return refused(code, "mhip_attn_bwd_chunks");
  return give(ws);
  END_HANDLE_TH_ERRORS
}

// (acc_out, acc_lse, block_out, block_lse, dst_out, dst_lse, final_out, final_lse) -> True
PyObject* merge_into(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  ENTER(8);
  const Tensor *bo = plain(a[2]), *bl = plain(a[3]);
  if (!bo || !bl || bo->device() != bl->device() || bo->dim() != 4) SLOW;
  const int64_t B = bo->size(0), Sq = bo->size(1), Hq = bo->size(2), D = bo->size(3);
  if (bo->scalar_type() != at::kBFloat16 || bo->stride(3) != 1 || !shape3(*bl, B, Hq, Sq) ||
      bl->scalar_type() != at::kFloat || bl->stride(2) != 1 || !fits({B, Sq, Hq, D}))
    SLOW;
  const Tensor *t[8];
  for (int i : {0, 1, 4, 5, 6, 7})
    if (!optional(a[i], *bo, t[i])) SLOW;
  for (int i : {0, 4, 6})
    if ((t[i] == nullptr) != (t[i + 1] == nullptr)) SLOW;
  for (int i : {0, 4})
    if (t[i] && (!shape4(*t[i], B, Sq, Hq, D) || !shape4(*t[i + 1], B, Sq, Hq, 1) || t[i]->scalar_type() != at::kFloat ||
                 t[i + 1]->scalar_type() != at::kFloat || t[i]->stride(3) != 1))
      SLOW;
  if (t[6] && (!shape4(*t[6], B, Sq, Hq, D) || !shape3(*t[7], B, Hq, Sq) || !t[6]->is_contiguous() ||
               !t[7]->is_contiguous() || t[6]->scalar_type() != at::kBFloat16 || t[7]->scalar_type() != at::kFloat))
    SLOW;
  OnDevice on(*bo);
  if (!on.current) SLOW;
  auto st = [](const Tensor* x, int i) { return x ? x->stride(i) : int64_t(0); };
  const int code = without_gil([&] {
    return entry.merge(floats(t[0]), floats(t[1]), bo->data_ptr(), floats(bl), floats(t[4]), floats(t[5]),
                       data(t[6]), floats(t[7]), B, Sq, Hq, D, st(t[0], 0), st(t[0], 1), st(t[0], 2),
                       st(t[1], 0), st(t[1], 1), st(t[1], 2), bo->stride(0), bo->stride(1), bo->stride(2),
                       bl->stride(0), bl->stride(1), st(t[4], 0), st(t[4], 1), st(t[4], 2), st(t[5], 0),
                       st(t[5], 1), st(t[5], 2), on.stream);
  });
  if (code != MHIP_OK) return refused(code, "mhip_lse_merge");
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

// (block_outs, block_lses, final_out, final_lse, row_begin or None): lists or tuples, or the blocks' results over all rows
// stacked in one tensor each, (n, B, Sq, Hq, D) and (n, B, Hq, Sq) -> True
PyObject* merge_many(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  ENTER(5);
  constexpr Py_ssize_t kMost = 64;
  if (const Tensor *outs = plain(a[0]), *lses = plain(a[1]); outs && lses) {
    const Tensor *out = plain(a[2]), *lse = plain(a[3]);
    if (a[4] != Py_None || !out || !lse || outs->dim() != 5 || lses->dim() != 4 || out->dim() != 4) SLOW;
    const int64_t n = outs->size(0), B = out->size(0), Sq = out->size(1), Hq = out->size(2), D = out->size(3);
    if (n < 1 || n > kMost || outs->sizes().slice(1) != out->sizes() || lses->size(0) != n || lses->size(1) != B || lses->size(2) != Hq ||
        lses->size(3) != Sq || outs->device() != out->device() || lses->device() != out->device() || lse->device() != out->device() ||
        outs->scalar_type() != at::kBFloat16 || !outs->is_contiguous() || lses->scalar_type() != at::kFloat || !lses->is_contiguous() ||
        out->scalar_type() != at::kBFloat16 || !out->is_contiguous() || !shape3(*lse, B, Hq, Sq) ||
        lse->scalar_type() != at::kFloat || !lse->is_contiguous() || B * Sq * Hq == 0 || !fits({B, Sq, Hq}))
      SLOW;
    const void* block_outs[kMost];
    const float* block_lses[kMost];
    int64_t strides[kMost];
    for (int64_t i = 0; i < n; ++i) {
      block_outs[i] = static_cast<const char*>(outs->data_ptr()) + 2 * i * outs->stride(0);
      block_lses[i] = floats(lses) + i * lses->stride(0);
      strides[i] = outs->stride(1);
    }
    OnDevice on(*out);
    if (!on.current) SLOW;
    const int code = without_gil([&] {
      return entry.many(block_outs, block_lses, strides, nullptr, (int)n, out->data_ptr(), floats(lse), B, Sq, Hq, D, outs->stride(2),
                        outs->stride(3), on.stream);
    });
    if (code != MHIP_OK) return refused(code, "mhip_lse_merge_many");
    Py_RETURN_TRUE;
  }
  auto list = [](PyObject* o) { return PyList_CheckExact(o) || PyTuple_CheckExact(o); };
  if (!list(a[0]) || !list(a[1]) || !(a[4] == Py_None || list(a[4]))) SLOW;
  const Py_ssize_t n = PySequence_Fast_GET_SIZE(a[0]);
  if (n < 1 || n > kMost || PySequence_Fast_GET_SIZE(a[1]) != n || (a[4] != Py_None && PySequence_Fast_GET_SIZE(a[4]) != n)) SLOW;
  const Tensor *out = plain(a[2]), *lse = plain(a[3]);
  if (!out || !lse || out->device() != lse->device() || out->dim() != 4) SLOW;
  const int64_t B = out->size(0), Sq = out->size(1), Hq = out->size(2), D = out->size(3);
  if (out->scalar_type() != at::kBFloat16 || !out->is_contiguous() || !shape3(*lse, B, Hq, Sq) ||
      lse->scalar_type() != at::kFloat || !lse->is_contiguous() || B * Sq * Hq == 0 || !fits({B, Sq, Hq}))
    SLOW;
  const void* outs[kMost];
  const float* lses[kMost];
  int64_t batch[kMost];
  int begins[kMost];
  int64_t ss = 0, sh = 0;
  for (Py_ssize_t i = 0; i < n; ++i) {
    const Tensor *bo = plain(PySequence_Fast_GET_ITEM(a[0], i)), *bl = plain(PySequence_Fast_GET_ITEM(a[1], i));
    if (!bo || !bl || bo->device() != out->device() || bl->device() != out->device() || bo->dim() != 4) SLOW;
    long begin = 0;
    if (a[4] != Py_None) {
      begin = PyLong_AsLong(PySequence_Fast_GET_ITEM(a[4], i));
      if (begin == -1 && PyErr_Occurred()) { PyErr_Clear(); SLOW; }
    }
    if (i == 0) { ss = bo->stride(1); sh = bo->stride(2); }
    // (a block that starts past the last row is left to the Python function)
    if (begin < 0 || begin >= Sq || !shape4(*bo, B, Sq - begin, Hq, D) || bo->scalar_type() != at::kBFloat16 ||
        bo->stride(3) != 1 || bo->stride(1) != ss || bo->stride(2) != sh || !shape3(*bl, B, Hq, Sq - begin) ||
        bl->scalar_type() != at::kFloat || !bl->is_contiguous())
      SLOW;
    outs[i] = bo->data_ptr();
    lses[i] = floats(bl);
    batch[i] = bo->stride(0);
    begins[i] = (int)begin;
  }
  OnDevice on(*out);
  if (!on.current) SLOW;
  const int code = without_gil([&] {
    return entry.many(outs, lses, batch, begins, (int)n, out->data_ptr(), floats(lse), B, Sq, Hq, D, ss, sh, on.stream);
  });
  if (code != MHIP_OK) return refused(code, "mhip_lse_merge_many");
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

// (block_out, block_lse, reduce_into) -> packed
PyObject* pack_block(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  ENTER(3);
  const Tensor *bo = plain(a[0]), *bl = plain(a[1]), *lhs;
  if (!bo || !bl || bo->device() != bl->device() || bo->dim() != 4 || !optional(a[2], *bo, lhs)) SLOW;
  const int64_t B = bo->size(0), Sq = bo->size(1), Hq = bo->size(2), D = bo->size(3);
  if (bo->scalar_type() != at::kBFloat16 || !bo->is_contiguous() || !shape3(*bl, B, Hq, Sq) ||
      bl->scalar_type() != at::kFloat || !bl->is_contiguous() || !fits({B, Sq, Hq, D}))
    SLOW;
  if (lhs && (!shape4(*lhs, B, Sq, Hq, D + 1) || lhs->scalar_type() != at::kFloat || !lhs->is_contiguous())) SLOW;
  OnDevice on(*bo);
  if (!on.current) SLOW;
  Tensor dst;
  const int code = without_gil([&] {
    dst = at::empty({B, Sq, Hq, D + 1}, bo->options().dtype(at::kFloat).requires_grad(false));
    return entry.pack(floats(lhs), bo->data_ptr(), floats(bl), floats(&dst), B, Sq, Hq, D, on.stream);
  });
  if (code != MHIP_OK) return refused(code, "mhip_pack_reduce");
  return give(dst);
  END_HANDLE_TH_ERRORS
}

// (buf, out, lse) -> True
PyObject* unpack_into(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  ENTER(3);
  Args in{a};
  const Tensor &buf = in.tensor(0), &out = in.tensor(1), &lse = in.tensor(2);
  if (!in.ok || out.dim() != 4) SLOW;
  const int64_t B = out.size(0), Sq = out.size(1), Hq = out.size(2), D = out.size(3);
  if (!shape4(buf, B, Sq, Hq, D + 1) || buf.scalar_type() != at::kFloat || !buf.is_contiguous() ||
      out.scalar_type() != at::kBFloat16 || !out.is_contiguous() || !shape3(lse, B, Hq, Sq) ||
      lse.scalar_type() != at::kFloat || !lse.is_contiguous() || !fits({B, Sq, Hq, D}))
    SLOW;
  OnDevice on(buf);
  if (!on.current) SLOW;
  const int code = without_gil([&] { return entry.unpack(floats(&buf), out.data_ptr(), floats(&lse), B, Sq, Hq, D, on.stream); });
  if (code != MHIP_OK) return refused(code, "mhip_unpack");
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

// (x) -> (x_q, scale)
PyObject* quantize_e4m3(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  ENTER(1);
  const Tensor* x = plain(a[0]);
  if (!x || (x->scalar_type() != at::kFloat && x->scalar_type() != at::kBFloat16) || !x->is_contiguous()) SLOW;
  OnDevice on(*x);
  if (!on.current) SLOW;
  Tensor xq, ws;                                   // ws: scale, scratch
  const int code = without_gil([&] {
    xq = at::empty(x->sizes(), x->options().dtype(at::kFloat8_e4m3fn).requires_grad(false));
    ws = at::empty({2}, x->options().dtype(at::kFloat).requires_grad(false));
    float* w = floats(&ws);
    return entry.quantize(x->data_ptr(), x->scalar_type() == at::kFloat ? MHIP_F32 : MHIP_BF16, x->numel(), xq.data_ptr(), w, w + 1,
                          on.stream);
  });
  if (code != MHIP_OK) return refused(code, "mhip_quantize_e4m3");
  return give2(xq, ws.select(0, 0));
  END_HANDLE_TH_ERRORS
}

// ({name: address}) of the library's entry points
PyObject* bind(PyObject*, PyObject* table) {
  auto get = [&](const char* name) -> void* {
    PyObject* v = PyDict_GetItemString(table, name);
    return v ? PyLong_AsVoidPtr(v) : nullptr;
  };
  bound = false;
  auto take = [&](auto& f, const char* name) { f = reinterpret_cast<std::decay_t<decltype(f)>>(get(name)); return f != nullptr; };
  const bool ok = take(entry.fwd, "mhip_attn_fwd_block") && take(entry.fwd_many, "mhip_attn_fwd_blocks") &&
                  take(entry.fwd_group, "mhip_attn_fwd_group") && take(entry.fwd_chain, "mhip_attn_fwd_chain") &&
                  take(entry.bwd_bytes, "mhip_attn_bwd_workspace_bytes") &&
                  take(entry.bwd, "mhip_attn_bwd_block") && take(entry.chunk, "mhip_attn_bwd_chunk") &&
                  take(entry.bwd_many, "mhip_attn_bwd_chunks") && take(entry.bwd_take, "mhip_attn_bwd_take") &&
                  take(entry.merge, "mhip_lse_merge") && take(entry.many, "mhip_lse_merge_many") &&
                  take(entry.pack, "mhip_pack_reduce") && take(entry.unpack, "mhip_unpack") &&
                  take(entry.quantize, "mhip_quantize_e4m3") && take(entry.error_string, "mhip_error_string");
  if (PyErr_Occurred()) return nullptr;
  bound = ok;
  return PyBool_FromLong(ok);
}

#define FAST(name) {#name, (PyCFunction)(void (*)(void))name, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    FAST(undispatched), FAST(written), FAST(apart), FAST(rows_fit), FAST(fwd_block), FAST(fwd_group), FAST(fwd_chain), FAST(fwd_blocks), FAST(no_dropout), FAST(bwd_block),
    FAST(bwd_chunk), FAST(bwd_group), FAST(bwd_chunks), FAST(merge_into), FAST(merge_many), FAST(pack_block), FAST(unpack_into), FAST(quantize_e4m3),
    {"bind", bind, METH_O, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_mercury_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// abi_version: of the header this module was compiled with; whoever binds a library compares it with the library's
PyMODINIT_FUNC PyInit__mercury_host() {
  PyObject* m = PyModule_Create(&module);
  if (m && PyModule_AddIntConstant(m, "abi_version", MHIP_ABI_VERSION) < 0) Py_CLEAR(m);
  return m;
}
