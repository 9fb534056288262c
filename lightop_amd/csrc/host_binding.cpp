// Host path of the calls a serving loop makes on every step: the whole fused-experts layer and the two routers.
//
// A one-token layer is two kernel launches, 17 us of GPU time; marshalling the same call through Python (argument
// checks on fifteen tensors, ctypes conversions, stream and workspace look-ups) took 25-27 us of host time and set
// the pace of the loop.  Here the ordinary call - tensors of the expected types, contiguous, on the current device,
// one chunk - is checked, given its workspace and launched natively.  Anything else (a conversion to make, several
// chunks, a tuning file, a stream being captured, an argument to refuse) is declined by returning None, and the Python
// code beside it does what it always did, error messages included: nothing is decided in two places.  What torch throws in
// here reaches Python as torch's own exception types (an allocation that fails is torch.OutOfMemoryError).
//
// The kernels' entry points are the C ABI of include/lightop_mi355.h, handed over by address (the library is the one
// `lightop_amd._lib` has loaded, whichever file that is).
#include <Python.h>

#include <ATen/Functions.h>
#include <ATen/core/Tensor.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cerrno>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <mutex>
#include <vector>

#include "../../include/lightop_mi355.h"

namespace {

decltype(&lo_fused_experts_block_int8) g_block = nullptr;
decltype(&lo_fused_experts_channel_int8) g_channel = nullptr;
decltype(&lo_fused_experts_workspace_bytes) g_ws_bytes = nullptr;
decltype(&lo_topk_softmax) g_topk_softmax = nullptr;
decltype(&lo_moe_fused_gate) g_gate = nullptr;
decltype(&lo_last_error) g_last_error = nullptr;

PyObject *s_preshuffled, *s_int4, *s_kmajor; // attribute names of weights in their load-time layout

// A torch.Tensor or nn.Parameter proper; subclasses may mean something else by their attributes and stay in Python.
const at::Tensor *tensor_of(PyObject *o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  return &THPVariable_Unpack(o);
}

// Whether the tensor object carries a true attribute `name` (an entry of its instance dictionary: asking for an attribute
// that is not there would raise and clear an exception on every call with row-major weights).
bool flag_of(PyObject *o, PyObject *name) {
  PyObject *d = PyObject_GenericGetDict(o, nullptr);
  PyObject *v = d ? PyDict_GetItemWithError(d, name) : nullptr;
  const int is = v ? PyObject_IsTrue(v) : 0;
  Py_XDECREF(d);
  if (PyErr_Occurred()) PyErr_Clear();
  return is == 1;
}

bool plain(const at::Tensor &t, int device) { return t.is_cuda() && t.get_device() == device && t.is_contiguous(); }

// LMSLIM_FUSED_MOE_CHUNK_SIZE as lightop_amd.envs reads it; -1 if it is not a plain number.
int64_t chunk_size() {
  for (const char *name : {"LMSLIM_FUSED_MOE_CHUNK_SIZE", "VLLM_FUSED_MOE_CHUNK_SIZE"}) {
    const char *v = std::getenv(name);
    if (!v || !*v) continue;
    char *end = nullptr;
    errno = 0;
    const long long n = std::strtoll(v, &end, 10);
    return errno || *end || n <= 0 ? -1 : n;
  }
  return 16 * 1024;
}

// Blocking work (allocations, which may wait for the GPU when memory is short; launches, which wait while the stream's queue
// is full and, for the first call of an activation, for its table) is done without the interpreter lock, as torch and ctypes
// do it: Python threads, or a callback on the stream, may have to run until it is through.  What it needs of the tensors is
// taken from them before.
struct NoGil {
  PyThreadState *state = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(state); }
};

// ---- workspaces ----------------------------------------------------------------------------------------
// The library's scratch for a whole-path call, one per (device, stream) and grown on demand, so that a serving loop
// does not allocate on every call.  Calls on one stream run in order and can share it; calls on different streams get
// workspaces of their own, and of several threads on one stream only one queues its launches at a time, so that
// a workspace holds one call's intermediates from the first launch to the last.  At most kMaxWorkspaces are kept: beyond
// that the one that was used longest ago goes back to the caching allocator (it was allocated on its own stream, so its
// memory is reused in that stream's order), as does one that a larger call outgrows.  A graph would keep the address of
// such memory, so none of it is ever captured: calls on a stream that is being captured are declined, and get scratch that
// lives as long as the graph.  The locks are taken without the interpreter lock, whose holder may be waiting for them.
struct Scratch {
  at::Tensor buf;
  std::mutex busy; // held while a call's launches are queued
};
struct Workspace {
  int device;
  hipStream_t stream;
  std::shared_ptr<Scratch> scratch;
};
constexpr size_t kMaxWorkspaces = 16;
std::vector<Workspace> &workspaces() { // most recently used first; never destroyed (the allocator may be gone by then)
  static auto *v = new std::vector<Workspace>();
  return *v;
}

std::shared_ptr<Scratch> new_workspace(int64_t bytes, int device) {
  auto s = std::make_shared<Scratch>();
  s->buf = at::empty({std::max<int64_t>(bytes, 1 << 20)},
                     at::TensorOptions().dtype(at::kByte).device(at::Device(at::kCUDA, static_cast<c10::DeviceIndex>(device))));
  return s;
}

std::shared_ptr<Scratch> workspace_for(int64_t bytes, int device, hipStream_t stream) {
  static std::mutex table;
  const std::lock_guard<std::mutex> lock(table);
  auto &all = workspaces();
  size_t i = 0;
  while (i < all.size() && !(all[i].device == device && all[i].stream == stream)) ++i;
  if (i == all.size()) {
    if (all.size() >= kMaxWorkspaces) all.pop_back();
    all.push_back({device, stream, new_workspace(bytes, device)});
    i = all.size() - 1;
  } else if (all[i].scratch->buf.numel() < bytes) {
    all[i].scratch.reset(); // back to the allocator first: the larger one may take its place
    try {
      all[i].scratch = new_workspace(bytes, device);
    } catch (...) {
      all.erase(all.begin() + static_cast<std::ptrdiff_t>(i));
      throw;
    }
  }
  for (; i > 0; --i) std::swap(all[i], all[i - 1]);
  return all[0].scratch;
}

PyObject *raise(int rc) {
  const char *msg = g_last_error ? g_last_error() : nullptr;
  PyErr_Format(PyExc_RuntimeError, "lightop_amd: %s (code %d)", msg && *msg ? msg : "error", rc);
  return nullptr;
}

// Whether work put on the stream goes into a graph (the legacy default stream cannot be captured).
bool capturing(hipStream_t stream) {
  if (!stream) return false;
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream, &status) == hipSuccess) return status != hipStreamCaptureStatusNone;
  (void)hipGetLastError();
  return true;
}

int device_now() {
  int d = -1;
  return hipGetDevice(&d) == hipSuccess ? d : -1;
}

int dtype_code(at::ScalarType t) {
  switch (t) {
  case at::kBFloat16: return LO_BF16;
  case at::kHalf: return LO_F16;
  case at::kFloat: return LO_F32;
  default: return -1;
  }
}

// fused_experts(hidden, w1, w2, topk_weights, topk_ids, cache13, w1_scale, w2_scale, expert_map, shared_output,
//               form, inplace, mul_on_input, global_num_experts, factor, flags) -> tensor, or None: not an ordinary call.
// form: 0 block scales, 1 per-channel scales, 2 packed int4 with K-group scales, 3 packed int4 with per-channel scales.
PyObject *fused_experts(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  if (nargs != 16) {
    PyErr_SetString(PyExc_TypeError, "fused_experts takes 16 arguments");
    return nullptr;
  }
  const at::Tensor *t[10];
  for (int i = 0; i < 8; ++i)
    if (!(t[i] = tensor_of(args[i]))) Py_RETURN_NONE;
  for (int i = 8; i < 10; ++i) {
    t[i] = nullptr;
    if (args[i] != Py_None && !(t[i] = tensor_of(args[i]))) Py_RETURN_NONE;
  }
  const long form = PyLong_AsLong(args[10]);
  const int inplace = PyObject_IsTrue(args[11]), mul_on_input = PyObject_IsTrue(args[12]);
  if (!PyLong_Check(args[13]) || !(PyFloat_Check(args[14]) || PyLong_Check(args[14]))) Py_RETURN_NONE;
  long long experts = PyLong_AsLongLong(args[13]);
  const double factor = PyFloat_AsDouble(args[14]);
  long flags = PyLong_AsLong(args[15]);
  if (inplace < 0 || mul_on_input < 0 || PyErr_Occurred()) return nullptr;
  HANDLE_TH_ERRORS
  const at::Tensor &x = *t[0], &w1 = *t[1], &w2 = *t[2], &tw = *t[3], &ids = *t[4], &cache = *t[5], &s1 = *t[6], &s2 = *t[7];
  if (!x.is_cuda() || x.get_device() != device_now()) Py_RETURN_NONE;
  const int dev = x.get_device();
  for (int i = 0; i < 10; ++i)
    if (t[i] && !plain(*t[i], dev)) Py_RETURN_NONE;
  const bool w4 = form >= 2, channel = form == 1 || form == 3;
  const int dtype = dtype_code(x.scalar_type());
  if (dtype < 0 || (dtype == LO_F32 && form != 0)) Py_RETURN_NONE;
  if (x.dim() != 2 || w1.dim() != 3 || w2.dim() != 3 || ids.dim() != 2 || tw.sizes() != ids.sizes()) Py_RETURN_NONE;
  const int64_t M = x.size(0), H = x.size(1), E = w1.size(0), N = w1.size(1), I = N / 2, k = ids.size(1);
  const int pack = w4 ? 2 : 1;
  if (M == 0 || ids.size(0) != M || N % 256 || H % 128 || w1.size(2) * pack != H || w2.size(0) != E || w2.size(1) != H ||
      w2.size(2) * pack != I)
    Py_RETURN_NONE;
  const at::ScalarType wt = w1.scalar_type();
  if (w2.scalar_type() != wt || !(wt == at::kChar || (w4 && wt == at::kByte))) Py_RETURN_NONE;
  if (tw.scalar_type() != at::kFloat || s1.scalar_type() != at::kFloat || s2.scalar_type() != at::kFloat) Py_RETURN_NONE;
  const bool ids64 = ids.scalar_type() == at::kLong;
  if (!ids64 && ids.scalar_type() != at::kInt) Py_RETURN_NONE;
  if (cache.scalar_type() != x.scalar_type() || cache.numel() < M * k * std::max(N, H)) Py_RETURN_NONE;
  if (t[8] && t[8]->scalar_type() != at::kInt) Py_RETURN_NONE;
  if (t[9] && (t[9]->scalar_type() != x.scalar_type() || t[9]->sizes() != x.sizes())) Py_RETURN_NONE;
  const bool pre = flag_of(args[1], s_preshuffled);
  if (flag_of(args[2], s_preshuffled) != pre) Py_RETURN_NONE;
  if (w4 && !(flag_of(args[1], s_int4) && flag_of(args[2], s_int4))) Py_RETURN_NONE;
  if (channel) {
    if (s1.numel() != E * N || s2.numel() != E * H) Py_RETURN_NONE;
  } else if (form == 2) {
    if (!flag_of(args[6], s_kmajor) || !flag_of(args[7], s_kmajor) || s1.sizes() != at::IntArrayRef({E, H / 128, N}) ||
        s2.sizes() != at::IntArrayRef({E, I / 128, H}))
      Py_RETURN_NONE;
  } else if (s1.sizes() != at::IntArrayRef({E, N / 128, H / 128}) || s2.sizes() != at::IntArrayRef({E, H / 128, I / 128})) {
    Py_RETURN_NONE;
  }
  if (experts == -1) experts = E;
  if (experts < E || experts > INT32_MAX || k < 1 || k > INT32_MAX) Py_RETURN_NONE;
  if (t[8] && t[8]->numel() < experts) Py_RETURN_NONE;
  const int64_t chunk = chunk_size();
  if (M > chunk) Py_RETURN_NONE; // several chunks, or a size that is not a number
  if (const char *d = std::getenv("TRITON_JSON_DIR"); d && *d) Py_RETURN_NONE; // a tuning file may hold a block size
  if (pre) flags |= LO_GEMM_W_PRESHUFFLED;
  if (w4) flags |= LO_GEMM_W4;

  const int64_t bytes = g_ws_bytes(M, static_cast<int32_t>(k), H, I, static_cast<int32_t>(experts), 0);
  if (bytes < 0) return raise(static_cast<int>(bytes));
  const hipStream_t stream = c10::hip::getCurrentHIPStream(static_cast<c10::DeviceIndex>(dev)).stream();
  if (capturing(stream)) Py_RETURN_NONE;
  const auto entry = channel ? g_channel : g_block;
  const auto sizes = x.sizes().vec();
  const auto options = x.options().requires_grad(false);
  const auto call = [=, xp = x.data_ptr(), w1p = static_cast<const int8_t *>(w1.data_ptr()), s1p = s1.data_ptr<float>(),
                     w2p = static_cast<const int8_t *>(w2.data_ptr()), s2p = s2.data_ptr<float>(), twp = tw.data_ptr<float>(),
                     idp = ids.data_ptr(), map = t[8] ? t[8]->data_ptr<int32_t>() : nullptr,
                     shared = t[9] ? t[9]->data_ptr() : nullptr, cp = cache.data_ptr()](void *dst, const at::Tensor &ws) { // dst null: in place
    const uintptr_t base = reinterpret_cast<uintptr_t>(ws.data_ptr()), aligned = (base + 255) / 256 * 256;
    return entry(xp, dtype, M, H, I, static_cast<int32_t>(E), static_cast<int32_t>(experts), static_cast<int32_t>(k), w1p, s1p,
                 w2p, s2p, twp, idp, ids64 ? LO_I64 : LO_I32, map, mul_on_input, static_cast<float>(factor), shared, cp, dst ? dst : xp,
                 reinterpret_cast<void *>(aligned), ws.numel() - static_cast<int64_t>(aligned - base), 0,
                 static_cast<int>(flags), stream);
  };
  at::Tensor out;
  int rc;
  {
    const NoGil nogil;
    const std::shared_ptr<Scratch> ws = workspace_for(bytes, dev, stream);
    if (!inplace) out = at::empty(sizes, options);
    const std::lock_guard<std::mutex> lock(ws->busy);
    rc = call(inplace ? nullptr : out.data_ptr(), ws->buf);
  }
  if (rc < 0) return raise(rc);
  if (inplace) {
    Py_INCREF(args[0]);
    return args[0];
  }
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// topk_softmax(weights, indices, source_rows, gating, renormalize) -> True, or None: not an ordinary call.
PyObject *topk_softmax(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  if (nargs != 5) {
    PyErr_SetString(PyExc_TypeError, "topk_softmax takes 5 arguments");
    return nullptr;
  }
  const at::Tensor *w = tensor_of(args[0]), *idx = tensor_of(args[1]), *g = tensor_of(args[3]), *src = nullptr;
  if (!w || !idx || !g || (args[2] != Py_None && !(src = tensor_of(args[2])))) Py_RETURN_NONE;
  const int renorm = PyObject_IsTrue(args[4]);
  if (renorm < 0) return nullptr;
  HANDLE_TH_ERRORS
  if (!g->is_cuda() || g->get_device() != device_now()) Py_RETURN_NONE;
  const int dev = g->get_device();
  if (!plain(*g, dev) || !plain(*w, dev) || !plain(*idx, dev) || (src && !plain(*src, dev))) Py_RETURN_NONE;
  if (g->dim() != 2 || w->dim() < 1) Py_RETURN_NONE;
  const int64_t T = g->size(0), E = g->size(1), k = w->size(-1);
  const int dtype = dtype_code(g->scalar_type());
  if (dtype < 0 || w->scalar_type() != at::kFloat || w->numel() != T * k || idx->numel() != T * k) Py_RETURN_NONE;
  const bool i64 = idx->scalar_type() == at::kLong;
  if (!i64 && idx->scalar_type() != at::kInt) Py_RETURN_NONE;
  if (src && (src->scalar_type() != at::kInt || src->numel() != T * k)) Py_RETURN_NONE;
  if (E > INT32_MAX || k > INT32_MAX) Py_RETURN_NONE;
  const hipStream_t stream = c10::hip::getCurrentHIPStream(static_cast<c10::DeviceIndex>(dev)).stream();
  const void *gp = g->data_ptr();
  float *const wp = w->data_ptr<float>();
  void *const ip = idx->data_ptr();
  int32_t *const sp = src ? src->data_ptr<int32_t>() : nullptr;
  int rc;
  {
    const NoGil nogil;
    rc = g_topk_softmax(gp, dtype, T, static_cast<int32_t>(E), static_cast<int32_t>(k), renorm, wp, ip, i64 ? LO_I64 : LO_I32, sp,
                        stream);
  }
  if (rc < 0) return raise(rc);
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

// fused_gate(input, bias, groups, topk_group, topk, n_share, factor, factor_on_output, int64_indices)
//   -> (weights, indices), or None: not an ordinary call.
PyObject *fused_gate(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  if (nargs != 9) {
    PyErr_SetString(PyExc_TypeError, "fused_gate takes 9 arguments");
    return nullptr;
  }
  const at::Tensor *x = tensor_of(args[0]), *b = tensor_of(args[1]);
  if (!x || !b) Py_RETURN_NONE;
  long v[4];
  for (int i = 0; i < 4; ++i) {
    if (!PyLong_Check(args[2 + i])) Py_RETURN_NONE;
    v[i] = PyLong_AsLong(args[2 + i]);
    if (PyErr_Occurred()) return nullptr;
    if (v[i] < 0 || v[i] > INT32_MAX) Py_RETURN_NONE;
  }
  if (!(PyFloat_Check(args[6]) || PyLong_Check(args[6]))) Py_RETURN_NONE;
  const double factor = PyFloat_AsDouble(args[6]);
  const int on_output = PyObject_IsTrue(args[7]), i64 = PyObject_IsTrue(args[8]);
  if (on_output < 0 || i64 < 0 || PyErr_Occurred()) return nullptr;
  HANDLE_TH_ERRORS
  if (!x->is_cuda() || x->get_device() != device_now()) Py_RETURN_NONE;
  const int dev = x->get_device();
  if (!plain(*x, dev) || !plain(*b, dev) || x->dim() != 2 || b->dim() != 1 || b->numel() != x->size(1)) Py_RETURN_NONE;
  const int dt = dtype_code(x->scalar_type()), bt = dtype_code(b->scalar_type());
  if (dt < 0 || bt < 0 || x->size(1) > INT32_MAX) Py_RETURN_NONE;
  const int64_t T = x->size(0), E = x->size(1), topk = v[2];
  const hipStream_t stream = c10::hip::getCurrentHIPStream(static_cast<c10::DeviceIndex>(dev)).stream();
  const void *xp = x->data_ptr(), *bp = b->data_ptr();
  const auto opts = x->options().requires_grad(false);
  at::Tensor weights, indices;
  int rc;
  {
    const NoGil nogil;
    weights = at::empty({T, topk}, opts.dtype(at::kFloat));
    indices = at::empty({T, topk}, opts.dtype(i64 ? at::kLong : at::kInt));
    rc = g_gate(xp, dt, bp, bt, T, static_cast<int32_t>(E), static_cast<int32_t>(v[0]), static_cast<int32_t>(v[1]),
                static_cast<int32_t>(v[2]), static_cast<int32_t>(v[3]), factor, on_output, weights.data_ptr<float>(),
                indices.data_ptr(), i64 ? LO_I64 : LO_I32, stream);
  }
  if (rc < 0) return raise(rc);
  PyObject *pw = THPVariable_Wrap(std::move(weights)), *pi = THPVariable_Wrap(std::move(indices));
  PyObject *pair = PyList_New(2);
  if (!pw || !pi || !pair) {
    Py_XDECREF(pw);
    Py_XDECREF(pi);
    Py_XDECREF(pair);
    return nullptr;
  }
  PyList_SET_ITEM(pair, 0, pw);
  PyList_SET_ITEM(pair, 1, pi);
  return pair;
  END_HANDLE_TH_ERRORS
}

// bind(lo_fused_experts_block_int8, lo_fused_experts_channel_int8, lo_fused_experts_workspace_bytes, lo_topk_softmax,
//      lo_moe_fused_gate, lo_last_error): addresses of the library's functions.
PyObject *bind(PyObject *, PyObject *args) {
  unsigned long long a[6];
  if (!PyArg_ParseTuple(args, "KKKKKK", &a[0], &a[1], &a[2], &a[3], &a[4], &a[5])) return nullptr;
  g_block = reinterpret_cast<decltype(g_block)>(a[0]);
  g_channel = reinterpret_cast<decltype(g_channel)>(a[1]);
  g_ws_bytes = reinterpret_cast<decltype(g_ws_bytes)>(a[2]);
  g_topk_softmax = reinterpret_cast<decltype(g_topk_softmax)>(a[3]);
  g_gate = reinterpret_cast<decltype(g_gate)>(a[4]);
  g_last_error = reinterpret_cast<decltype(g_last_error)>(a[5]);
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"bind", bind, METH_VARARGS, nullptr},
    {"fused_experts", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(fused_experts)), METH_FASTCALL, nullptr},
    {"topk_softmax", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(topk_softmax)), METH_FASTCALL, nullptr},
    {"fused_gate", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(fused_gate)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

} // namespace

PyMODINIT_FUNC PyInit__host(void) {
  s_preshuffled = PyUnicode_InternFromString("lo_preshuffled");
  s_int4 = PyUnicode_InternFromString("lo_int4");
  s_kmajor = PyUnicode_InternFromString("lo_kmajor");
  if (!s_preshuffled || !s_int4 || !s_kmajor) return nullptr;
  PyObject *m = PyModule_Create(&module);
  if (m && PyModule_AddStringConstant(m, "built_for", LO_BUILT_FOR) < 0) { // checked before the first call
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
