// One packed product from Python in one call: the checks of ops.quantized_matmul, the result's allocation and the library's entry point.  Through the interpreter (reads of shapes and
// addresses, an allocation, a foreign call of fourteen arguments) one row of 4096 x 4096 took 10.8 us, here 6.4 to 6.7, where the kernel alone takes 5.0; 27 rows of 8192 x 3072, whose
// kernel is most of the call, 11.7 -> 8.7.  Up to 255 rows, and up to 4096 where they go as groups of 32 (gbx_qlinear_groups).
// Whatever is not plain -- other layouts, types that want a cast, subclasses, transforms, modes, traces, other rows -- is answered with None: the general path then takes or refuses it.
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

namespace {

// entry points of the library that the package has loaded (_lib.py hands their addresses over)
typedef int (*ForwardFn)(const void*, const void*, const void*, const void*, const void*, void*, int64_t, int32_t, int32_t, int32_t, int32_t, int32_t, void*);
typedef int (*ForwardWsFn)(const void*, const void*, const void*, const void*, const void*, void*, int64_t, int32_t, int32_t, int32_t, int32_t, int32_t, void*, size_t, void*);
typedef size_t (*WorkspaceFn)(int64_t, int32_t, int32_t, int32_t, int32_t);
ForwardFn forward_fn = nullptr;
ForwardWsFn forward_ws_fn = nullptr;
WorkspaceFn workspace_fn = nullptr;
typedef int (*GroupsFn)(const void*, const void*, const void*, const void*, const void*, void*, int64_t, int32_t, int32_t, int32_t, int32_t, int32_t, int32_t, void*);
GroupsFn groups_fn = nullptr;
typedef int (*GroupsWinFn)(int64_t, int32_t, int32_t, int32_t, int32_t);
GroupsWinFn groups_win_fn = nullptr;

// From the first on a resident image of the weight goes before groups of 32, from the second on these do wherever they win; what they do not take is decided in ops.py.
constexpr int64_t FEW_ROWS = 256, MANY_ROWS = 1024;
constexpr int F16 = 0, BF16 = 1;

bool plain(const at::Tensor& t, at::Device device) {
  static const uint64_t usual = (c10::DispatchKeySet(c10::DispatchKey::CUDA) | c10::DispatchKeySet(c10::DispatchKey::AutogradCUDA) |
                                 c10::DispatchKeySet(c10::DispatchKey::ADInplaceOrView) | c10::DispatchKeySet(c10::DispatchKey::AutocastCUDA)).raw_repr();
  return (t.key_set().raw_repr() & ~usual) == 0 && t.device() == device && t.is_contiguous() && t.has_storage();
}

bool watched() {                            // something is to see every operation
  return c10::impl::dispatch_mode_enabled() || c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) ||
         c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::Tracer);
}

// A launch waits where the queue is full: other threads run meanwhile, as they do during a foreign call.
struct WithoutLock {
  PyThreadState* state = PyEval_SaveThread();
  ~WithoutLock() { PyEval_RestoreThread(state); }
};

PyObject* bind(PyObject*, PyObject* args) {
  unsigned long long f, w, s, g, gw;
  if (!PyArg_ParseTuple(args, "KKKKK", &f, &w, &s, &g, &gw)) return nullptr;
  forward_fn = reinterpret_cast<ForwardFn>(static_cast<uintptr_t>(f));
  forward_ws_fn = reinterpret_cast<ForwardWsFn>(static_cast<uintptr_t>(w));
  workspace_fn = reinterpret_cast<WorkspaceFn>(static_cast<uintptr_t>(s));
  groups_fn = reinterpret_cast<GroupsFn>(static_cast<uintptr_t>(g));
  groups_win_fn = reinterpret_cast<GroupsWinFn>(static_cast<uintptr_t>(gw));
  Py_RETURN_NONE;
}

// few_rows(x, qweight, scales, zeros, group_size, bits, bias or None[, whether 256 to 1023 rows may go as groups of 32]) -> y, None (not a call for this path) or the library's error code
PyObject* few_rows(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  if ((n_args != 7 && n_args != 8) || !forward_fn) Py_RETURN_NONE;
  for (int i = 0; i < 4; ++i)
    if (!THPVariable_CheckExact(args[i])) Py_RETURN_NONE;
  const bool has_bias = args[6] != Py_None;
  if ((has_bias && !THPVariable_CheckExact(args[6])) || !PyLong_CheckExact(args[4]) || !PyLong_CheckExact(args[5]) || watched()) Py_RETURN_NONE;
  const at::Tensor &x = THPVariable_Unpack(args[0]), &w = THPVariable_Unpack(args[1]), &sc = THPVariable_Unpack(args[2]), &ze = THPVariable_Unpack(args[3]);
  const auto type = x.scalar_type();
  if (!x.is_cuda() || (type != at::kBFloat16 && type != at::kHalf) || (w.scalar_type() != at::kInt && w.scalar_type() != at::ScalarType::UInt32) || sc.scalar_type() != type ||
      ze.scalar_type() != type)
    Py_RETURN_NONE;
  const at::Device device = x.device();
  if (!plain(x, device) || !plain(w, device) || !plain(sc, device) || !plain(ze, device)) Py_RETURN_NONE;
  const int64_t group = PyLong_AsLongLong(args[4]), bits = PyLong_AsLongLong(args[5]);
  if (x.dim() < 1 || w.dim() != 2 || sc.dim() != 2 || ze.dim() != 2 || group < 1 || bits < 1 || group > 1024 || bits > 32) Py_RETURN_NONE;
  const int64_t n = w.size(0), words = w.size(1);
  if (words * 32 % bits) Py_RETURN_NONE;
  const int64_t k = words * 32 / bits;
  if (k < 1 || n < 1 || k > 0x7fffffff || n > 0x7fffffff || x.size(-1) != k || k % group || sc.size(0) != n || sc.size(1) != k / group || ze.size(0) != n || ze.size(1) != k / group)
    Py_RETURN_NONE;
  const int64_t m = x.numel() / k;
  // rows of several sequences keep the order of sums that they had (see quantized_matmul in ops.py)
  const bool grouped = m > 32 && !(x.dim() == 3 && x.size(0) > 1) && groups_win_fn(m, static_cast<int32_t>(n), static_cast<int32_t>(k), static_cast<int32_t>(bits), static_cast<int32_t>(group));
  if (m < 1 || (m >= FEW_ROWS && (!grouped || (m < MANY_ROWS && (n_args < 8 || args[7] != Py_True))))) Py_RETURN_NONE;
  const void* bias = nullptr;
  if (has_bias) {
    const at::Tensor& b = THPVariable_Unpack(args[6]);
    if (b.scalar_type() != type || b.dim() != 1 || b.size(0) != n || !plain(b, device)) Py_RETURN_NONE;
    bias = b.const_data_ptr();
  }
  auto shape = x.sizes().vec();
  shape.back() = n;
  at::Tensor y = at::empty(shape, x.options().requires_grad(false));
  if (!plain(y, device)) Py_RETURN_NONE;
  void* stream = c10::hip::getCurrentHIPStream(device.index()).stream();
  const int act = type == at::kBFloat16 ? BF16 : F16;
  const int32_t N = static_cast<int32_t>(n), K = static_cast<int32_t>(k), B = static_cast<int32_t>(bits), G = static_cast<int32_t>(group);
  const void *px = x.const_data_ptr(), *pw = w.const_data_ptr(), *ps = sc.const_data_ptr(), *pz = ze.const_data_ptr();
  void* py = y.mutable_data_ptr();
  int rc;
  if (grouped) {
    {
      WithoutLock free;
      rc = groups_fn(px, pw, ps, pz, bias, py, m, N, K, B, G, act, 0, stream);
    }
    if (rc == 0) return THPVariable_Wrap(std::move(y));
    if (rc != 1) return PyLong_FromLong(rc);
    if (m >= FEW_ROWS) Py_RETURN_NONE;
  }
  // scratch: decode batches and short prompts split k across workgroups
  const size_t need = (m >= 2 && m <= 32) || m > 64 ? workspace_fn(m, N, K, B, G) : 0;
  if (need) {
    at::Tensor ws = at::empty({static_cast<int64_t>(need)}, x.options().dtype(at::kByte).requires_grad(false));
    void* pws = ws.mutable_data_ptr();
    WithoutLock free;
    rc = forward_ws_fn(px, pw, ps, pz, bias, py, m, N, K, B, G, act, pws, need, stream);
  } else {
    WithoutLock free;
    rc = forward_fn(px, pw, ps, pz, bias, py, m, N, K, B, G, act, stream);
  }
  if (rc) return PyLong_FromLong(rc);
  return THPVariable_Wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {{"bind", bind, METH_VARARGS, nullptr},
                         {"few_rows", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(few_rows)), METH_FASTCALL, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_gbx_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__gbx_host(void) { return PyModule_Create(&module); }
