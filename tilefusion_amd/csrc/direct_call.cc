// Python module tilefusion_amd._direct: the ops called without the work that the dispatcher does for any op from Python.
//
// A call of torch.ops.tilefusion.* from Python costs ~2 us beside the launch (matching the arguments to the schema,
// boxing them, three dispatch keys under which nothing is done), as much as the launch of a small kernel.  The functions
// here take a call only where the dispatcher would do nothing but call what is registered for the CUDA key: plain
// device tensors, no gradient asked for, nothing that watches or rewrites ops (see `plain`).  Otherwise they
// return False (None), having done nothing, and the wrapper in tilefusion_amd/ops goes through torch.ops, as it does for
// torch.compile and torch.jit.script.  What is called is the dispatcher's CUDA kernel of the op, an implementation that a
// program registers in place of the library's included.
// us a call in a loop, through torch.ops / as here: gemm 128 x 64 x 256 4.6 / 3.7; fused 16384 x 128 x 128 x 128 4.7 / 4.4 and decoding
// 32 x 1999 x 64 9.4 / 9.4, whose kernels take as long.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/Context.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/dispatch/Dispatcher.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/record_function.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cmath>

namespace {

// Dispatch keys above CUDA that plain tensors come with: nothing is done under them where no gradient is asked for, unless a
// program registers something there (has_observer).
const c10::DispatchKeySet kPassed =
    c10::DispatchKeySet(c10::DispatchKey::AutogradCUDA) | c10::DispatchKeySet(c10::DispatchKey::ADInplaceOrView) |
    c10::DispatchKeySet(c10::DispatchKey::BackendSelect);
const c10::DispatchKeySet kCuda(c10::DispatchKey::CUDA);

// The ops of torch_bind.cc (loaded by the package before this module).
template <typename Signature>
c10::TypedOperatorHandle<Signature> find_op(const char* name) {
  return c10::Dispatcher::singleton().findSchemaOrThrow(name, "").typed<Signature>();
}
using AttentionOp = void(const at::Tensor&, const at::Tensor&, const at::Tensor&, at::Tensor&, double, bool);

// A program has registered something under the keys that are passed.
bool has_observer(const c10::OperatorHandle& op) {
  return op.hasKernelForAnyDispatchKey(kPassed) || op.hasKernelForDispatchKey(c10::DispatchKey::Autograd);
}

// Takes the tensors out of args[0 .. n); false unless every one is an ordinary torch.Tensor (no subclass) on a GPU that
// wants no gradient, and no mode, transform, autocast, tracer, profiler or observer of `op` is to see the call.
bool plain(const c10::OperatorHandle& op, PyObject* const* args, int n, at::Tensor* out) {
  c10::DispatchKeySet keys;
  for (int i = 0; i < n; ++i) {
    if (!THPVariable_CheckExact(args[i])) return false;
    const at::Tensor& t = THPVariable_Unpack(args[i]);
    if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided) return false;
    if (t.requires_grad() || t._fw_grad(0).defined()) return false;
    keys = keys | t.key_set();
    out[i] = t;   // (held while the interpreter is unlocked)
  }
  const auto local = c10::impl::tls_local_dispatch_key_set();
  keys = ((keys | local.included_) - local.excluded_) - (kPassed | kCuda);
  return keys.highestFunctionalityKey() == c10::DispatchKey::Undefined && !at::impl::torch_function_mode_enabled() &&
         !at::hasCallbacks() && !has_observer(op);
}

// ints only (a bool, a numpy number or a tensor is the dispatcher's business)
bool ints(PyObject* const* args, int n, int64_t* out) {
  for (int i = 0; i < n; ++i) {
    if (!PyLong_CheckExact(args[i])) return false;
    out[i] = PyLong_AsLongLong(args[i]);
    if (out[i] == -1 && PyErr_Occurred()) {
      PyErr_Clear();
      return false;
    }
  }
  return true;
}

struct NoGil {   // as the dispatcher: other threads run while a call is prepared
  PyThreadState* state = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(state); }
};

// at::empty(shape, like.options()) for a tensor that `plain` has passed: the same allocator and tensor, without the dispatcher's way to
// them (0.3 us instead of 0.7).
at::Tensor empty_output(at::IntArrayRef shape, const at::Tensor& like) {
  const auto& context = at::globalContext();
  if (context.deterministicAlgorithms() && context.deterministicFillUninitializedMemory()) return at::empty(shape, like.options());
  return at::Tensor(at::detail::empty_cuda(shape, like.scalar_type(), like.device(), c10::nullopt));
}

// at::empty_like(like), which gives a dense tensor its strides, also the ones that address nothing (of extents of 1).
at::Tensor empty_output_like(const at::Tensor& like) {
  int64_t in_order = 1;
  for (int64_t i = like.dim() - 1; i >= 0; --i) {
    if (like.stride(i) != in_order) return at::empty_like(like);
    in_order *= like.size(i);
  }
  return empty_output(like.sizes(), like);
}

bool is_half_type(const at::Tensor& t) { return t.scalar_type() == at::kHalf || t.scalar_type() == at::kBFloat16; }

PyObject* gemm(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  at::Tensor t[3];
  int64_t i[5];
  using Op = void(const at::Tensor&, const at::Tensor&, at::Tensor&, int64_t, int64_t, int64_t, int64_t, int64_t);
  static const auto op = find_op<Op>("tilefusion::gemm");
  if (nargs != 8 || !plain(op, args, 3, t) || !ints(args + 3, 5, i)) Py_RETURN_FALSE;
  {
    NoGil unlocked;
    op.redispatch(kCuda, t[0], t[1], t[2], i[0], i[1], i[2], i[3], i[4]);
  }
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

PyObject* fused_two_gemms(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  at::Tensor t[4];
  int64_t i[4];
  using Op = void(const at::Tensor&, const at::Tensor&, const at::Tensor&, at::Tensor&, int64_t, int64_t, int64_t, int64_t);
  static const auto op = find_op<Op>("tilefusion::fused_two_gemms");
  if (nargs != 8 || !plain(op, args, 4, t) || !ints(args + 4, 4, i)) Py_RETURN_FALSE;
  for (const at::Tensor& x : t)   // (other types: the wrapper's own errors)
    if (!is_half_type(x) || x.scalar_type() != t[0].scalar_type()) Py_RETURN_FALSE;
  {
    NoGil unlocked;
    op.redispatch(kCuda, t[0], t[1], t[2], t[3], i[0], i[1], i[2], i[3]);
  }
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

PyObject* scatter_nd(PyObject*, PyObject* const* args, Py_ssize_t nargs) {   // data, updates, indices
  HANDLE_TH_ERRORS
  at::Tensor t[3];
  static const auto op = find_op<void(const at::Tensor&, at::Tensor&, const at::Tensor&)>("tilefusion::scatter_nd");
  if (nargs != 3 || !plain(op, args, 3, t)) Py_RETURN_FALSE;
  {
    NoGil unlocked;
    op.redispatch(kCuda, t[0], t[1], t[2]);
  }
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

// (query, key [.., D, Lkv], value, tile_length_q, tile_length_kv, tile_hidden_qk, tile_hidden_v, softmax_scale, causal)
// -> output, or None
PyObject* flash_attention(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  at::Tensor t[3];
  int64_t tile[4];
  static const auto op = find_op<AttentionOp>("tilefusion::flash_attention_fwd");
  static const auto op_kt = find_op<AttentionOp>("tilefusion::flash_attention_fwd_kt");
  if (nargs != 9 || !plain(op, args, 3, t) || has_observer(op_kt) || !ints(args + 3, 4, tile) || !PyFloat_CheckExact(args[7]) ||
      !PyBool_Check(args[8]))
    Py_RETURN_NONE;
  const at::Tensor &q = t[0], &k = t[1], &v = t[2];
  if (q.dim() < 2 || k.dim() < 2 || v.dim() < 2) Py_RETURN_NONE;
  const int64_t extent[4] = {q.size(-2), v.size(-2), q.size(-1), v.size(-1)};
  for (int i = 0; i < 4; ++i)
    if (tile[i] <= 0 || extent[i] % tile[i] != 0) Py_RETURN_NONE;
  const double scale = PyFloat_AS_DOUBLE(args[7]);
  const bool causal = args[8] == Py_True;
  at::Tensor out;
  {
    NoGil unlocked;
    at::DimVector shape(q.sizes());
    shape.back() = v.size(-1);
    out = empty_output(shape, q);
    // (a [D, Lkv] matrix in order is no [Lkv, D] one in order, unless one of the two is 1, or there is nothing in it)
    const bool kt = k.is_contiguous() && k.size(-1) > 1 && k.size(-2) > 1 && k.numel() > 0;
    if (kt)
      op_kt.redispatch(kCuda, q.contiguous(), k, v.contiguous(), out, scale, causal);
    else
      op.redispatch(kCuda, q.contiguous(), k.transpose(-1, -2).contiguous(), v.contiguous(), out, scale, causal);
  }
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

// (query, key, value, num_splits, softmax_scale or None) -> output, or None
PyObject* flash_decode(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  at::Tensor t[3];
  int64_t num_splits;
  using Op = void(const at::Tensor&, const at::Tensor&, const at::Tensor&, at::Tensor&, int64_t, double);
  static const auto op = find_op<Op>("tilefusion::flash_decode");
  if (nargs != 5 || !plain(op, args, 3, t) || !ints(args + 3, 1, &num_splits)) Py_RETURN_NONE;
  if (args[4] != Py_None && !PyFloat_CheckExact(args[4])) Py_RETURN_NONE;
  const at::Tensor &q = t[0], &k = t[1], &v = t[2];
  if (q.dim() < 1 || q.size(-1) < 1) Py_RETURN_NONE;
  const double scale = args[4] == Py_None ? 1.0 / std::sqrt((double)q.size(-1)) : PyFloat_AS_DOUBLE(args[4]);
  at::Tensor out;
  {
    NoGil unlocked;
    out = empty_output_like(q);
    op.redispatch(kCuda, q.contiguous(), k.contiguous(), v.contiguous(), out, num_splits, scale);
  }
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

template <PyObject* (*kFunction)(PyObject*, PyObject* const*, Py_ssize_t)>
constexpr PyMethodDef method(const char* name) {
  return {name, (PyCFunction)(void (*)(void))kFunction, METH_FASTCALL, nullptr};
}
PyMethodDef methods[] = {method<gemm>("gemm"), method<fused_two_gemms>("fused_two_gemms"), method<scatter_nd>("scatter_nd"),
                         method<flash_attention>("flash_attention"), method<flash_decode>("flash_decode"),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_direct", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__direct() { return PyModule_Create(&module); }
