// The host side of one attention call as native code: what dense_attention and the cache manager's step() do per call
// between Python and lbm_attn_run_call - looking at the tensors, allocating the result, finding the stream, filling the
// record.  In Python that is two dozen attribute reads and calls, 3.8 us of a dense_attention call whose launch takes the
// HIP runtime 2.4 us and the GPU 5.1 (261 tokens, 16 heads).  Nothing is kept between calls.  A call that these functions
// do not recognise - tensors of a subclass, on the CPU, of other shapes, strides or types - is for Python's general way,
// which converts it or raises.
#include <Python.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/ops/empty_like.h>
#include <c10/hip/HIPStream.h>
#include <cstring>
#include "../../include/lbm_paged_attn.h"

namespace {

// a plain CUDA tensor [tokens, heads, head_dim], contiguous, bf16 or fp32
const at::Tensor* rows_of(PyObject* obj) {
  if (!THPVariable_CheckExact(obj)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(obj);
  if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || t.dim() != 3 || !t.is_contiguous()) return nullptr;
  if (t.scalar_type() != at::kBFloat16 && t.scalar_type() != at::kFloat) return nullptr;
  return &t;
}
bool alike(const at::Tensor& a, const at::Tensor& b) {
  return a.sizes() == b.sizes() && a.scalar_type() == b.scalar_type() && a.device() == b.device();
}
bool three(PyObject* const* args, const at::Tensor* (&t)[3]) {
  for (int i = 0; i < 3; ++i)
    if (!(t[i] = rows_of(args[i])) || !alike(*t[0], *t[i])) return false;
  return true;
}

// frames_key(q, k, v, num_streams): what a dense_attention call's plan goes by - (tokens, heads, head_dim, num_streams,
// fp32, device index) - or None
PyObject* frames_key(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  const at::Tensor* t[3];
  if (n != 4 || !PyLong_CheckExact(args[3]) || !three(args, t)) Py_RETURN_NONE;
  const long long streams = PyLong_AsLongLong(args[3]);
  if (streams == -1 && PyErr_Occurred()) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  const int64_t rows = t[0]->size(0);
  if (streams < 1 || streams > LBM_MAX_STREAMS || rows <= 0 || rows % streams) Py_RETURN_NONE;
  return Py_BuildValue("(LLLLii)", (long long)rows, (long long)t[0]->size(1), (long long)t[0]->size(2), streams,
                       (int)(t[0]->scalar_type() == at::kFloat), (int)t[0]->get_device());
  END_HANDLE_TH_ERRORS
}

// rows_fit(q, k, v, tokens, heads, head_dim, fp32): whether a cache's call may take all three as they are
PyObject* rows_fit(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  const at::Tensor* t[3];
  if (n != 7 || !three(args, t)) Py_RETURN_FALSE;
  for (int i = 0; i < 3; ++i)
    if (t[0]->size(i) != PyLong_AsLongLong(args[3 + i])) Py_RETURN_FALSE;
  if ((t[0]->scalar_type() == at::kFloat) != (args[6] == Py_True)) Py_RETURN_FALSE;
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

// attend(q, k, v, pool, kv_rows, live_kv_tokens, append_rows, streams, workspace, sm_scale, tail): lbm_attn_run_call on
// the current stream.  q, k, v as frames_key or rows_fit has accepted them; pool and workspace tensors; the four addresses
// as integers; tail: the record's fields from append_tokens on (attn_call_tail).  Returns the result, or the error code.
PyObject* attend(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  const at::Tensor* t[3];
  constexpr size_t kTail = sizeof(lbm_attn_call) - offsetof(lbm_attn_call, append_tokens);
  static_assert(kTail == 7 * sizeof(int32_t), "attn_call_tail packs the fields from append_tokens on");
  if (n != 11 || !three(args, t) || !THPVariable_Check(args[3]) || !THPVariable_Check(args[8]) || !PyBytes_CheckExact(args[10]) ||
      PyBytes_GET_SIZE(args[10]) != (Py_ssize_t)kTail) {
    PyErr_SetString(PyExc_TypeError, "attend: tensors q, k, v alike, pool, four addresses, workspace, scale, tail");
    return nullptr;
  }
  const at::Tensor& ws = THPVariable_Unpack(args[8]);
  lbm_attn_call c = {};
  c.q = t[0]->const_data_ptr();
  c.self_k = t[1]->const_data_ptr();
  c.self_v = t[2]->const_data_ptr();
  c.pool = THPVariable_Unpack(args[3]).data_ptr();
  c.kv_rows = (const int32_t*)PyLong_AsVoidPtr(args[4]);
  c.live_kv_tokens = (const int32_t*)PyLong_AsVoidPtr(args[5]);
  c.append_rows = (const int32_t*)PyLong_AsVoidPtr(args[6]);
  c.streams = (const lbm_attn_stream*)PyLong_AsVoidPtr(args[7]);
  c.workspace = ws.data_ptr();
  c.workspace_bytes = (size_t)ws.nbytes();
  c.sm_scale = (float)PyFloat_AsDouble(args[9]);
  std::memcpy(&c.append_tokens, PyBytes_AS_STRING(args[10]), kTail);
  if (PyErr_Occurred()) return nullptr;
  at::Tensor out = at::empty_like(*t[0]);
  c.out = out.data_ptr();
  void* const stream = (void*)c10::hip::getCurrentHIPStream(t[0]->get_device()).stream();
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = lbm_attn_run_call(&c, stream);
  Py_END_ALLOW_THREADS
  if (rc != LBM_OK) return PyLong_FromLong(rc);
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

PyMethodDef kMethods[] = {
    {"frames_key", (PyCFunction)(void*)frames_key, METH_FASTCALL, nullptr},
    {"rows_fit", (PyCFunction)(void*)rows_fit, METH_FASTCALL, nullptr},
    {"attend", (PyCFunction)(void*)attend, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "lbm_host", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_lbm_host() {
  PyObject* module = PyModule_Create(&kModule);
  // (the layout of lbm_attn_call that attend fills in)
  if (module && PyModule_AddIntConstant(module, "ABI_VERSION", LBM_ABI_VERSION) != 0) Py_CLEAR(module);
  return module;
}
