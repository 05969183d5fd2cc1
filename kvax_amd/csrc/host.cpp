// Host side of the calls in native code: what a call of create_attention_mask, of the attention forward and of its
// backward does between Python and the C ABI - look at the tensors, allocate outputs and workspace, fill in the
// argument structure, launch - as one C++ function each, without the interpreter and ctypes.
//
// These functions take the plain case only: strided tensors of the current GPU whose types, shapes and layouts need no
// conversion and no error message, and no Python rule (of a tensor subclass or a mode) that has to see the torch calls.  For anything else they return None, before they have done anything, and the caller
// goes on with the Python code of the same name, which converts or raises.  The library's functions are
// handed in as addresses (bind), so that this module serves whichever library the package has loaded.
//
// What it is worth, us a pass with the interpreter and ctypes -> now: three masks of a packed 32k batch 22.9 -> 14.6, mask
// and forward of a decoding token 45.3 -> 23.2, of a prompt of 777 tokens 49.6 -> 28.9, forward and backward of a 2k row of
// 8 heads 170 -> 110.  What is left of the decoding token's: three kernel launches (10 us), torch's autograd.Function (4),
// the context manager of the specs and the checks in Python (6), four allocations.
#include <Python.h>

#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>

#include <cstring>

#include "kvax_amd.h"

namespace {

struct Library {
  decltype(&kvax_fa_fwd_workspace_bytes) fwd_bytes;
  decltype(&kvax_fa_fwd) fwd;
  decltype(&kvax_fa_bwd_workspace_bytes) bwd_bytes;
  decltype(&kvax_fa_bwd) bwd;
  decltype(&kvax_mask_workspace_bytes) mask_bytes;
  decltype(&kvax_mask_build) mask_build;
} lib{};

// Releases the interpreter lock for the launches, as ctypes does.
struct WithoutGil {
  PyThreadState* state = PyEval_SaveThread();
  ~WithoutGil() { PyEval_RestoreThread(state); }
};

// The type of the mode behind torch.set_default_device(), looked up in bind(): an import may hand the interpreter lock to
// another thread, which must not then wait here for the import to end.
PyObject* device_context;

// Whether a mode that overrides torch functions is active (TorchFunctionMode): it has to see the allocations of a call.
// The one behind torch.set_default_device() and `with torch.device(...)` is passed over: it changes calls that name no
// device, and those of the Python code name theirs.
bool functions_overridden() {
  if (!at::impl::torch_function_mode_enabled()) return false;
  for (int64_t i = 0; i < at::impl::PythonTorchFunctionTLS::stack_len(); i++) {
    const auto& mode = at::impl::PythonTorchFunctionTLS::get_stack_at(i);
    if ((PyObject*)Py_TYPE(mode->ptr(&mode->pyinterpreter())) != device_context) return true;
  }
  return false;
}

// An ordinary tensor in the memory of GPU `device`: a torch.Tensor or a Parameter and no other subclass, not a wrapper, a
// view with pending conjugation or negation, or one that a transform or a Python dispatch rule stands in front of.
const at::Tensor* plain(PyObject* o, int device) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  constexpr c10::DispatchKeySet special({c10::DispatchKey::Python, c10::DispatchKey::Conjugate, c10::DispatchKey::Negative,
                                         c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                         c10::DispatchKey::Functionalize, c10::DispatchKey::Batched});
  if (!t.defined() || !t.is_cuda() || t.device().index() != device || t.layout() != at::kStrided || t.key_set().has_any(special)) return nullptr;
  return &t;
}

// int32, contiguous, [batch, length]
const at::Tensor* plain_ids(PyObject* o, int device, int64_t batch, int64_t length) {
  const at::Tensor* t = plain(o, device);
  return t && t->scalar_type() == at::kInt && t->dim() == 2 && t->size(0) == batch && t->size(1) == length && t->is_contiguous() ? t : nullptr;
}

bool plain_rows(const at::Tensor& t) { return t.dim() == 4 && t.stride(3) == 1; }

// The four arrays of a mask with [batch, shards, blocks] entries (no shards, and longer rows of a single one, are
// allowed as in _check_mask).
bool plain_mask(PyObject* mask, int device, int64_t batch, int64_t shards, int64_t length, int64_t block, const int32_t* out[4]) {
  if (!PyTuple_Check(mask) || PyTuple_GET_SIZE(mask) != 4 || block <= 0 || batch <= 0 || length <= 0) return false;
  const int64_t rows = batch * shards, blocks = (length + block - 1) / block;
  for (int i = 0; i < 4; i++) {
    const at::Tensor* t = plain(PyTuple_GET_ITEM(mask, i), device);
    if (!t || t->scalar_type() != at::kInt || !t->is_contiguous()) return false;
    const bool fits = shards > 1 ? t->dim() == 3 && t->size(0) == batch && t->size(1) == shards && t->size(2) == blocks
                                 : t->numel() == rows * blocks || (rows == 1 && t->numel() > blocks);
    if (!fits) return false;
    out[i] = static_cast<const int32_t*>(t->data_ptr());
  }
  return true;
}

void strides3(const at::Tensor& t, int64_t out[3]) {
  for (int i = 0; i < 3; i++) out[i] = t.stride(i);
}

// What forward and backward have in common; false: not the plain case.
struct Inputs {
  const at::Tensor *q, *k, *v;
  kvax_fa_args a{};
  bool read(PyObject* const* o, int device, double scale, const int64_t blocks[4]) {
    q = plain(o[0], device), k = plain(o[1], device), v = plain(o[2], device);
    if (!q || !k || !v || !plain_rows(*q) || !plain_rows(*k) || !plain_rows(*v)) return false;
    const auto type = q->scalar_type();
    if ((type != at::kBFloat16 && type != at::kHalf) || k->scalar_type() != type || v->scalar_type() != type) return false;
    const int64_t b = q->size(0), sq = q->size(1), hq = q->size(2), d = q->size(3), sk = k->size(1), hkv = k->size(2);
    if (k->size(0) != b || k->size(3) != d || v->size(0) != b || v->size(1) != sk || v->size(2) != hkv) return false;
    if (b <= 0 || sq <= 0 || sk <= 0 || hq <= 0 || hkv <= 0 || hq % hkv) return false;
    if ((b | sq | sk | hq | d) >> 31 || v->size(3) <= 0 || v->size(3) > INT16_MAX) return false;
    const at::Tensor* ids[4];
    for (int i = 0; i < 4; i++) {
      ids[i] = plain_ids(o[3 + i], device, b, i < 2 ? sq : sk);
      if (!ids[i]) return false;
    }
    a.q = q->data_ptr(), a.k = k->data_ptr(), a.v = v->data_ptr();
    a.q_pos = (const int32_t*)ids[0]->data_ptr(), a.q_seg = (const int32_t*)ids[1]->data_ptr();
    a.kv_pos = (const int32_t*)ids[2]->data_ptr(), a.kv_seg = (const int32_t*)ids[3]->data_ptr();
    strides3(*q, a.q_strides), strides3(*k, a.k_strides), strides3(*v, a.v_strides);
    a.batch = (int32_t)b, a.q_len = (int32_t)sq, a.kv_len = (int32_t)sk;
    a.num_heads = (int32_t)hq, a.num_kv_heads = (int32_t)hkv, a.head_dim = (int32_t)d, a.v_head_dim = (int16_t)v->size(3);
    a.fwd_query_block = (int32_t)blocks[0], a.fwd_kv_block = (int32_t)blocks[1];
    a.bwd_query_block = (int32_t)blocks[2], a.bwd_kv_block = (int32_t)blocks[3];
    a.dtype = type == at::kBFloat16 ? KVAX_BF16 : KVAX_F16;
    a.scale = (float)scale;
    return true;
  }
};

at::Tensor workspace(size_t bytes, const at::Tensor& like) {
  return at::empty({(int64_t)std::max<size_t>(bytes, 16)}, like.options().dtype(at::kByte));
}

bool integers(PyObject* const* o, int n, int64_t* out) {
  for (int i = 0; i < n; i++) {
    if (!PyLong_Check(o[i])) return false;
    out[i] = PyLong_AsLongLong(o[i]);
    if (out[i] == -1 && PyErr_Occurred()) {
      PyErr_Clear();
      return false;
    }
    if (out[i] < INT32_MIN || out[i] > INT32_MAX) return false;
  }
  return true;
}

bool stream_handle(PyObject* o, void** out) {
  *out = PyLong_AsVoidPtr(o);
  if (!*out && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}

// bind(ABI version, bytes of kvax_fa_args, bytes of kvax_mask_desc, torch version, 6 addresses): the functions behind the
// addresses and the tensors read here are only what this module was compiled against if the first four are.
PyObject* bind(PyObject*, PyObject* const* o, Py_ssize_t n) {
  if (n != 10) return PyErr_Format(PyExc_TypeError, "bind takes 10 arguments");
  const long version = PyLong_AsLong(o[0]), args = PyLong_AsLong(o[1]), desc = PyLong_AsLong(o[2]);
  const char* torch = PyUnicode_Check(o[3]) ? PyUnicode_AsUTF8(o[3]) : "";
  if (!torch || PyErr_Occurred()) return nullptr;
  if (version != KVAX_ABI_VERSION || args != (long)sizeof(kvax_fa_args) || desc != (long)sizeof(kvax_mask_desc))
    return PyErr_Format(PyExc_ImportError, "built for version %d of the C ABI with structures of %d and %d bytes, not %ld, %ld and %ld",
                        KVAX_ABI_VERSION, (int)sizeof(kvax_fa_args), (int)sizeof(kvax_mask_desc), version, args, desc);
  if (strcmp(torch, KVAX_TORCH_VERSION) != 0)
    return PyErr_Format(PyExc_ImportError, "built for torch " KVAX_TORCH_VERSION ", not %s", torch);
  PyObject* module = PyImport_ImportModule("torch.utils._device");
  device_context = module ? PyObject_GetAttrString(module, "DeviceContext") : nullptr;
  Py_XDECREF(module);
  PyErr_Clear();
  void* p[6];
  for (int i = 0; i < 6; i++)
    if (!(p[i] = PyLong_AsVoidPtr(o[4 + i]))) return PyErr_Occurred() ? nullptr : PyErr_Format(PyExc_ValueError, "null address");
  lib.fwd_bytes = (decltype(lib.fwd_bytes))p[0], lib.fwd = (decltype(lib.fwd))p[1];
  lib.bwd_bytes = (decltype(lib.bwd_bytes))p[2], lib.bwd = (decltype(lib.bwd))p[3];
  lib.mask_bytes = (decltype(lib.mask_bytes))p[4], lib.mask_build = (decltype(lib.mask_build))p[5];
  Py_RETURN_NONE;
}

// forward(q, k, v, q_pos, q_seg, kv_pos, kv_seg, mask, scale, 4 block sizes, device, stream) -> (out, lse, code) or None
PyObject* forward(PyObject*, PyObject* const* o, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 15) return PyErr_Format(PyExc_TypeError, "forward takes 15 arguments");
  int64_t ints[5];
  void* stream;
  Inputs in;
  if (functions_overridden() || !PyFloat_Check(o[8]) || !integers(o + 9, 5, ints) || !stream_handle(o[14], &stream)) Py_RETURN_NONE;
  if (!in.read(o, (int)ints[4], PyFloat_AS_DOUBLE(o[8]), ints)) Py_RETURN_NONE;
  kvax_fa_args& a = in.a;
  if (!plain_mask(o[7], (int)ints[4], a.batch, 1, a.q_len, a.fwd_query_block, a.fwd_mask)) Py_RETURN_NONE;
  at::Tensor out = a.v_head_dim == a.head_dim ? at::empty_like(*in.q)
                                              : at::empty({a.batch, a.q_len, a.num_heads, a.v_head_dim}, in.q->options());
  at::Tensor lse = at::empty({a.batch, a.num_heads, a.q_len}, in.q->options().dtype(at::kFloat));
  if (out.stride(3) != 1) Py_RETURN_NONE;
  a.out = out.data_ptr(), a.lse = (float*)lse.data_ptr();
  strides3(out, a.o_strides);
  const size_t bytes = lib.fwd_bytes(&a);
  at::Tensor ws = workspace(bytes, *in.q);
  int rc;
  {
    void* p = ws.data_ptr();
    WithoutGil released;
    rc = lib.fwd(&a, p, (size_t)ws.numel(), stream);
  }
  return Py_BuildValue("NNi", THPVariable_Wrap(std::move(out)), THPVariable_Wrap(std::move(lse)), rc);
  END_HANDLE_TH_ERRORS
}

// backward(q, k, v, q_pos, q_seg, kv_pos, kv_seg, dq_mask, dkdv_mask, out, lse, dout, scale, 4 block sizes, shards, device,
// stream) -> (dq, dk, dv, code) or None
PyObject* backward(PyObject*, PyObject* const* o, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 20) return PyErr_Format(PyExc_TypeError, "backward takes 20 arguments");
  int64_t ints[6];
  void* stream;
  Inputs in;
  if (functions_overridden() || !PyFloat_Check(o[12]) || !integers(o + 13, 6, ints) || !stream_handle(o[19], &stream)) Py_RETURN_NONE;
  const int64_t shards = ints[4];
  const int device = (int)ints[5];
  if (shards < 1 || shards > INT16_MAX || !in.read(o, device, PyFloat_AS_DOUBLE(o[12]), ints)) Py_RETURN_NONE;
  kvax_fa_args& a = in.a;
  const at::Tensor *out = plain(o[9], device), *lse = plain(o[10], device), *dout = plain(o[11], device);
  if (!out || !lse || !dout || !plain_rows(*out) || !plain_rows(*dout)) Py_RETURN_NONE;
  const auto shape = out->sizes();
  if (shape != at::IntArrayRef({a.batch, a.q_len, a.num_heads, a.v_head_dim}) || dout->sizes() != shape ||
      out->scalar_type() != in.q->scalar_type() || dout->scalar_type() != in.q->scalar_type() ||
      lse->scalar_type() != at::kFloat || !lse->is_contiguous())
    Py_RETURN_NONE;
  if (!plain_mask(o[7], device, a.batch, 1, a.q_len, a.bwd_kv_block, a.dq_mask) ||
      !plain_mask(o[8], device, a.batch, shards, a.kv_len, a.bwd_kv_block, a.dkdv_mask))
    Py_RETURN_NONE;
  at::Tensor dq = at::empty_like(*in.q), dk = at::empty(in.k->sizes(), in.k->options()), dv = at::empty(in.v->sizes(), in.v->options());
  if (dq.stride(3) != 1) Py_RETURN_NONE;
  a.out = out->data_ptr(), a.lse = (float*)lse->data_ptr(), a.dout = dout->data_ptr();
  a.dq = dq.data_ptr(), a.dk = dk.data_ptr(), a.dv = dv.data_ptr();
  strides3(*out, a.o_strides), strides3(*dout, a.do_strides);
  strides3(dq, a.dq_strides), strides3(dk, a.dk_strides), strides3(dv, a.dv_strides);
  a.dkdv_shards = (int16_t)shards;
  const size_t bytes = lib.bwd_bytes(&a);
  at::Tensor ws = workspace(bytes, *in.q);
  int rc;
  {
    void* p = ws.data_ptr();
    WithoutGil released;
    rc = lib.bwd(&a, p, (size_t)ws.numel(), stream);
  }
  return Py_BuildValue("NNNi", THPVariable_Wrap(std::move(dq)), THPVariable_Wrap(std::move(dk)), THPVariable_Wrap(std::move(dv)), rc);
  END_HANDLE_TH_ERRORS
}

// masks(q_pos, q_seg, kv_pos, kv_seg, requests, skip_pad, shards, device, stream) -> (code, [the arrays]) or None.  One
// allocation holds the workspace and every array, whose tensors are views of it: four per request, [batch, shards, blocks],
// masks on 16-byte boundaries.
PyObject* masks(PyObject*, PyObject* const* o, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 9) return PyErr_Format(PyExc_TypeError, "masks takes 9 arguments");
  int64_t ints[3];
  void* stream;
  if (functions_overridden() || !integers(o + 5, 3, ints) || !stream_handle(o[8], &stream) || !PyTuple_Check(o[4])) Py_RETURN_NONE;
  const int64_t skip_pad = ints[0], num_shards = ints[1];
  const int device = (int)ints[2];
  const at::Tensor *first = plain(o[0], device), *keys = plain(o[2], device);
  if (!first || !keys || first->dim() != 2 || keys->dim() != 2) Py_RETURN_NONE;
  const int64_t b = first->size(0), sq = first->size(1), sk = keys->size(1);
  if (b <= 0 || sq <= 0 || sk <= 0 || num_shards < 1 || (b | sq | sk) >> 31) Py_RETURN_NONE;
  const int32_t* ids[4];
  for (int i = 0; i < 4; i++) {
    const at::Tensor* t = plain_ids(o[i], device, b, i < 2 ? sq : sk);
    if (!t) Py_RETURN_NONE;
    ids[i] = static_cast<const int32_t*>(t->data_ptr());
  }
  const Py_ssize_t count = PyTuple_GET_SIZE(o[4]);
  if (count < 1 || count > KVAX_MAX_MASKS) Py_RETURN_NONE;
  kvax_mask_desc descs[KVAX_MAX_MASKS] = {};
  int64_t at_word[KVAX_MAX_MASKS], shape[KVAX_MAX_MASKS][2], words = 0;
  for (Py_ssize_t i = 0; i < count; i++) {
    PyObject* r = PyTuple_GET_ITEM(o[4], i);
    if (!PyTuple_Check(r) || PyTuple_GET_SIZE(r) != 3) Py_RETURN_NONE;
    int64_t v[3];
    PyObject* items[3] = {PyTuple_GET_ITEM(r, 0), PyTuple_GET_ITEM(r, 1), PyTuple_GET_ITEM(r, 2)};
    if (!integers(items, 3, v) || v[0] <= 0 || v[1] <= 0) Py_RETURN_NONE;
    const bool kv_outer = v[2] != 0;
    descs[i].query_block_size = (int32_t)v[0], descs[i].kv_block_size = (int32_t)v[1], descs[i].kv_outer = kv_outer;
    shape[i][0] = kv_outer ? num_shards : 1;
    shape[i][1] = kv_outer ? (sk + v[1] - 1) / v[1] : (sq + v[0] - 1) / v[0];
    at_word[i] = words;
    words += (4 * b * shape[i][0] * shape[i][1] + 3) / 4 * 4;
  }
  const size_t bytes = lib.mask_bytes((int)b, (int)sq, (int)sk, descs, (int)count);
  const int64_t ws_words = (int64_t)(std::max<size_t>(bytes, 16) + 15) / 16 * 4;
  at::Tensor buf = at::empty({ws_words + words}, first->options());
  int32_t* base = static_cast<int32_t*>(buf.data_ptr());
  for (Py_ssize_t i = 0; i < count; i++) {
    const int64_t entries = b * shape[i][0] * shape[i][1];
    int32_t* p = base + ws_words + at_word[i];
    descs[i].lower = p, descs[i].upper = p + entries, descs[i].lower_full = p + 2 * entries, descs[i].upper_full = p + 3 * entries;
  }
  int rc;
  {
    WithoutGil released;
    rc = lib.mask_build(ids[0], ids[1], ids[2], ids[3], (int)b, (int)sq, (int)sk, (int)num_shards, (int)skip_pad, descs, (int)count,
                        base, bytes, stream);
  }
  PyObject* list = PyTuple_New(4 * count);
  if (!list) return nullptr;
  for (Py_ssize_t i = 0; i < count; i++) {
    const int64_t entries = b * shape[i][0] * shape[i][1];
    for (int j = 0; j < 4; j++)
      PyTuple_SET_ITEM(list, 4 * i + j, THPVariable_Wrap(buf.as_strided({b, shape[i][0], shape[i][1]}, {shape[i][0] * shape[i][1], shape[i][1], 1},
                                                                        ws_words + at_word[i] + j * entries)));
  }
  return Py_BuildValue("iN", rc, list);
  END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"bind", (PyCFunction)(void*)bind, METH_FASTCALL, nullptr},
    {"forward", (PyCFunction)(void*)forward, METH_FASTCALL, nullptr},
    {"backward", (PyCFunction)(void*)backward, METH_FASTCALL, nullptr},
    {"masks", (PyCFunction)(void*)masks, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "kvax_amd._host", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__host() { return PyModule_Create(&module); }
