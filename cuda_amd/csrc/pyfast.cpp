// Python calls of the plain case, in one native step: the extension module
// cuda_amd._native.
//
// Each function takes the arguments of the api.py entry point of its name. When
// they are what a program normally passes - CUDA tensors of the exact type,
// contiguous and 16-byte aligned, of matching shapes and types - it allocates
// the outputs and the workspace, makes the C ABI call (include/cuda_llm_abi.h)
// on the current stream and returns the result. In every other case, errors
// included, it returns None and has done nothing: api.py then goes through its
// own checks, copies and messages. Small calls are bound by the host: a prefill
// call's checks, allocations and ctypes conversions took about 9 us in Python,
// an append with a paged decode 26.
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <climits>
#include <cmath>
#include <cstdint>
#include <cstdlib>
#include <cstring>

#include "../../include/cuda_llm_abi.h"

namespace {

// The library's functions, bound by address from the handle that api.py uses.
struct Abi {
  decltype(&ca_flash_attention_fwd) flash_attention_fwd;
  decltype(&ca_flash_attention_fwd_lse) flash_attention_fwd_lse;
  decltype(&ca_flash_attention_bwd) flash_attention_bwd;
  decltype(&ca_flash_attention_bwd_workspace_bytes) flash_attention_bwd_workspace_bytes;
  decltype(&ca_fused_rope_flash_attention) fused_rope_flash_attention;
  decltype(&ca_rope_workspace_bytes) rope_workspace_bytes;
  decltype(&ca_flash_decode) flash_decode;
  decltype(&ca_flash_decode_workspace_bytes) flash_decode_workspace_bytes;
  decltype(&ca_paged_attention) paged_attention;
  decltype(&ca_fp8_paged_attention) fp8_paged_attention;
  decltype(&ca_paged_decode_workspace_bytes) paged_decode_workspace_bytes;
  decltype(&ca_paged_kv_append) paged_kv_append;
  decltype(&ca_fused_microscaled_attention) fused_microscaled_attention;
  decltype(&ca_mx_workspace_bytes) mx_workspace_bytes;
} abi;

bool type_code(at::ScalarType t, ca_dtype* out) {
  if (t == at::kBFloat16) *out = CA_BF16;
  else if (t == at::kHalf) *out = CA_F16;
  else if (t == at::kFloat) *out = CA_F32;
  else return false;
  return true;
}
bool is_codes(at::ScalarType t) { return t == at::kByte || t == at::kChar || t == at::kFloat8_e4m3fn; }

// A tensor the kernels can take as it is: the class itself (no subclass, no
// functorch wrapper), strided storage on a GPU, contiguous, and the data
// pointer a multiple of `align`.
const at::Tensor* plain(PyObject* o, int dim, size_t align = 16) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  static const c10::DispatchKeySet wrapped(
      {c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize,
       c10::DispatchKey::Python, c10::DispatchKey::Negative, c10::DispatchKey::ZeroTensor});
  if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || t.key_set().has_any(wrapped) || !t.has_storage() ||
      !t.is_contiguous() || (dim >= 0 && t.dim() != dim))
    return nullptr;
  if (reinterpret_cast<uintptr_t>(t.const_data_ptr()) % align) return nullptr;
  return &t;
}
int n(const at::Tensor& t, int i) { return (int)t.size(i); }
bool fits(const at::Tensor& t) {  // sizes that the ABI's ints hold
  for (const auto s : t.sizes())
    if (s > INT_MAX) return false;
  return true;
}
const void* in(const at::Tensor& t) { return t.const_data_ptr(); }
void* out(const at::Tensor& t) { return t.mutable_data_ptr(); }

// softmax_scale: None is 1 / sqrt(head_dim)
bool scale_of(PyObject* o, int d, float* scale) {
  if (o == Py_None) *scale = (float)(1.0 / std::sqrt((double)d));
  else if (PyFloat_CheckExact(o)) *scale = (float)PyFloat_AS_DOUBLE(o);
  else return false;
  return true;
}
bool flag_of(PyObject* o, int* flag) {
  if (!PyBool_Check(o)) return false;
  *flag = o == Py_True;
  return true;
}
// a debug check asked for in the environment is the general path's
bool debug_asked(const char* name) {
  const char* v = std::getenv(name);
  return v && *v && !(v[0] == '0' && !v[1]);
}

at::Tensor like(const at::Tensor& t) { return at::empty(t.sizes(), t.options().requires_grad(false)); }
struct Workspace {
  at::Tensor t;
  size_t bytes;
  Workspace(size_t n, const at::Tensor& like) : bytes(n) {
    if (n) t = at::empty({(int64_t)n}, like.options().dtype(at::kByte).requires_grad(false));
  }
  void* ptr() const { return bytes ? t.mutable_data_ptr() : nullptr; }
};
void* stream() { return c10::hip::getCurrentHIPStream().stream(); }

// The ABI call without the interpreter lock, as ctypes makes it.
template <typename F>
bool ok(F f) {
  struct Unlocked {
    PyThreadState* state = PyEval_SaveThread();
    ~Unlocked() { PyEval_RestoreThread(state); }
  } unlocked;
  return f() == CA_OK;
}

bool prefill_args(PyObject* const* a, const at::Tensor*& q, const at::Tensor*& k, const at::Tensor*& v, ca_dtype* dt) {
  if (!(q = plain(a[0], 4)) || !(k = plain(a[1], 4)) || !(v = plain(a[2], 4))) return false;
  const auto d = q->size(3);
  return k->sizes() == v->sizes() && q->scalar_type() == k->scalar_type() && q->scalar_type() == v->scalar_type() &&
         type_code(q->scalar_type(), dt) && fits(*q) && k->size(0) == q->size(0) && k->size(2) == q->size(2) &&
         k->size(3) == d && k->size(1) >= 1 && q->size(1) % k->size(1) == 0 && (d == 64 || d == 128);
}

// (q, k, v, is_causal, softmax_scale) -> out
PyObject* flash_attention_forward(PyObject* const* a) {
  const at::Tensor *q, *k, *v;
  ca_dtype dt;
  int causal;
  float scale;
  if (!prefill_args(a, q, k, v, &dt) || !flag_of(a[3], &causal) || !scale_of(a[4], n(*q, 3), &scale)) return nullptr;
  const at::Tensor o = like(*q);
  if (!ok([&] {
        return abi.flash_attention_fwd(dt, in(*q), in(*k), in(*v), out(o), n(*q, 0), n(*q, 1), n(*k, 1), n(*q, 2),
                                       n(*q, 3), scale, causal, stream());
      }))
    return nullptr;
  return THPVariable_Wrap(o);
}

// (q, k, v, is_causal, softmax_scale) -> (out, lse)
PyObject* flash_attention_forward_lse(PyObject* const* a) {
  const at::Tensor *q, *k, *v;
  ca_dtype dt;
  int causal;
  float scale;
  if (!prefill_args(a, q, k, v, &dt) || !flag_of(a[3], &causal) || !scale_of(a[4], n(*q, 3), &scale)) return nullptr;
  const at::Tensor o = like(*q);
  const at::Tensor lse = at::empty({q->size(0), q->size(1), q->size(2)},
                                   q->options().dtype(at::kFloat).requires_grad(false));
  if (!ok([&] {
        return abi.flash_attention_fwd_lse(dt, in(*q), in(*k), in(*v), out(o), (float*)out(lse), n(*q, 0), n(*q, 1),
                                           n(*k, 1), n(*q, 2), n(*q, 3), scale, causal, stream());
      }))
    return nullptr;
  return Py_BuildValue("(NN)", THPVariable_Wrap(o), THPVariable_Wrap(lse));
}

// (dout, q, k, v, out, lse, is_causal, softmax_scale) -> [dq, dk, dv]
PyObject* flash_attention_backward(PyObject* const* a) {
  const at::Tensor *q, *k, *v, *g = plain(a[0], 4), *o = plain(a[4], 4), *lse = plain(a[5], 3, 4);
  ca_dtype dt;
  int causal;
  float scale;
  if (!g || !o || !lse || !prefill_args(a + 1, q, k, v, &dt) || !flag_of(a[6], &causal) ||
      !scale_of(a[7], n(*q, 3), &scale) || g->sizes() != q->sizes() || o->sizes() != q->sizes() ||
      g->scalar_type() != q->scalar_type() || o->scalar_type() != q->scalar_type() || lse->scalar_type() != at::kFloat ||
      lse->sizes() != q->sizes().slice(0, 3))
    return nullptr;
  const at::Tensor dq = like(*q), dk = like(*k), dv = like(*v);
  const Workspace ws(abi.flash_attention_bwd_workspace_bytes(n(*q, 0), n(*q, 1), n(*q, 2)), *q);
  if (!ok([&] {
        return abi.flash_attention_bwd(dt, in(*q), in(*k), in(*v), in(*o), in(*g), (const float*)in(*lse), out(dq),
                                       out(dk), out(dv), n(*q, 0), n(*q, 1), n(*k, 1), n(*q, 2), n(*q, 3), scale,
                                       causal, ws.ptr(), ws.bytes, stream());
      }))
    return nullptr;
  return Py_BuildValue("[NNN]", THPVariable_Wrap(dq), THPVariable_Wrap(dk), THPVariable_Wrap(dv));
}

// (q, k, v, cos_tab, sin_tab, is_causal, softmax_scale) -> out
PyObject* fused_rope_flash_attention(PyObject* const* a) {
  const at::Tensor *q, *k, *v, *cs = plain(a[3], 2), *sn = plain(a[4], 2);
  ca_dtype dt;
  int causal;
  float scale;
  if (!cs || !sn || !prefill_args(a, q, k, v, &dt) || !flag_of(a[5], &causal) || !scale_of(a[6], n(*q, 3), &scale) ||
      cs->scalar_type() != at::kFloat || sn->scalar_type() != at::kFloat || cs->sizes() != q->sizes().slice(2, 2) ||
      sn->sizes() != cs->sizes())
    return nullptr;
  const at::Tensor o = like(*q);
  const Workspace ws(abi.rope_workspace_bytes(dt, n(*q, 0), n(*q, 1), n(*k, 1), n(*q, 2), n(*q, 3)), *q);
  if (!ok([&] {
        return abi.fused_rope_flash_attention(dt, in(*q), in(*k), in(*v), (const float*)in(*cs), (const float*)in(*sn),
                                              out(o), n(*q, 0), n(*q, 1), n(*k, 1), n(*q, 2), n(*q, 3), scale, causal,
                                              ws.ptr(), ws.bytes, stream());
      }))
    return nullptr;
  return THPVariable_Wrap(o);
}

// (q, k, v, softmax_scale) -> out
PyObject* async_flash_decode(PyObject* const* a) {
  const at::Tensor *q = plain(a[0], 4), *k = plain(a[1], 4), *v = plain(a[2], 4);
  ca_dtype dt;
  float scale;
  if (!q || !k || !v || q->size(2) != 1 || k->sizes() != v->sizes() || q->scalar_type() != k->scalar_type() ||
      q->scalar_type() != v->scalar_type() || !type_code(q->scalar_type(), &dt) || !fits(*q) || !fits(*k) ||
      k->size(0) != q->size(0) || k->size(3) != q->size(3) || k->size(1) < 1 || q->size(1) % k->size(1) ||
      (q->size(3) != 64 && q->size(3) != 128) || !scale_of(a[3], n(*q, 3), &scale))
    return nullptr;
  const at::Tensor o = like(*q);
  const Workspace ws(abi.flash_decode_workspace_bytes(dt, n(*q, 0), n(*q, 1), n(*k, 1), n(*k, 2), n(*q, 3)), *q);
  if (!ok([&] {
        return abi.flash_decode(dt, in(*q), in(*k), in(*v), out(o), n(*q, 0), n(*q, 1), n(*k, 1), n(*k, 2), n(*q, 3),
                                scale, ws.ptr(), ws.bytes, stream());
      }))
    return nullptr;
  return THPVariable_Wrap(o);
}

// block tables and lengths of a paged call over `seqs` sequences
bool tables_of(PyObject* bt, PyObject* cl, int64_t seqs, const at::Tensor*& tables, const at::Tensor*& lens) {
  tables = plain(bt, 2, 4);
  lens = plain(cl, 1, 4);
  return tables && lens && tables->scalar_type() == at::kInt && lens->scalar_type() == at::kInt &&
         tables->size(0) == seqs && lens->size(0) == seqs && tables->size(1) <= INT_MAX / 16;
}
bool caches_of(PyObject* ko, PyObject* vo, const at::Tensor& q, const at::Tensor*& kc, const at::Tensor*& vc) {
  kc = plain(ko, 4);
  vc = plain(vo, 4);
  const auto d = q.size(2);
  return kc && vc && kc->sizes() == vc->sizes() && fits(*kc) && fits(q) && (d == 64 || d == 128) && kc->size(2) == d &&
         kc->size(3) == 16 && kc->size(1) >= 1 && q.size(1) % kc->size(1) == 0;
}
// fp32 scales per head or per (page, head)
bool scales_of(PyObject* ko, PyObject* vo, const at::Tensor& kc, const at::Tensor*& ks, const at::Tensor*& vs) {
  ks = plain(ko, -1, 4);
  vs = plain(vo, -1, 4);
  if (!ks || !vs || ks->scalar_type() != at::kFloat || vs->scalar_type() != at::kFloat || ks->sizes() != vs->sizes())
    return false;
  return ks->dim() == 2 ? ks->sizes() == kc.sizes().slice(0, 2) : ks->dim() == 1 && ks->size(0) == kc.size(1);
}

// (query, key_cache, value_cache, block_tables, context_lens, softmax_scale) -> out
PyObject* paged_attention_forward(PyObject* const* a) {
  const at::Tensor *q = plain(a[0], 3), *kc, *vc, *bt, *cl;
  ca_dtype dt;
  float scale;
  if (!q || !caches_of(a[1], a[2], *q, kc, vc) || !tables_of(a[3], a[4], q->size(0), bt, cl) ||
      kc->scalar_type() != q->scalar_type() || vc->scalar_type() != q->scalar_type() ||
      !type_code(q->scalar_type(), &dt) || !scale_of(a[5], n(*q, 2), &scale) ||
      debug_asked("CUDA_LLM_CHECK_BLOCK_TABLES"))
    return nullptr;
  const at::Tensor o = like(*q);
  const Workspace ws(abi.paged_decode_workspace_bytes(dt, 0, n(*q, 0), n(*q, 1), n(*kc, 1), n(*q, 2), n(*bt, 1)), *q);
  if (!ok([&] {
        return abi.paged_attention(dt, in(*q), in(*kc), in(*vc), (const int32_t*)in(*bt), (const int32_t*)in(*cl),
                                   out(o), n(*q, 0), n(*q, 1), n(*kc, 1), n(*q, 2), n(*bt, 1), 16, n(*kc, 0), scale,
                                   ws.ptr(), ws.bytes, stream());
      }))
    return nullptr;
  return THPVariable_Wrap(o);
}

// (query, key_cache, value_cache, k_scale, v_scale, block_tables, context_lens, softmax_scale) -> out
PyObject* fp8_paged_attention_forward(PyObject* const* a) {
  const at::Tensor *q = plain(a[0], 3), *kc, *vc, *ks, *vs, *bt, *cl;
  ca_dtype dt;
  float scale;
  if (!q || !caches_of(a[1], a[2], *q, kc, vc) || !scales_of(a[3], a[4], *kc, ks, vs) ||
      !tables_of(a[5], a[6], q->size(0), bt, cl) || !is_codes(kc->scalar_type()) || !is_codes(vc->scalar_type()) ||
      !type_code(q->scalar_type(), &dt) || !scale_of(a[7], n(*q, 2), &scale) ||
      debug_asked("CUDA_LLM_CHECK_BLOCK_TABLES"))
    return nullptr;
  const at::Tensor o = like(*q);
  const Workspace ws(abi.paged_decode_workspace_bytes(dt, 1, n(*q, 0), n(*q, 1), n(*kc, 1), n(*q, 2), n(*bt, 1)), *q);
  if (!ok([&] {
        return abi.fp8_paged_attention(dt, in(*q), (const uint8_t*)in(*kc), (const uint8_t*)in(*vc),
                                       (const float*)in(*ks), (const float*)in(*vs), ks->dim() == 2,
                                       (const int32_t*)in(*bt), (const int32_t*)in(*cl), out(o), n(*q, 0), n(*q, 1),
                                       n(*kc, 1), n(*q, 2), n(*bt, 1), 16, n(*kc, 0), scale, ws.ptr(), ws.bytes,
                                       stream());
      }))
    return nullptr;
  return THPVariable_Wrap(o);
}

// (key, value, key_cache, value_cache, block_tables, context_lens, new_lens, k_scale, v_scale) -> True
PyObject* paged_kv_append(PyObject* const* a) {
  const at::Tensor *k = plain(a[0], 4), *v = plain(a[1], 4), *kc = plain(a[2], 4), *vc = plain(a[3], 4), *bt, *cl;
  const at::Tensor *ks = nullptr, *vs = nullptr, *nl = nullptr;
  ca_dtype dt;
  if (!k || !v || !kc || !vc || k->sizes() != v->sizes() || k->scalar_type() != v->scalar_type() || !fits(*k) ||
      !fits(*kc) || !type_code(k->scalar_type(), &dt) || dt == CA_F32 || kc->sizes() != vc->sizes() ||
      kc->size(1) != k->size(1) || kc->size(2) != k->size(3) || kc->size(3) != 16 ||
      (k->size(3) != 64 && k->size(3) != 128) || !tables_of(a[4], a[5], k->size(0), bt, cl))
    return nullptr;
  const bool fp8 = is_codes(kc->scalar_type());
  if (fp8 ? !is_codes(vc->scalar_type()) || !scales_of(a[7], a[8], *kc, ks, vs)
          : kc->scalar_type() != k->scalar_type() || vc->scalar_type() != k->scalar_type())
    return nullptr;
  if (a[6] != Py_None && (!(nl = plain(a[6], 1, 4)) || nl->scalar_type() != at::kInt || nl->size(0) != k->size(0)))
    return nullptr;
  if (!ok([&] {
        return abi.paged_kv_append(dt, fp8, in(*k), in(*v), out(*kc), out(*vc), fp8 ? (float*)out(*ks) : nullptr,
                                   fp8 ? (float*)out(*vs) : nullptr, fp8 && ks->dim() == 2, (const int32_t*)in(*bt),
                                   (const int32_t*)in(*cl), nl ? (const int32_t*)in(*nl) : nullptr, n(*k, 0), n(*k, 1),
                                   n(*k, 3), n(*k, 2), n(*bt, 1), n(*kc, 0), stream());
      }))
    return nullptr;
  Py_RETURN_TRUE;
}

// (q, q_scale, k, k_scale, v, v_scale, is_causal, softmax_scale, half) -> out; e8m0 scale bytes; half: the
// output is fp16, otherwise bf16
PyObject* fused_microscaled_attention(PyObject* const* a) {
  const at::Tensor* t[6];
  int causal, half;
  float scale;
  for (int i = 0; i < 6; ++i)
    if (!(t[i] = plain(a[i], 4, i == 1 ? 4 : i == 5 ? 1 : 16))) return nullptr;
  const at::Tensor &q = *t[0], &k = *t[2], &v = *t[4];
  if (q.sizes() != k.sizes() || q.sizes() != v.sizes() || q.size(3) != 128 || !fits(q) || !is_codes(q.scalar_type()) ||
      !is_codes(k.scalar_type()) || !is_codes(v.scalar_type()) || !flag_of(a[6], &causal) ||
      !scale_of(a[7], 128, &scale) || !flag_of(a[8], &half))
    return nullptr;
  for (int i = 1; i < 6; i += 2)
    if ((t[i]->scalar_type() != at::kByte && t[i]->scalar_type() != at::kFloat8_e8m0fnu) || t[i]->size(3) != 4 ||
        t[i]->sizes().slice(0, 3) != q.sizes().slice(0, 3))
      return nullptr;
  const at::Tensor o =
      at::empty(q.sizes(), q.options().dtype(half ? at::kHalf : at::kBFloat16).requires_grad(false));
  const Workspace ws(abi.mx_workspace_bytes(CA_SCALE_E8M0, n(q, 0), n(q, 1), n(q, 2), 128), q);
  if (!ok([&] {
        return abi.fused_microscaled_attention(half ? CA_F16 : CA_BF16, (const uint8_t*)in(q), in(*t[1]),
                                               (const uint8_t*)in(k), in(*t[3]), (const uint8_t*)in(v), in(*t[5]),
                                               CA_SCALE_E8M0, out(o), n(q, 0), n(q, 1), n(q, 2), 128, scale, causal,
                                               ws.ptr(), ws.bytes, stream());
      }))
    return nullptr;
  return THPVariable_Wrap(o);
}

// A function of exactly N arguments; anything it does not take, and any C++
// exception (an allocation that fails, say), is None.
template <PyObject* (*F)(PyObject* const*), int N>
PyObject* call(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs == N) {
    try {
      if (PyObject* r = F(args)) return r;
    } catch (const std::exception&) {
    }
  }
  if (PyErr_Occurred()) return nullptr;
  Py_RETURN_NONE;
}

// bind(addresses of Abi's functions, in its order)
PyObject* bind(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  constexpr Py_ssize_t kFunctions = sizeof(Abi) / sizeof(void*);
  if (nargs != kFunctions) {
    PyErr_SetString(PyExc_TypeError, "bind: one address per function");
    return nullptr;
  }
  void* p[kFunctions];
  for (Py_ssize_t i = 0; i < kFunctions; ++i) {
    p[i] = PyLong_AsVoidPtr(args[i]);
    if (!p[i]) return nullptr;
  }
  static_assert(sizeof(p) == sizeof(abi), "one pointer per function");
  std::memcpy(&abi, p, sizeof(abi));
  Py_RETURN_NONE;
}

#define CA_FAST(F, N) {#F, (PyCFunction)(void (*)(void))call<F, N>, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {{"bind", (PyCFunction)(void (*)(void))bind, METH_FASTCALL, nullptr},
                         CA_FAST(flash_attention_forward, 5),
                         CA_FAST(flash_attention_forward_lse, 5),
                         CA_FAST(flash_attention_backward, 8),
                         CA_FAST(fused_rope_flash_attention, 7),
                         CA_FAST(async_flash_decode, 4),
                         CA_FAST(paged_attention_forward, 6),
                         CA_FAST(fp8_paged_attention_forward, 8),
                         CA_FAST(paged_kv_append, 9),
                         CA_FAST(fused_microscaled_attention, 9),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native() { return PyModule_Create(&module); }
