// The eager calls' host side in C++: what `paged_kernels.paged_decode`,
// `paged_kernels.paged_prefill` and `rope.rope_kv_write` do in Python before
// they reach the C ABI (reading the
// operands, the checks, the output and workspace, the call).
//
// A decode layer over a few short contexts runs ~8 us on the GPU, and its two
// calls took 31 us of Python and ctypes (about half checks and attribute
// reads, half converting ~60 arguments); through here they take 15.
//
// Each function serves exactly what the Python code would pass on unchanged:
// plain torch tensors on one ROCm device, in the layouts and dtypes the C ABI
// takes. For anything else (another device or dtype, a layout that needs a
// copy, a shape that does not match, a tensor subclass) it does nothing and
// returns None, and the Python code, which converts or raises, runs as
// before. A failed call returns its status for the Python code to raise.
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/ATen.h>
#include <Python.h>

#include <cmath>
#include <cstdint>

#include "../../include/liteinfer_amd.h"

namespace {

using PlanFn = decltype(&li_paged_decode_plan);
using DecodeFn = decltype(&li_paged_decode_write);
using PrefillPlanFn = decltype(&li_paged_prefill_plan);
using PrefillFn = decltype(&li_paged_prefill_ex);
using RopeFn = decltype(&li_rope_kv_write);
using RopeF8Fn = decltype(&li_rope_kv_write_fp8);
PlanFn g_plan = nullptr;
DecodeFn g_decode = nullptr;
PrefillPlanFn g_prefill_plan = nullptr;
PrefillFn g_prefill = nullptr;
RopeFn g_rope = nullptr;
RopeF8Fn g_rope_f8 = nullptr;

// The interpreter lock is given up for the allocation and the launch, as
// torch's own calls and ctypes do.
struct Unlocked {
  PyThreadState* state = PyEval_SaveThread();
  ~Unlocked() { PyEval_RestoreThread(state); }
};

// A plain tensor (no subclass, so no __torch_function__ of its own) that
// holds device memory of its own, or nullptr.
const at::Tensor* plain(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || !t.has_storage()) return nullptr;
  const auto keys = t.key_set();
  if (keys.has(c10::DispatchKey::Python) || keys.has(c10::DispatchKey::FuncTorchBatched) ||
      keys.has(c10::DispatchKey::FuncTorchGradWrapper) || keys.has(c10::DispatchKey::Functionalize) ||
      t.is_neg() || t.is_conj())
    return nullptr;
  return &t;
}

int code_of(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return LI_F32;
    case at::kHalf: return LI_F16;
    case at::kBFloat16: return LI_BF16;
    case at::kFloat8_e4m3fn: return LI_FP8_E4M3;
    default: return -1;
  }
}

bool pools_ok(const at::Tensor& k, const at::Tensor& v) {
  return k.dim() == 3 && v.dim() == 3 && k.sizes() == v.sizes() && k.strides() == v.strides() && k.stride(2) == 1 &&
         k.scalar_type() == v.scalar_type();
}

// The pool's element code beside 16- or 32-bit rows of type `rows` (scales
// checked for an fp8 pool), or -1.
int pool_code(at::ScalarType rows, const at::Tensor& pool, double k_scale, double v_scale) {
  const int code = code_of(rows);
  if (code < 0 || code == LI_FP8_E4M3) return -1;
  if (pool.scalar_type() == rows) return code;
  if (pool.scalar_type() != at::kFloat8_e4m3fn || code == LI_F32) return -1;
  if (!(k_scale > 0) || !(v_scale > 0) || !std::isfinite(k_scale) || !std::isfinite(v_scale)) return -1;
  return LI_FP8_E4M3;
}

// 1: a number into *out; 0: not one this serves.
bool number(PyObject* o, double* out) {
  if (PyFloat_CheckExact(o)) *out = PyFloat_AS_DOUBLE(o);
  else if (PyLong_CheckExact(o)) *out = PyLong_AsDouble(o);
  else return false;
  if (PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}

bool integer(PyObject* o, int64_t* out) {
  if (!PyLong_CheckExact(o)) return false;
  int overflow = 0;
  *out = PyLong_AsLongLongAndOverflow(o, &overflow);
  return !overflow && !PyErr_Occurred();
}

// decode(query, key_pool, value_pool, slot_table, context_lens, scaling, groups, block_kv, num_splits (0: None),
//        flags, k_scale, v_scale, new_key or None, new_value or None, stream) -> out, status, or None
PyObject* decode(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 15 || !g_decode) Py_RETURN_NONE;
  const at::Tensor *q = plain(a[0]), *kp = plain(a[1]), *vp = plain(a[2]), *st = plain(a[3]), *cl = plain(a[4]);
  double scaling, k_scale, v_scale;
  int64_t groups, block_kv, splits, flags, stream;
  if (!q || !kp || !vp || !st || !cl || !number(a[5], &scaling) || !integer(a[6], &groups) || !integer(a[7], &block_kv) ||
      !integer(a[8], &splits) || !integer(a[9], &flags) || !number(a[10], &k_scale) || !number(a[11], &v_scale) ||
      !integer(a[14], &stream))
    Py_RETURN_NONE;
  const auto device = q->device();
  if (kp->device() != device || vp->device() != device || st->device() != device || cl->device() != device) Py_RETURN_NONE;
  if (!pools_ok(*kp, *vp) || kp->size(0) >= (int64_t(1) << 31)) Py_RETURN_NONE;
  const int kv = pool_code(q->scalar_type(), *kp, k_scale, v_scale);
  if (kv < 0 || q->dim() != 3 || q->stride(2) != 1 || st->dim() != 2 || st->scalar_type() != at::kLong ||
      st->stride(1) != 1 || cl->dim() != 1 || cl->scalar_type() != at::kInt || cl->stride(0) != 1)
    Py_RETURN_NONE;
  const int64_t batch = q->size(0), heads = q->size(1), dim = q->size(2), kv_heads = kp->size(1), width = st->size(1);
  constexpr int64_t kInt = 0x7fffffff;
  if (groups < 1 || heads % groups || heads / groups != kv_heads || dim != kp->size(2) || st->size(0) != batch ||
      cl->size(0) != batch || batch < 1 || batch > kInt || heads > kInt || width > kInt || splits < 0 || splits > kInt ||
      block_kv < 0 || block_kv > kInt || flags < 0 || flags > kInt)
    Py_RETURN_NONE;
  const at::Tensor *nk = nullptr, *nv = nullptr;
  if (a[12] != Py_None || a[13] != Py_None) {
    nk = plain(a[12]), nv = plain(a[13]);
    if (!nk || !nv) Py_RETURN_NONE;
    for (const at::Tensor* t : {nk, nv})
      if (t->dim() != 3 || t->size(0) != batch || t->size(1) != kv_heads || t->size(2) != dim || t->stride(2) != 1 ||
          t->scalar_type() != q->scalar_type() || t->device() != device)
        Py_RETURN_NONE;
    if (nk->strides() != nv->strides()) Py_RETURN_NONE;
  }
  size_t need = 0;
  if (g_plan((int)batch, (int)heads, (int)kv_heads, (int)dim, (int)width, (int)splits, 0, (int)block_kv, nullptr, nullptr,
             &need) != LI_OK)
    Py_RETURN_NONE;
  try {
    at::Tensor out, workspace;
    int status;
    {
      Unlocked unlocked;
      at::AutoDispatchBelowADInplaceOrView below;
      out = at::empty_like(*q);
      if (need) workspace = at::empty({(int64_t)need}, q->options().dtype(at::kByte));
      status = g_decode(q->data_ptr(), q->stride(0), q->stride(1), kp->data_ptr(), vp->data_ptr(), kp->stride(0),
                        kp->stride(1), st->const_data_ptr<int64_t>(), st->stride(0), (int)width,
                        cl->const_data_ptr<int32_t>(), nk ? nk->data_ptr() : nullptr, nv ? nv->data_ptr() : nullptr,
                        nk ? nk->stride(0) : 0, nk ? nk->stride(1) : 0, kp->size(0), nullptr, out.data_ptr(),
                        out.stride(0), out.stride(1), (int)batch, (int)heads, (int)kv_heads, (int)dim, (float)scaling,
                        (int)splits, (int)block_kv, need ? workspace.data_ptr() : nullptr, need,
                        code_of(q->scalar_type()), kv, (float)k_scale, (float)v_scale, (int)flags,
                        reinterpret_cast<void*>(stream));
    }
    if (status != LI_OK) return PyLong_FromLong(status);
    return THPVariable_Wrap(std::move(out));
  } catch (const std::exception&) {
    // (An allocation that failed: the Python code tries it again and raises torch's own error.)
    Py_RETURN_NONE;
  }
}

// prefill(query, key_pool, value_pool, slot_table, context_lens, query_start_loc, max_query_len, scaling, groups,
//         block_kv, block_q, flags, k_scale, v_scale, out or None, stream) -> out, status, or None
PyObject* prefill(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 16 || !g_prefill) Py_RETURN_NONE;
  const at::Tensor* t[6];
  for (int i = 0; i < 6; ++i)
    if (!(t[i] = plain(a[i])) || t[i]->device() != t[0]->device()) Py_RETURN_NONE;
  const at::Tensor &q = *t[0], &kp = *t[1], &vp = *t[2], &st = *t[3], &cl = *t[4], &qsl = *t[5];
  double scaling, k_scale, v_scale;
  int64_t longest, groups, block_kv, block_q, flags, stream;
  if (!integer(a[6], &longest) || !number(a[7], &scaling) || !integer(a[8], &groups) || !integer(a[9], &block_kv) ||
      !integer(a[10], &block_q) || !integer(a[11], &flags) || !number(a[12], &k_scale) || !number(a[13], &v_scale) ||
      !integer(a[15], &stream) || !pools_ok(kp, vp) || kp.size(0) >= (int64_t(1) << 31))
    Py_RETURN_NONE;
  const int kv = pool_code(q.scalar_type(), kp, k_scale, v_scale);
  if (kv < 0 || q.dim() != 3 || q.stride(2) != 1 || st.dim() != 2 || st.scalar_type() != at::kLong || st.stride(1) != 1 ||
      cl.dim() != 1 || cl.scalar_type() != at::kInt || cl.stride(0) != 1 || qsl.dim() != 1 ||
      qsl.scalar_type() != at::kInt || qsl.stride(0) != 1)
    Py_RETURN_NONE;
  const int64_t batch = cl.size(0), heads = q.size(1), dim = q.size(2), kv_heads = kp.size(1), width = st.size(1);
  constexpr int64_t kInt = 0x7fffffff;
  if (groups < 1 || heads % groups || heads / groups != kv_heads || dim != kp.size(2) || st.size(0) != batch ||
      qsl.size(0) != batch + 1 || batch < 1 || batch > kInt || heads > kInt || width > kInt || longest < 0 ||
      longest > kInt || block_kv < 0 || block_kv > kInt || block_q < 0 || block_q > kInt || flags < 0 || flags > kInt)
    Py_RETURN_NONE;
  const at::Tensor* given = nullptr;
  if (a[14] != Py_None) {
    given = plain(a[14]);
    if (!given || given->sizes() != q.sizes() || given->scalar_type() != q.scalar_type() ||
        given->device() != q.device() || given->stride(2) != 1)
      Py_RETURN_NONE;
  }
  size_t need = 0;
  if (g_prefill_plan((int)batch, (int)heads, (int)kv_heads, (int)dim, (int)width, 0, &need) != LI_OK) Py_RETURN_NONE;
  try {
    at::Tensor out, workspace;
    int status;
    {
      Unlocked unlocked;
      at::AutoDispatchBelowADInplaceOrView below;
      if (!given) out = at::empty_like(q);
      const at::Tensor& o = given ? *given : out;
      if (need) workspace = at::empty({(int64_t)need}, q.options().dtype(at::kByte));
      status = g_prefill(q.data_ptr(), q.stride(0), q.stride(1), kp.data_ptr(), vp.data_ptr(), kp.stride(0), kp.stride(1),
                         st.const_data_ptr<int64_t>(), st.stride(0), (int)width, cl.const_data_ptr<int32_t>(),
                         qsl.const_data_ptr<int32_t>(), (int)batch, (int)longest, o.data_ptr(), o.stride(0), o.stride(1),
                         (int)heads, (int)kv_heads, (int)dim, (float)scaling, (int)block_q, (int)block_kv,
                         need ? workspace.data_ptr() : nullptr, need, code_of(q.scalar_type()), kv, (float)k_scale,
                         (float)v_scale, (int)flags, reinterpret_cast<void*>(stream));
    }
    if (status != LI_OK) return PyLong_FromLong(status);
    if (given) return (Py_INCREF(a[14]), a[14]);
    return THPVariable_Wrap(std::move(out));
  } catch (const std::exception&) {
    Py_RETURN_NONE;
  }
}

// rope(q, k, v, cos, sin, slots, key_pool, value_pool, k_scale, v_scale, bad_slots or None, stream)
//   -> rotated q, status, or None
PyObject* rope(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 12 || !g_rope) Py_RETURN_NONE;
  const at::Tensor* t[8];
  for (int i = 0; i < 8; ++i)
    if (!(t[i] = plain(a[i])) || t[i]->device() != t[0]->device()) Py_RETURN_NONE;
  const at::Tensor &q = *t[0], &k = *t[1], &v = *t[2], &cos = *t[3], &sin = *t[4], &slots = *t[5], &kp = *t[6], &vp = *t[7];
  double k_scale, v_scale;
  int64_t stream;
  if (!number(a[8], &k_scale) || !number(a[9], &v_scale) || !integer(a[11], &stream) || !pools_ok(kp, vp)) Py_RETURN_NONE;
  const auto dtype = q.scalar_type();
  const int kv = pool_code(dtype, kp, k_scale, v_scale);
  if (kv < 0 || q.dim() != 4 || k.dim() != 4 || v.dim() != 4 || cos.dim() != 3 || sin.dim() != 3) Py_RETURN_NONE;
  for (int i = 1; i < 5; ++i)
    if (t[i]->scalar_type() != dtype) Py_RETURN_NONE;
  const int64_t batch = q.size(0), heads = q.size(1), tokens = q.size(2), dim = q.size(3), kv_heads = k.size(1);
  if (k.sizes() != v.sizes() || k.size(0) != batch || k.size(2) != tokens || k.size(3) != dim || kv_heads != kp.size(1) ||
      dim != kp.size(2) || dim % 2 || cos.sizes() != sin.sizes() || cos.strides() != sin.strides() ||
      cos.size(1) != tokens || cos.size(2) != dim || (cos.size(0) != 1 && cos.size(0) != batch))
    Py_RETURN_NONE;
  if (slots.scalar_type() != at::kLong || !slots.is_contiguous() || slots.numel() != batch * tokens || slots.numel() < 1)
    Py_RETURN_NONE;
  int32_t* bad = nullptr;
  if (a[10] != Py_None) {
    const at::Tensor* b = plain(a[10]);
    if (!b || b->scalar_type() != at::kInt || b->numel() < 1 || b->device() != q.device()) Py_RETURN_NONE;
    bad = b->data_ptr<int32_t>();
  }
  const int64_t cs[3] = {cos.size(0) == 1 ? 0 : cos.stride(0), cos.stride(1), cos.stride(2)};
  try {
    at::Tensor out;
    int status;
    {
      Unlocked unlocked;
      at::AutoDispatchBelowADInplaceOrView below;
      out = at::empty({batch, tokens, heads, dim}, q.options()).transpose(1, 2);
      const int64_t os[4] = {out.stride(0), out.stride(1), out.stride(2), out.stride(3)};
      void* s = reinterpret_cast<void*>(stream);
      const int64_t* sl = slots.const_data_ptr<int64_t>();
      if (kv == LI_FP8_E4M3)
        status = g_rope_f8(q.data_ptr(), q.strides().data(), k.data_ptr(), k.strides().data(), v.data_ptr(),
                           v.strides().data(), cos.data_ptr(), sin.data_ptr(), cs, batch, tokens, sl, out.data_ptr(), os,
                           kp.data_ptr(), vp.data_ptr(), kp.size(0), kp.stride(0), kp.stride(1), (int)heads,
                           (int)kv_heads, (int)dim, code_of(dtype), (float)k_scale, (float)v_scale, bad, s);
      else
        status = g_rope(q.data_ptr(), q.strides().data(), k.data_ptr(), k.strides().data(), v.data_ptr(),
                        v.strides().data(), cos.data_ptr(), sin.data_ptr(), cs, batch, tokens, sl, out.data_ptr(), os,
                        kp.data_ptr(), vp.data_ptr(), kp.size(0), kp.stride(0), kp.stride(1), (int)heads, (int)kv_heads,
                        (int)dim, code_of(dtype), bad, s);
    }
    if (status != LI_OK) return PyLong_FromLong(status);
    return THPVariable_Wrap(std::move(out));
  } catch (const std::exception&) {
    Py_RETURN_NONE;
  }
}

// bind(decode plan, decode_write, prefill plan, prefill, rope, rope_fp8): the loaded library's entry points, as addresses.
PyObject* bind(PyObject*, PyObject* const* a, Py_ssize_t n) {
  int64_t p[6];
  for (int i = 0; i < 6; ++i)
    if (n != 6 || !integer(a[i], &p[i])) {
      PyErr_SetString(PyExc_TypeError, "bind takes six addresses");
      return nullptr;
    }
  g_plan = reinterpret_cast<PlanFn>(p[0]);
  g_decode = reinterpret_cast<DecodeFn>(p[1]);
  g_prefill_plan = reinterpret_cast<PrefillPlanFn>(p[2]);
  g_prefill = reinterpret_cast<PrefillFn>(p[3]);
  g_rope = reinterpret_cast<RopeFn>(p[4]);
  g_rope_f8 = reinterpret_cast<RopeF8Fn>(p[5]);
  Py_RETURN_NONE;
}

PyMethodDef kMethods[] = {
    {"decode", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(decode)), METH_FASTCALL, nullptr},
    {"prefill", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(prefill)), METH_FASTCALL, nullptr},
    {"rope", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(rope)), METH_FASTCALL, nullptr},
    {"bind", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(bind)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_fast_calls", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

extern "C" __attribute__((visibility("default"))) PyObject* PyInit__fast_calls() {
  PyObject* m = PyModule_Create(&kModule);
  if (m && PyModule_AddStringConstant(m, "build_id", LI_BUILD_ID) < 0) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
