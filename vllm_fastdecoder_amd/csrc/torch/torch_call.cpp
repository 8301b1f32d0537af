// The ordinary form of ops.paged_decode and of the cache writes taken from
// torch tensors straight to the C ABI, in one native call.
//
// What bounds a small launch is the host: through ctypes a decode call took
// 13-15 us (about forty attribute reads and checks in Python, two tensor
// allocations through torch's Python layer, the conversion of 33 arguments),
// more than the kernel of a small batch. Here the same reads are direct: see
// ops.py for the figures.
//
// Each function handles exactly the calls whose every check in ops.py would
// pass, with all index tensors on the GPU, and returns None for any other
// (including tensor subclasses, functorch wrappers and active torch-function
// or dispatch modes), before anything is allocated or written: ops.py then
// runs its own checks and raises its own errors. Nothing is kept between
// calls: workspaces come from ops.WORKSPACE on every call, and host-tier
// addresses from pinned.device_ptr.
#include <Python.h>

#include <ATen/TensorSubclassLikeUtils.h>
#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/empty_like.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <torch/csrc/Device.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <cstring>

#include "../../../include/fdattn.h"

namespace {

// Python objects set once by init(): ops.WORKSPACE.get, pinned.device_ptr and
// torch's raw current-stream query.
PyObject* g_workspace_get = nullptr;
PyObject* g_device_ptr = nullptr;
PyObject* g_raw_stream = nullptr;

struct PyRef {  // an owned reference
  PyObject* p = nullptr;
  explicit PyRef(PyObject* o = nullptr) : p(o) {}
  PyRef(const PyRef&) = delete;
  PyRef& operator=(const PyRef&) = delete;
  ~PyRef() { Py_XDECREF(p); }
};

PyObject* not_here() { Py_RETURN_NONE; }

// A plain strided tensor with storage of its own.
const at::Tensor* plain(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || t.layout() != at::kStrided || !t.has_storage() ||
      at::isTensorSubclassLike(t) || t.is_conj() || t.is_neg())
    return nullptr;
  return &t;
}

const at::Tensor* plain_gpu(PyObject* o, at::ScalarType want) {
  const at::Tensor* t = plain(o);
  return t != nullptr && t->is_cuda() && t->scalar_type() == want ? t : nullptr;
}

int dtype_code(at::ScalarType s) {
  switch (s) {
    case at::kHalf: return FD_F16;
    case at::kBFloat16: return FD_BF16;
    case at::kFloat: return FD_F32;
    default: return -1;
  }
}

// False (with no Python error set) when o is no int that fits.
bool to_int64(PyObject* o, int64_t* out) {
  if (!PyLong_CheckExact(o)) return false;
  const long long v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  *out = v;
  return true;
}

bool fits32(int64_t x) { return x >= 0 && x <= INT32_MAX; }

// Calls that torch modes would have to see go through Python.
bool modes_active() {
  return at::impl::torch_function_mode_enabled() ||
         c10::impl::TorchDispatchModeTLS::any_modes_set();
}

// The current stream of device idx; false with a Python error set.
bool current_stream(int64_t idx, void** stream) {
  PyRef i(PyLong_FromLongLong(idx));
  if (i.p == nullptr) return false;
  PyRef s(PyObject_CallOneArg(g_raw_stream, i.p));
  if (s.p == nullptr) return false;
  *stream = reinterpret_cast<void*>(PyLong_AsUnsignedLongLong(s.p));
  return !(PyErr_Occurred());
}

// The (current) stream's workspace of at least `need` bytes and the counters behind it
// (ops._counters_ptr: on the next 256-byte boundary, where the buffer has
// them); `hold` keeps it alive over the launch. False with a Python error set.
bool workspace(const at::Tensor& q, size_t need, void* stream, PyRef& hold, void** ws,
               size_t* bytes, uint32_t** counters) {
  *ws = nullptr;
  *bytes = 0;
  *counters = nullptr;
  if (need == 0) return true;
  PyRef dev(THPDevice_New(q.device()));
  if (dev.p == nullptr) return false;
  PyRef n(PyLong_FromSize_t(need)), s(PyLong_FromVoidPtr(stream));
  if (n.p == nullptr || s.p == nullptr) return false;
  int32_t capturing = 1;  // (an error: the slower answer is right in either case)
  (void)fd_stream_capturing(stream, &capturing);
  hold.p = PyObject_CallFunctionObjArgs(g_workspace_get, dev.p, n.p, s.p, Py_False,
                                        capturing != 0 ? Py_True : Py_False, nullptr);
  if (hold.p == nullptr) return false;
  const at::Tensor& buf = THPVariable_Unpack(hold.p);
  *ws = buf.data_ptr();
  *bytes = (size_t)buf.numel();
  const size_t head = (*bytes + 255) / 256 * 256;
  if (buf.storage().nbytes() >= head + 4 * FD_DECODE_COUNTERS)
    *counters = reinterpret_cast<uint32_t*>(static_cast<char*>(*ws) + head);
  return true;
}

// The GPU's address of a cache tensor (HBM, or a view of pinned memory).
bool cache_ptr(PyObject* o, const at::Tensor& t, const void** p) {
  if (t.is_cuda()) {
    *p = t.data_ptr();
    return true;
  }
  PyRef r(PyObject_CallOneArg(g_device_ptr, o));
  if (r.p == nullptr) return false;
  *p = reinterpret_cast<const void*>(PyLong_AsUnsignedLongLong(r.p));
  return !PyErr_Occurred();
}

bool same_layout(const at::Tensor& a, const at::Tensor& b) {
  return a.sizes().equals(b.sizes()) && a.strides().equals(b.strides());
}

// q [n, H, D] on the GPU, of a KV dtype, contiguous in D, n > 0.
const at::Tensor* query(PyObject* o) {
  const at::Tensor* q = plain(o);
  if (q == nullptr || !q->is_cuda() || q->dim() != 3 || dtype_code(q->scalar_type()) < 0 ||
      q->size(0) <= 0 || q->stride(2) != 1 || !fits32(q->size(0)))
    return nullptr;
  return q;
}

// Table [n, W] (W > 0) and lengths [n] of int32 on q's device.
bool index_pair(const at::Tensor& q, PyObject* bt_o, PyObject* lens_o, const at::Tensor** bt,
                const at::Tensor** lens) {
  *bt = plain_gpu(bt_o, at::kInt);
  *lens = plain_gpu(lens_o, at::kInt);
  return *bt != nullptr && *lens != nullptr && (*bt)->dim() == 2 && (*bt)->size(0) == q.size(0) &&
         (*bt)->size(1) > 0 && (*bt)->stride(1) == 1 && fits32((*bt)->size(1)) &&
         (*lens)->dim() == 1 && (*lens)->size(0) == q.size(0) && (*lens)->is_contiguous() &&
         (*bt)->device() == q.device() && (*lens)->device() == q.device();
}

// row_order: None or a contiguous int32 [n] on q's device.
bool order_of(const at::Tensor& q, PyObject* o, const int32_t** order) {
  *order = nullptr;
  if (o == Py_None) return true;
  const at::Tensor* t = plain_gpu(o, at::kInt);
  if (t == nullptr || t->dim() != 1 || t->size(0) != q.size(0) || !t->is_contiguous() ||
      t->device() != q.device())
    return false;
  *order = t->data_ptr<int32_t>();
  return true;
}

// The outputs given, or room for new ones (undefined until allocate()).
struct Outputs {
  at::Tensor out, lse;
  bool ok = false;
  Outputs(const at::Tensor& q, PyObject* out_o, PyObject* lse_o) {
    const int64_t n = q.size(0), H = q.size(1);
    if (out_o != Py_None) {
      const at::Tensor* t = plain(out_o);
      if (t == nullptr || !t->is_cuda() || t->device() != q.device() ||
          !t->sizes().equals(q.sizes()) || t->stride(2) != 1 ||
          (t->scalar_type() != q.scalar_type() && t->scalar_type() != at::kFloat))
        return;
      out = *t;
    }
    if (lse_o != Py_None) {
      const at::Tensor* t = plain_gpu(lse_o, at::kFloat);
      if (t == nullptr || t->device() != q.device() || t->dim() != 2 || t->size(0) != H ||
          t->size(1) != n || t->stride(1) != 1)
        return;
      lse = *t;
    }
    ok = true;
  }
  bool allocate(const at::Tensor& q) {
    if (!out.defined()) out = at::empty_like(q);
    if (!lse.defined()) lse = at::empty({q.size(1), q.size(0)}, q.options().dtype(at::kFloat));
    // (empty_like keeps a dense q's strides: the last dim may not be the contiguous one)
    return out.stride(2) == 1;
  }
};

// (out, lse), or (status,) of a refused call for _lib.check.
PyObject* result(int status, const Outputs& o) {
  if (status != FD_OK) return Py_BuildValue("(i)", status);
  PyRef a(THPVariable_Wrap(o.out));
  PyRef b(THPVariable_Wrap(o.lse));
  if (a.p == nullptr || b.p == nullptr) return nullptr;
  return PyTuple_Pack(2, a.p, b.p);
}

// Runs a library call without the GIL: a launch may wait for room in its
// queue, as torch's own launches do without it. The GIL is back before an
// exception (a tensor's data_ptr may throw) leaves.
template <typename F>
int without_gil(F&& f) {
  struct Released {
    PyThreadState* save = PyEval_SaveThread();
    ~Released() { PyEval_RestoreThread(save); }
  } released;
  return f();
}

// No C++ exception leaves an entry point: it becomes a Python RuntimeError.
template <typename F>
PyObject* guarded(F&& f) {
  try {
    return f();
  } catch (const c10::Error& e) {
    PyErr_SetString(PyExc_RuntimeError, e.what_without_backtrace());
  } catch (const std::exception& e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
  }
  return nullptr;
}

// paged_decode(q, key_cache, value_cache, block_table, seqused_k, scale, out,
//              lse, row_order, max_seqlen_k, total_tokens)
PyObject* paged_decode(PyObject*, PyObject* const* a, Py_ssize_t na) {
  return guarded([&]() -> PyObject* {
    if (na != 11 || modes_active()) return not_here();
    const at::Tensor* q = query(a[0]);
    const at::Tensor* k = plain(a[1]);
    const at::Tensor* v = plain(a[2]);
    const at::Tensor *bt, *lens;
    if (q == nullptr || k == nullptr || v == nullptr || !k->is_cuda() || !v->is_cuda() ||
        k->device() != q->device() || v->device() != q->device() || k->dim() != 4 ||
        !same_layout(*k, *v) || k->scalar_type() != q->scalar_type() ||
        v->scalar_type() != q->scalar_type() || k->stride(3) != 1 || k->size(3) != q->size(2) ||
        !index_pair(*q, a[3], a[4], &bt, &lens) || !PyFloat_CheckExact(a[5]))
      return not_here();
    const int64_t n = q->size(0), H = q->size(1), D = q->size(2);
    const int64_t B = k->size(0), BS = k->size(1), KVH = k->size(2);
    if (!fits32(H) || !fits32(D) || !fits32(BS) || !fits32(KVH) || BS == 0) return not_here();
    int64_t width = bt->size(1), total = 0, longest = 0;
    if (a[9] != Py_None) {
      if (!to_int64(a[9], &longest) || longest < 0 || longest > INT32_MAX) return not_here();
      width = std::min(width, std::max<int64_t>(1, (longest + BS - 1) / BS));
    }
    if (a[10] != Py_None && !to_int64(a[10], &total)) return not_here();
    const int32_t* order;
    if (!order_of(*q, a[8], &order)) return not_here();
    Outputs o(*q, a[6], a[7]);
    if (!o.ok) return not_here();
    const int kv = dtype_code(q->scalar_type());
    const float scale = (float)PyFloat_AS_DOUBLE(a[5]);
    size_t need = 0;
    int32_t host = 0;  // a GPU tensor may lie over mapped host memory
    if (fd_in_host_memory(k->data_ptr(), &host) != FD_OK ||
        fd_decode_workspace_need((int32_t)n, (int32_t)H, (int32_t)KVH, (int32_t)D, (int32_t)BS,
                                 (int32_t)width, kv, host, total, &need) != FD_OK)
      return not_here();  // sizes the call refuses: with Python's message
    if (!o.allocate(*q)) return not_here();
    PyRef hold;
    void *ws, *stream;
    size_t ws_bytes;
    uint32_t* counters;
    if (!current_stream(q->get_device(), &stream) ||
        !workspace(*q, need, stream, hold, &ws, &ws_bytes, &counters))
      return nullptr;
    const int status = without_gil([&] { return fd_paged_decode_counted(
        q->data_ptr(), q->stride(0), q->stride(1), k->data_ptr(), v->data_ptr(), k->stride(0),
        k->stride(2), k->stride(1), B, bt->data_ptr<int32_t>(), bt->stride(0), (int32_t)width,
        lens->data_ptr<int32_t>(), order, (int32_t)n, (int32_t)H, (int32_t)KVH, (int32_t)D,
        (int32_t)BS, scale, kv, o.out.data_ptr(), o.out.stride(0), o.out.stride(1),
        dtype_code(o.out.scalar_type()), o.lse.data_ptr<float>(), o.lse.stride(0), ws, ws_bytes,
        stream, total, counters); });
    return result(status, o);
  });
}

// key and value rows [T, KVH, D] of one shape, T given by the slots.
bool kv_rows(const at::Tensor* key, const at::Tensor* value) {
  return key != nullptr && value != nullptr && key->is_cuda() && value->device() == key->device() &&
         key->dim() == 3 && value->sizes().equals(key->sizes()) &&
         value->scalar_type() == key->scalar_type() && dtype_code(key->scalar_type()) >= 0 &&
         key->stride(2) == 1 && value->stride(2) == 1;
}

// A cache the rows go to: [B, BS, KVH, D] views with token and head dims 1
// and 2, or the host tier's [C, KVH, BS, D] with 2 and 1. 1: filled in; 0: not
// for this path; -1: a Python error is set.
int cache_target(const at::Tensor& key, PyObject* k_o, PyObject* v_o, PyObject* slots_o, int token,
                 int head, fd_cache_target* c, int64_t* T, int64_t* BS) {
  const at::Tensor* k = plain(k_o);
  const at::Tensor* v = plain(v_o);
  const at::Tensor* slots = plain_gpu(slots_o, at::kLong);
  if (k == nullptr || v == nullptr || slots == nullptr || k->dim() != 4 || !same_layout(*k, *v) ||
      slots->dim() != 1 || !slots->is_contiguous() || slots->device() != key.device())
    return 0;
  *T = slots->size(0);
  *BS = k->size(token);
  if (*T <= 0 || !fits32(*T) || key.size(0) < *T || k->size(head) != key.size(1) ||
      k->size(3) != key.size(2) || !fits32(*BS))
    return 0;
  for (const at::Tensor* t : {k, v})
    if (t->scalar_type() != key.scalar_type() ||
        !(t->is_cuda() ? t->device() == key.device() : t->is_cpu()))
      return 0;
  const void *kp, *vp;
  if (!cache_ptr(k_o, *k, &kp) || !cache_ptr(v_o, *v, &vp)) return -1;
  c->k_cache = const_cast<void*>(kp);
  c->v_cache = const_cast<void*>(vp);
  c->stride_block = k->stride(0);
  c->stride_token = k->stride(token);
  c->stride_head = k->stride(head);
  c->num_blocks = k->size(0);
  c->slot_mapping = slots->data_ptr<int64_t>();
  return 1;
}

// None, or an int32 device counter's address.
bool device_counter(PyObject* o, int32_t** c) {
  *c = nullptr;
  if (o == Py_None) return true;
  const at::Tensor* t = plain_gpu(o, at::kInt);
  if (t != nullptr) *c = t->data_ptr<int32_t>();
  return t != nullptr;
}

// cache_write(key, value, key_cache, value_cache, slots, error_count,
//             write_gate): the caches as [B, BS, KVH, D] views -> status
PyObject* cache_write(PyObject*, PyObject* const* a, Py_ssize_t na) {
  return guarded([&]() -> PyObject* {
    if (na != 7 || modes_active()) return not_here();
    const at::Tensor* key = plain(a[0]);
    const at::Tensor* value = plain(a[1]);
    int32_t *err, *gate;
    if (!kv_rows(key, value) || !device_counter(a[5], &err) || !device_counter(a[6], &gate) ||
        (err != nullptr && err == gate))
      return not_here();
    fd_cache_target c{};
    int64_t T, BS;
    const int got = cache_target(*key, a[2], a[3], a[4], 1, 2, &c, &T, &BS);
    if (got <= 0) return got == 0 ? not_here() : nullptr;
    void* stream;
    if (!current_stream(key->get_device(), &stream)) return nullptr;
    const int status = without_gil([&] { return fd_reshape_and_cache(
        key->data_ptr(), key->stride(0), key->stride(1), value->data_ptr(), value->stride(0),
        value->stride(1), c.k_cache, c.v_cache, c.stride_block, c.stride_token, c.stride_head,
        c.num_blocks, c.slot_mapping, (int32_t)T, (int32_t)key->size(1), (int32_t)key->size(2),
        (int32_t)BS, dtype_code(key->scalar_type()), err, gate, stream); });
    return PyLong_FromLong(status);
  });
}

// cache_write_tiers(key, value, key_cache, value_cache, slots, host_k, host_v,
//                   host_slots, write_gate): the host caches as [C, KVH, BS, D]
PyObject* cache_write_tiers(PyObject*, PyObject* const* a, Py_ssize_t na) {
  return guarded([&]() -> PyObject* {
    if (na != 9 || modes_active()) return not_here();
    const at::Tensor* key = plain(a[0]);
    const at::Tensor* value = plain(a[1]);
    int32_t* gate;
    if (!kv_rows(key, value) || !device_counter(a[8], &gate)) return not_here();
    fd_cache_target c[2] = {};
    int64_t T[2], BS[2];
    for (int t = 0; t < 2; ++t) {
      PyObject* const* x = a + 2 + 3 * t;
      const int got = cache_target(*key, x[0], x[1], x[2], t == 0 ? 1 : 2, t == 0 ? 2 : 1, &c[t],
                                   &T[t], &BS[t]);
      if (got <= 0) return got == 0 ? not_here() : nullptr;
    }
    if (T[0] != T[1] || BS[0] != BS[1]) return not_here();
    void* stream;
    if (!current_stream(key->get_device(), &stream)) return nullptr;
    const int status = without_gil([&] { return fd_reshape_and_cache_tiers(
        key->data_ptr(), key->stride(0), key->stride(1), value->data_ptr(), value->stride(0),
        value->stride(1), &c[0], &c[1], (int32_t)T[0], (int32_t)key->size(1),
        (int32_t)key->size(2), (int32_t)BS[0], dtype_code(key->scalar_type()), gate, stream); });
    return PyLong_FromLong(status);
  });
}

// init(WORKSPACE.get, pinned.device_ptr, raw current-stream query,
//      torch.__version__): an ImportError where the module was built against
// another torch, whose tensors it would read by the wrong layout, or beside a
// library of another ABI.
PyObject* init(PyObject*, PyObject* args) {
  PyObject *ws, *dp, *rs;
  const char* torch_version;
  if (!PyArg_ParseTuple(args, "OOOs", &ws, &dp, &rs, &torch_version)) return nullptr;
  if (strcmp(torch_version, FD_BUILT_FOR_TORCH) != 0)
    return PyErr_Format(PyExc_ImportError, "_torch_call was built for torch %s, not %s",
                        FD_BUILT_FOR_TORCH, torch_version);
  if (fd_abi_version() != FD_ABI_VERSION)
    return PyErr_Format(PyExc_ImportError, "_torch_call was built for ABI %d of the library, not %d",
                        FD_ABI_VERSION, fd_abi_version());
  Py_INCREF(ws);
  Py_INCREF(dp);
  Py_INCREF(rs);
  g_workspace_get = ws;
  g_device_ptr = dp;
  g_raw_stream = rs;
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"init", init, METH_VARARGS, nullptr},
    {"paged_decode", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(paged_decode)),
     METH_FASTCALL, nullptr},
    {"cache_write", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(cache_write)),
     METH_FASTCALL, nullptr},
    {"cache_write_tiers",
     reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(cache_write_tiers)), METH_FASTCALL,
     nullptr},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_torch_call", nullptr, -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

extern "C" PyObject* PyInit__torch_call() { return PyModule_Create(&module); }
