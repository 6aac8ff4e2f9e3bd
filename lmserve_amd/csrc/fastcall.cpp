/* _kvc_fast: CPython entry to the two per-layer plan calls of libkvcache.
 *
 * A forward pass calls the K/V write once per layer; at decode sizes the launch
 * is host-bound, so what the binding adds per call is what a serving loop feels.
 * ctypes converts and type-checks every argument through Python objects (about
 * 0.8 us for nine arguments) and the layout checks of three or five tensors cost
 * another microsecond of attribute reads in Python. Here the tensors are
 * unpacked in C++ (pointer, strides, sizes, dtype and device are plain member
 * reads) and the integers are read straight off the argument vector.
 *
 * The same holds for the drop-in per-layer calls (`append_paged`,
 * `reshape_and_cache`, `rotary_pos_emb`, `rotary_append_paged`): up to twelve
 * tensors checked here instead of in Python.
 *
 * The wrappers add nothing to the C ABI: each forwards to the entry point of
 * the same name in include/kvcache.h. They only accept the layouts the common
 * case produces and return NOT_FAST (1) for anything else, so that the Python
 * caller can run its own checks, which name what is wrong or handle the rare
 * layout; a negative return is the kvc_status of the library call.
 */
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/core/Tensor.h>

#include <hip/hip_runtime_api.h>

#include <cstdint>

#if PY_VERSION_HEX < 0x030B0000
#include <longintrepr.h>
#endif

#include <ATen/ops/empty.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/variable.h>

#include <algorithm>
#include <cstring>
#include <vector>

#include "kvcache.h"
#include "kvcache_experimental.h"

namespace {

constexpr long NOT_FAST = 1;
constexpr long kInterface = 2;  // changes with the names or arguments of the functions below; _lib.py checks it

bool as_ptr(PyObject* o, void** out) {
  if (o == Py_None) {
    *out = nullptr;
    return true;
  }
  *out = PyLong_AsVoidPtr(o);
  return !(*out == nullptr && PyErr_Occurred());
}

bool as_i64(PyObject* o, int64_t* out) {
  *out = (int64_t)PyLong_AsLongLong(o);
  return !(*out == -1 && PyErr_Occurred());
}

// Token-major rows, dense inside a token: [n, width] or [n, heads, dim] with
// heads * dim == width. Returns the token stride in elements, or -1.
int64_t row_stride(const at::Tensor& t, int64_t n, int64_t width, int dtype, int device) {
  if ((int)t.scalar_type() != dtype || !t.is_cuda() || t.device().index() != device) return -1;
  const auto sizes = t.sizes();
  const auto strides = t.strides();
  if (sizes.size() == 2) {
    if (sizes[0] != n || sizes[1] != width || strides[1] != 1) return -1;
  } else if (sizes.size() == 3) {
    if (sizes[0] != n || sizes[1] * sizes[2] != width || strides[2] != 1 ||
        (sizes[1] > 1 && strides[1] != sizes[2]))
      return -1;
  } else {
    return -1;
  }
  if (n > 1 && strides[0] < width) return -1;
  return n > 1 ? strides[0] : width;
}

// One layer of the pool, [num_pages, 2, page_size, H, D] with contiguous pages.
// Returns the page stride in elements, or -1.
int64_t page_stride(const at::Tensor& c, int64_t page_size, int64_t heads, int64_t dim, int dtype,
                    int device, int64_t* num_pages) {
  if ((int)c.scalar_type() != dtype || !c.is_cuda() || c.device().index() != device) return -1;
  const auto sizes = c.sizes();
  const auto strides = c.strides();
  if (sizes.size() != 5 || sizes[1] != 2 || sizes[2] != page_size || sizes[3] != heads || sizes[4] != dim)
    return -1;
  const int64_t row = heads * dim;
  if (strides[4] != 1 || strides[3] != dim || strides[2] != row || strides[1] != page_size * row) return -1;
  *num_pages = sizes[0];
  if (sizes[0] < 1) return -1;
  if (sizes[0] > 1 && strides[0] < 2 * page_size * row) return -1;  // overlapping pages
  return sizes[0] > 1 ? strides[0] : 2 * page_size * row;
}

const at::Tensor* tensor_of(PyObject* o) {
  return THPVariable_Check(o) ? &THPVariable_Unpack(o) : nullptr;
}

// rows as above, but the tensor may hold more rows than are written
int64_t row_stride_at_least(const at::Tensor& t, int64_t n, int64_t width, int dtype, int device) {
  if (t.dim() < 1 || t.sizes()[0] < n) return -1;
  if (t.sizes()[0] == n) return row_stride(t, n, width, dtype, device);
  const int64_t st = row_stride(t, t.sizes()[0], width, dtype, device);
  return st < 0 ? -1 : (n > 1 ? st : width);
}

// dense 1-D index array of the given integer type on the device
bool index_array(const at::Tensor& t, int device, at::ScalarType type) {
  if (!t.is_cuda() || t.device().index() != device || t.dim() != 1 || t.scalar_type() != type) return false;
  return t.sizes()[0] <= 1 || t.strides()[0] == 1;
}

// the launch goes to the current device: anything else is left to the caller's slow path
bool on_current_device(int device) {
  int cur = -1;
  return hipGetDevice(&cur) == hipSuccess && cur == device;
}

/* append_paged(key, value, batch_indices, positions, cache, kv_indices, kv_indptr,
 *              kv_last_page_len, device, stream): kvc_append_paged_kv_cache on tensors */
PyObject* fast_append_paged(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 10) {
    PyErr_SetString(PyExc_TypeError, "append_paged takes 10 arguments");
    return nullptr;
  }
  int64_t device;
  void* stream;
  if (!as_i64(args[8], &device) || !as_ptr(args[9], &stream)) return nullptr;
  const at::Tensor* t[8];
  for (int i = 0; i < 8; ++i)
    if (!(t[i] = tensor_of(args[i]))) return PyLong_FromLong(NOT_FAST);
  const at::Tensor &k = *t[0], &v = *t[1], &bi = *t[2], &pos = *t[3], &c = *t[4], &ind = *t[5],
                   &ptr = *t[6], &last = *t[7];
  const int dev = (int)device;
  if (!on_current_device(dev)) return PyLong_FromLong(NOT_FAST);
  if (!index_array(bi, dev, at::kInt) || !index_array(pos, dev, at::kInt) || !index_array(ind, dev, at::kInt) ||
      !index_array(ptr, dev, at::kInt) || !index_array(last, dev, at::kInt))
    return PyLong_FromLong(NOT_FAST);
  const int64_t nnz = bi.sizes()[0];
  if (pos.sizes()[0] != nnz || ptr.sizes()[0] < 1 || c.dim() != 5) return PyLong_FromLong(NOT_FAST);
  const auto cs = c.sizes();
  const int64_t page_size = cs[2], heads = cs[3], dim = cs[4], row = heads * dim;
  const int dtype = (int)c.scalar_type();
  int64_t num_pages = 0;
  const int64_t ps = page_stride(c, page_size, heads, dim, dtype, dev, &num_pages);
  const int64_t ks = row_stride_at_least(k, nnz, row, dtype, dev);
  const int64_t vs = row_stride_at_least(v, nnz, row, dtype, dev);
  if (ps < 0 || ks < 0 || vs < 0 || nnz == 0 || row == 0) return PyLong_FromLong(NOT_FAST);
  return PyLong_FromLong(kvc_append_paged_kv_cache(
      k.data_ptr(), v.data_ptr(), (const int32_t*)bi.data_ptr(), (const int32_t*)pos.data_ptr(),
      c.data_ptr(), (const int32_t*)ind.data_ptr(), (const int32_t*)ptr.data_ptr(),
      (const int32_t*)last.data_ptr(), nnz, ptr.sizes()[0] - 1, ind.sizes()[0], heads, dim, page_size,
      ks, vs, ps, num_pages, (int)c.element_size(), stream));
}

/* reshape_and_cache(key, value, cache, slot_mapping, device, stream): kvc_reshape_and_cache
 * on one layer of the interleaved pool, [num_blocks, 2, block_size, H, D] */
PyObject* fast_reshape_and_cache(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 6) {
    PyErr_SetString(PyExc_TypeError, "reshape_and_cache takes 6 arguments");
    return nullptr;
  }
  int64_t device;
  void* stream;
  if (!as_i64(args[4], &device) || !as_ptr(args[5], &stream)) return nullptr;
  const at::Tensor* k = tensor_of(args[0]);
  const at::Tensor* v = tensor_of(args[1]);
  const at::Tensor* c = tensor_of(args[2]);
  const at::Tensor* sl = tensor_of(args[3]);
  if (!k || !v || !c || !sl) return PyLong_FromLong(NOT_FAST);
  const int dev = (int)device;
  if (!on_current_device(dev) || c->dim() != 5) return PyLong_FromLong(NOT_FAST);
  const int slot_bytes = sl->scalar_type() == at::kLong ? 8 : 4;
  if (!index_array(*sl, dev, slot_bytes == 8 ? at::kLong : at::kInt)) return PyLong_FromLong(NOT_FAST);
  const int64_t n = sl->sizes()[0];
  const auto cs = c->sizes();
  const int64_t bs = cs[2], heads = cs[3], dim = cs[4], row = heads * dim;
  const int dtype = (int)c->scalar_type();
  int64_t num_blocks = 0;
  const int64_t stride = page_stride(*c, bs, heads, dim, dtype, dev, &num_blocks);
  const int64_t ks = row_stride(*k, n, row, dtype, dev);
  const int64_t vs = row_stride(*v, n, row, dtype, dev);
  if (stride < 0 || ks < 0 || vs < 0 || n == 0 || row == 0) return PyLong_FromLong(NOT_FAST);
  char* kc = (char*)c->data_ptr();
  return PyLong_FromLong(kvc_reshape_and_cache(k->data_ptr(), v->data_ptr(), kc,
                                               kc + bs * row * (int64_t)c->element_size(), sl->data_ptr(),
                                               slot_bytes, n, row, ks, vs, bs, stride, row, num_blocks,
                                               (int)c->element_size(), stream));
}

/* write_plan_append(plan, nnz, heads, dim, page_size, dtype, device, key, value, cache, stream) */
PyObject* fast_write_plan_append(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  void *plan, *stream;
  int64_t nnz, heads, dim, page_size, dtype, device;
  if (nargs != 11) {
    PyErr_SetString(PyExc_TypeError, "write_plan_append takes 11 arguments");
    return nullptr;
  }
  if (!as_ptr(args[0], &plan) || !as_i64(args[1], &nnz) || !as_i64(args[2], &heads) ||
      !as_i64(args[3], &dim) || !as_i64(args[4], &page_size) || !as_i64(args[5], &dtype) ||
      !as_i64(args[6], &device) || !as_ptr(args[10], &stream))
    return nullptr;
  const at::Tensor* k = tensor_of(args[7]);
  const at::Tensor* v = tensor_of(args[8]);
  const at::Tensor* c = tensor_of(args[9]);
  if (!k || !v || !c) return PyLong_FromLong(NOT_FAST);
  const int64_t row = heads * dim;
  const int64_t ks = row_stride(*k, nnz, row, (int)dtype, (int)device);
  const int64_t vs = row_stride(*v, nnz, row, (int)dtype, (int)device);
  int64_t num_pages = 0;
  const int64_t ps = page_stride(*c, page_size, heads, dim, (int)dtype, (int)device, &num_pages);
  if (ks < 0 || vs < 0 || ps < 0) return PyLong_FromLong(NOT_FAST);
  return PyLong_FromLong(kvc_write_plan_append((const kvc_write_plan*)plan, k->data_ptr(), v->data_ptr(),
                                               ks, vs, c->data_ptr(), ps, num_pages, stream));
}

/* rotary_plan_run(plan, nnz, q_heads, heads, dim, page_size, dtype, device,
 *                 query, key, value, query_out, key_out | None, cache, stream) */
PyObject* fast_rotary_plan_run(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  void *plan, *stream;
  int64_t nnz, q_heads, heads, dim, page_size, dtype, device;
  if (nargs != 15) {
    PyErr_SetString(PyExc_TypeError, "rotary_plan_run takes 15 arguments");
    return nullptr;
  }
  if (!as_ptr(args[0], &plan) || !as_i64(args[1], &nnz) || !as_i64(args[2], &q_heads) ||
      !as_i64(args[3], &heads) || !as_i64(args[4], &dim) || !as_i64(args[5], &page_size) ||
      !as_i64(args[6], &dtype) || !as_i64(args[7], &device) || !as_ptr(args[14], &stream))
    return nullptr;
  const at::Tensor* q = tensor_of(args[8]);
  const at::Tensor* k = tensor_of(args[9]);
  const at::Tensor* v = tensor_of(args[10]);
  const at::Tensor* qo = tensor_of(args[11]);
  const at::Tensor* ko = args[12] == Py_None ? nullptr : tensor_of(args[12]);
  const at::Tensor* c = tensor_of(args[13]);
  if (!q || !k || !v || !qo || !c || (args[12] != Py_None && !ko)) return PyLong_FromLong(NOT_FAST);
  const int64_t q_row = q_heads * dim, kv_row = heads * dim;
  const int dt = (int)dtype, dev = (int)device;
  const int64_t qs = row_stride(*q, nnz, q_row, dt, dev);
  const int64_t ks = row_stride(*k, nnz, kv_row, dt, dev);
  const int64_t vs = row_stride(*v, nnz, kv_row, dt, dev);
  // outputs are written with dense rows
  if (qs < 0 || ks < 0 || vs < 0 || row_stride(*qo, nnz, q_row, dt, dev) != q_row ||
      (ko && row_stride(*ko, nnz, kv_row, dt, dev) != kv_row))
    return PyLong_FromLong(NOT_FAST);
  int64_t num_pages = 0;
  const int64_t ps = page_stride(*c, page_size, heads, dim, dt, dev, &num_pages);
  if (ps < 0) return PyLong_FromLong(NOT_FAST);
  return PyLong_FromLong(kvc_rotary_plan_run((const kvc_rotary_plan*)plan, q->data_ptr(), k->data_ptr(),
                                             v->data_ptr(), qs, ks, vs, qo->data_ptr(),
                                             ko ? ko->data_ptr() : nullptr, c->data_ptr(), ps, num_pages,
                                             stream));
}

// [n, width] or [n, heads, dim] rows, dense inside a token: width and token stride, or false
bool token_rows(const at::Tensor& t, int64_t n, at::ScalarType type, int device, int64_t* width,
                int64_t* stride) {
  if (t.scalar_type() != type || (t.dim() != 2 && t.dim() != 3) || t.sizes()[0] != n) return false;
  *width = t.dim() == 2 ? t.sizes()[1] : t.sizes()[1] * t.sizes()[2];
  *stride = row_stride(t, n, *width, (int)type, device);
  return *stride >= 0;
}

int kvc_dtype_of(at::ScalarType t) {
  return t == at::kBFloat16 ? KVC_DTYPE_BF16 : t == at::kHalf ? KVC_DTYPE_F16 : t == at::kFloat ? KVC_DTYPE_F32 : -1;
}

// cos/sin table [max_position, 2 * rotary_dim], contiguous
bool cos_sin_table(const at::Tensor& cs, at::ScalarType type, int device) {
  return cs.is_cuda() && cs.device().index() == device && cs.scalar_type() == type && cs.dim() == 2 &&
         cs.sizes()[1] % 2 == 0 && cs.strides()[1] == 1 && (cs.sizes()[0] <= 1 || cs.strides()[0] == cs.sizes()[1]);
}

// A dense, uninitialised tensor of a tensor's shape, type and device.
at::Tensor dense_like(const at::Tensor& t) {
  return at::empty(t.sizes(), at::TensorOptions().dtype(t.scalar_type()).device(t.device()));
}

/* rotary_pos_emb(query, key, positions, cos_sin_cache, head_dim, device, stream) -> 1, a negative kvc_status, or
 * (query_out, key_out): kvc_rotary_pos_emb on tensors into new dense ones (allocated here: through the interpreter
 * a call takes 9.5 us, so 5.0) */
PyObject* fast_rotary_pos_emb(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS  // an allocation that fails is a Python exception
  if (nargs != 7) {
    PyErr_SetString(PyExc_TypeError, "rotary_pos_emb takes 7 arguments");
    return nullptr;
  }
  int64_t head_dim, device;
  void* stream;
  if (!as_i64(args[4], &head_dim) || !as_i64(args[5], &device) || !as_ptr(args[6], &stream)) return nullptr;
  const at::Tensor* q = tensor_of(args[0]);
  const at::Tensor* k = tensor_of(args[1]);
  const at::Tensor* pos = tensor_of(args[2]);
  const at::Tensor* cs = tensor_of(args[3]);
  if (!q || !k || !pos || !cs || head_dim <= 0) return PyLong_FromLong(NOT_FAST);
  const int dev = (int)device;
  const at::ScalarType type = q->scalar_type();
  const int kd = kvc_dtype_of(type);
  if (kd < 0 || !on_current_device(dev) || !cos_sin_table(*cs, type, dev)) return PyLong_FromLong(NOT_FAST);
  const bool pos64 = pos->scalar_type() == at::kLong;
  if (!index_array(*pos, dev, pos64 ? at::kLong : at::kInt)) return PyLong_FromLong(NOT_FAST);
  const int64_t n = pos->sizes()[0];
  int64_t qw, qs, kw, ks;
  if (n == 0 || !token_rows(*q, n, type, dev, &qw, &qs) || !token_rows(*k, n, type, dev, &kw, &ks) ||
      qw % head_dim || kw % head_dim)
    return PyLong_FromLong(NOT_FAST);
  at::Tensor qo, ko;
  {
    pybind11::gil_scoped_release no_lock;  // the allocator may wait
    qo = dense_like(*q);
    ko = dense_like(*k);
  }
  const int rc = kvc_rotary_pos_emb(q->data_ptr(), k->data_ptr(), pos->data_ptr(), pos64 ? 8 : 4, cs->data_ptr(),
                                    cs->sizes()[0], n, qw / head_dim, kw / head_dim, head_dim, cs->sizes()[1] / 2, qs,
                                    ks, qo.data_ptr(), ko.data_ptr(), qw, kw, kd, stream);
  if (rc < 0) return PyLong_FromLong(rc);
  return Py_BuildValue("(NN)", THPVariable_Wrap(std::move(qo)), THPVariable_Wrap(std::move(ko)));
  END_HANDLE_TH_ERRORS
}

/* rotary_append_paged(query, key, value, batch_indices, positions, cos_sin_cache, head_dim, cache,
 *                     kv_indices, kv_indptr, kv_last_page_len, query_out, key_out | None, device, stream):
 * kvc_rotary_pos_emb_and_append_paged on tensors */
PyObject* fast_rotary_append_paged(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 15) {
    PyErr_SetString(PyExc_TypeError, "rotary_append_paged takes 15 arguments");
    return nullptr;
  }
  int64_t head_dim, device;
  void* stream;
  if (!as_i64(args[6], &head_dim) || !as_i64(args[13], &device) || !as_ptr(args[14], &stream)) return nullptr;
  const at::Tensor* q = tensor_of(args[0]);
  const at::Tensor* k = tensor_of(args[1]);
  const at::Tensor* v = tensor_of(args[2]);
  const at::Tensor* bi = tensor_of(args[3]);
  const at::Tensor* pos = tensor_of(args[4]);
  const at::Tensor* cs = tensor_of(args[5]);
  const at::Tensor* c = tensor_of(args[7]);
  const at::Tensor* ind = tensor_of(args[8]);
  const at::Tensor* ptr = tensor_of(args[9]);
  const at::Tensor* last = tensor_of(args[10]);
  const at::Tensor* qo = tensor_of(args[11]);
  const at::Tensor* ko = args[12] == Py_None ? nullptr : tensor_of(args[12]);
  if (!q || !k || !v || !bi || !pos || !cs || !c || !ind || !ptr || !last || !qo ||
      (args[12] != Py_None && !ko) || head_dim <= 0)
    return PyLong_FromLong(NOT_FAST);
  const int dev = (int)device;
  const at::ScalarType type = q->scalar_type();
  const int kd = kvc_dtype_of(type);
  if (kd < 0 || !on_current_device(dev) || !cos_sin_table(*cs, type, dev)) return PyLong_FromLong(NOT_FAST);
  if (!index_array(*bi, dev, at::kInt) || !index_array(*pos, dev, at::kInt) || !index_array(*ind, dev, at::kInt) ||
      !index_array(*ptr, dev, at::kInt) || !index_array(*last, dev, at::kInt) || ptr->sizes()[0] < 1)
    return PyLong_FromLong(NOT_FAST);
  const int64_t n = pos->sizes()[0];
  if (n == 0 || bi->sizes()[0] != n || c->dim() != 5 || c->sizes()[4] != head_dim) return PyLong_FromLong(NOT_FAST);
  const int64_t page_size = c->sizes()[2], heads = c->sizes()[3], row = heads * head_dim;
  int64_t num_pages = 0;
  const int64_t ps = page_stride(*c, page_size, heads, head_dim, (int)type, dev, &num_pages);
  int64_t qw, qs, kw, ks, vw, vs, ow, os;
  if (ps < 0 || !token_rows(*q, n, type, dev, &qw, &qs) || !token_rows(*k, n, type, dev, &kw, &ks) ||
      !token_rows(*v, n, type, dev, &vw, &vs) || qw % head_dim || kw != row || vw != row)
    return PyLong_FromLong(NOT_FAST);
  if (!token_rows(*qo, n, type, dev, &ow, &os) || ow != qw || os != qw) return PyLong_FromLong(NOT_FAST);
  if (ko && (!token_rows(*ko, n, type, dev, &ow, &os) || ow != kw || os != kw)) return PyLong_FromLong(NOT_FAST);
  return PyLong_FromLong(kvc_rotary_pos_emb_and_append_paged(
      q->data_ptr(), k->data_ptr(), v->data_ptr(), (const int32_t*)bi->data_ptr(),
      (const int32_t*)pos->data_ptr(), cs->data_ptr(), cs->sizes()[0], n, qw / head_dim, heads, head_dim,
      cs->sizes()[1] / 2, qs, ks, vs, qo->data_ptr(), ko ? ko->data_ptr() : nullptr, qw, row, c->data_ptr(),
      (const int32_t*)ind->data_ptr(), (const int32_t*)ptr->data_ptr(), ptr->sizes()[0] - 1,
      ind->sizes()[0], page_size, ps, num_pages, kd, stream));
}

// ---- a step's requests, read where the scheduler's objects lie ---------------------------
// The interpreter's own way over a batch of 256 requests with 34 000 block ids (attribute
// reads, list concatenation, struct.pack, an array copy) takes 215 us; reading the integers
// straight into the pinned buffer the index kernel reads takes about a third of that.
struct Requests {
  struct One {
    int64_t input_len, context_len, num_ids;
    PyObject* ids;  // owned: a list or tuple
    int64_t filled_len;  // where asked for
  };
  std::vector<One> in_order;     // by decreasing input_len, stable
  std::vector<int64_t> order;    // their places in the caller's list
  int64_t tokens = 0, ids = 0, prefill_tokens = 0;
  ~Requests() {
    for (const One& r : in_order) Py_XDECREF(r.ids);
  }
};

// An int of one digit (30 bits) is read in place: a step of 34 000 block ids 181 -> 158 us. A subclass may convert
// to something else than it stores.
inline bool int_of(PyObject* o, int64_t* out) {
  if (!PyLong_CheckExact(o)) return false;
#if PY_VERSION_HEX >= 0x030C0000
  if (PyUnstable_Long_IsCompact((PyLongObject*)o)) {
    *out = PyUnstable_Long_CompactValue((PyLongObject*)o);
    return true;
  }
#else
  const Py_ssize_t digits = Py_SIZE(o);
  if (digits == 0 || digits == 1) {
    *out = digits ? (int64_t)((PyLongObject*)o)->ob_digit[0] : 0;
    return true;
  }
#endif
  int overflow = 0;
  *out = PyLong_AsLongLongAndOverflow(o, &overflow);
  return !overflow && !(*out == -1 && PyErr_Occurred());
}

bool int_attr(PyObject* o, PyObject* name, int64_t* out) {
  PyObject* v = PyObject_GetAttr(o, name);
  if (!v) return false;
  const bool ok = int_of(v, out);
  Py_DECREF(v);
  return ok;
}

// Sequences whose storage is what reading them gives; a subclass may map or load its elements on the way.
bool plain_sequence(PyObject* o) { return PyList_CheckExact(o) || PyTuple_CheckExact(o); }

// False (no Python error set) when the requests are anything but a list or tuple of objects
// with int input_len and context_len and a list or tuple block_ids, none of them of a
// subclass: the caller's own path then reads them, or says why not.
bool read_requests(PyObject* inputs, Requests* out, bool with_filled = false) {
  static PyObject* const s_input = PyUnicode_InternFromString("input_len");
  static PyObject* const s_context = PyUnicode_InternFromString("context_len");
  static PyObject* const s_ids = PyUnicode_InternFromString("block_ids");
  static PyObject* const s_filled = PyUnicode_InternFromString("filled_token_len");
  if (!plain_sequence(inputs)) return false;
  const Py_ssize_t n = PySequence_Fast_GET_SIZE(inputs);
  out->in_order.reserve(n);
  bool sorted = true;
  for (Py_ssize_t i = 0; i < n; ++i) {
    if (PySequence_Fast_GET_SIZE(inputs) != n) return false;  // an attribute that is a property may run anything
    PyObject* r = PySequence_Fast_GET_ITEM(inputs, i);
    Requests::One one{0, 0, 0, nullptr, 0};
    Py_INCREF(r);
    if (int_attr(r, s_input, &one.input_len) && int_attr(r, s_context, &one.context_len) &&
        (!with_filled || int_attr(r, s_filled, &one.filled_len)))
      one.ids = PyObject_GetAttr(r, s_ids);
    Py_DECREF(r);
    if (!one.ids || !plain_sequence(one.ids)) {
      Py_XDECREF(one.ids);
      PyErr_Clear();
      return false;
    }
    one.num_ids = PySequence_Fast_GET_SIZE(one.ids);
    out->in_order.push_back(one);
    if (one.input_len < 0 || one.input_len > INT32_MAX || one.context_len < INT32_MIN || one.context_len > INT32_MAX)
      return false;
    out->tokens += one.input_len;
    out->ids += one.num_ids;
    if (one.input_len > 1) out->prefill_tokens += one.input_len;
    if (i > 0 && one.input_len > out->in_order[i - 1].input_len) sorted = false;
  }
  out->order.resize(n);
  for (Py_ssize_t i = 0; i < n; ++i) out->order[i] = i;
  if (!sorted) {
    const std::vector<Requests::One> was = out->in_order;
    std::stable_sort(out->order.begin(), out->order.end(),
                     [&](int64_t x, int64_t y) { return was[x].input_len > was[y].input_len; });
    for (Py_ssize_t i = 0; i < n; ++i) out->in_order[i] = was[out->order[i]];
  }
  return out->tokens <= INT32_MAX && out->ids <= INT32_MAX;
}

// The block ids of a list or tuple as int32; false where one is no int or does not fit.
bool copy_ids(PyObject* seq, int64_t n, int32_t* dst) {
  if (PySequence_Fast_GET_SIZE(seq) != n) return false;
  PyObject** items = PySequence_Fast_ITEMS(seq);
  for (int64_t i = 0; i < n; ++i) {
    int64_t v;
    if (!int_of(items[i], &v)) {
      PyErr_Clear();
      return false;
    }
    if (v < INT32_MIN || v > INT32_MAX) return false;
    dst[i] = (int32_t)v;
  }
  return true;
}

// input_lens | context_lens | num_blocks, `stride` words each, then the tables at `ids_at`
bool pack_requests(const Requests& q, int64_t stride, int64_t ids_at, int32_t* dst) {
  int64_t at = ids_at, b = 0;
  for (const Requests::One& r : q.in_order) {
    dst[b] = (int32_t)r.input_len;
    dst[stride + b] = (int32_t)r.context_len;
    dst[2 * stride + b] = (int32_t)r.num_ids;
    if (!copy_ids(r.ids, r.num_ids, dst + at)) return false;
    at += r.num_ids;
    ++b;
  }
  for (; b < stride; ++b) dst[b] = dst[stride + b] = dst[2 * stride + b] = 0;  // padding: no new tokens
  for (; at % 4; ++at) dst[at] = 0;
  return true;
}

// Bytes of a step that go through the staging ring (4 million block ids): its buffers keep the size they have grown
// to, here 16 MiB each. The callers' own paths take larger ones.
constexpr int64_t kStagingMost = (int64_t(16) << 20) - 4096;

// A staging buffer, without the interpreter's lock: where the device is far behind this waits for one, and what
// the device waits for may be another thread's work. KVC_ERR_STAGING: there is no pinned memory for it, and the
// callers' own paths need none.
int acquire_staging(int64_t bytes, void** out) {
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = kvc_staging_acquire(bytes, out);
  Py_END_ALLOW_THREADS
  return rc;
}

bool stream_is_capturing(void* stream) {
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  return hipStreamIsCapturing((hipStream_t)stream, &status) != hipSuccess || status != hipStreamCaptureStatusNone;
}

// `n` elements of `type` at byte `offset` of the storage of `of`, as a tensor of its own
PyObject* piece(const at::Tensor& of, at::ScalarType type, int64_t n, int64_t offset) {
  auto impl = c10::make_intrusive<c10::TensorImpl>(c10::Storage(of.storage()), of.key_set(), c10::scalarTypeToTypeMeta(type));
  impl->set_storage_offset(offset / (int64_t)c10::elementSize(type));
  impl->set_sizes_contiguous({n});
  return THPVariable_Wrap(at::Tensor(std::move(impl)));
}

// An uninitialised buffer of whole 8-byte words on the device; the allocator may wait, so without the lock.
at::Tensor device_bytes(int64_t bytes, int device) {
  at::Tensor t;
  pybind11::gil_scoped_release no_lock;
  t = at::empty({bytes / 8}, at::TensorOptions().dtype(at::kLong).device(at::kCUDA, (c10::DeviceIndex)device));
  return t;
}

/* build_index(requests, page_size, with_slots, device, stream) -> 1, or (cu_seqlens_q, kv_indptr,
 * kv_last_page_len, kv_indices, batch_indices, positions, slot_mapping | None, prefill tokens):
 * requests packed into a staging buffer, kvc_build_write_index_staged into one allocation */
PyObject* fast_build_index(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS  // an allocation that fails is a Python exception
  int64_t page_size, with_slots, device;
  void* stream;
  if (nargs != 5) {
    PyErr_SetString(PyExc_TypeError, "build_index takes 5 arguments");
    return nullptr;
  }
  if (!as_i64(args[1], &page_size) || !as_i64(args[2], &with_slots) || !as_i64(args[3], &device) ||
      !as_ptr(args[4], &stream))
    return nullptr;
  Requests q;
  if (page_size <= 0 || !on_current_device((int)device) || stream_is_capturing(stream) ||
      !read_requests(args[0], &q) || q.in_order.empty())
    return PyLong_FromLong(NOT_FAST);
  const int64_t B = (int64_t)q.in_order.size(), N = q.ids, T = q.tokens;
  const int64_t ids_at = (3 * B + 3) / 4 * 4;
  if ((ids_at + N + 4) * 4 > kStagingMost) return PyLong_FromLong(NOT_FAST);
  void* staged = nullptr;
  int rc = acquire_staging((ids_at + N + 4) * 4, &staged);
  if (rc < 0) return PyLong_FromLong(rc == KVC_ERR_STAGING ? NOT_FAST : rc);
  if (!pack_requests(q, B, ids_at, (int32_t*)staged)) return PyLong_FromLong(NOT_FAST);
  // one allocation, every piece 16-byte aligned: slots first (8 bytes an element), then int32 pieces
  const auto up = [](int64_t bytes) { return (bytes + 15) / 16 * 16; };
  const int64_t o_cu = with_slots ? up(8 * T) : 0, o_ptr = o_cu + up(4 * (B + 1)), o_last = o_ptr + up(4 * (B + 1)),
                o_ids = o_last + up(4 * B), o_bi = o_ids + up(4 * N), o_pos = o_bi + up(4 * T), end = o_pos + up(4 * T);
  const at::Tensor buf = device_bytes(end, (int)device);
  char* p = (char*)buf.data_ptr();
  rc = kvc_build_write_index_staged(B, N, page_size, T, (int32_t*)(p + o_cu), (int32_t*)(p + o_ptr),
                                    (int32_t*)(p + o_last), (int32_t*)(p + o_ids), (int32_t*)(p + o_bi),
                                    (int32_t*)(p + o_pos), with_slots ? (int64_t*)p : nullptr, stream);
  if (rc < 0) return PyLong_FromLong(rc);
  PyObject* slots;
  if (with_slots) slots = piece(buf, at::kLong, T, 0);
  else Py_INCREF(slots = Py_None);
  return Py_BuildValue("(NNNNNNNL)", piece(buf, at::kInt, B + 1, o_cu), piece(buf, at::kInt, B + 1, o_ptr),
                       piece(buf, at::kInt, B, o_last), piece(buf, at::kInt, N, o_ids), piece(buf, at::kInt, T, o_bi),
                       piece(buf, at::kInt, T, o_pos), slots, (long long)q.prefill_tokens);
  END_HANDLE_TH_ERRORS
}

/* host_index(requests, page_size) -> 1, or (position_ids, cu_seqlens_q, prefill tokens, kv_indices, kv_indptr,
 * kv_last_page_len, batch_indices, positions, slots, order): the index arrays of a step as bytearrays of int32
 * (slots: int64). 1 also where a request is inconsistent: the caller's own path names it. */
PyObject* fast_host_index(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS  // an allocation that fails is a Python exception
  if (nargs != 2) {
    PyErr_SetString(PyExc_TypeError, "host_index takes 2 arguments");
    return nullptr;
  }
  int64_t page_size;
  if (!int_of(args[1], &page_size) || page_size <= 0 || page_size > INT32_MAX) return PyLong_FromLong(NOT_FAST);
  Requests q;
  if (!read_requests(args[0], &q, true) || q.tokens == 0 || q.ids == 0) return PyLong_FromLong(NOT_FAST);
  for (const Requests::One& r : q.in_order)
    if (r.filled_len < 0 || r.context_len - r.filled_len != r.input_len ||
        r.num_ids < (r.context_len + page_size - 1) / page_size)
      return PyLong_FromLong(NOT_FAST);
  const int64_t B = (int64_t)q.in_order.size(), T = q.tokens;
  const int64_t bytes[8] = {4 * T, 4 * (B + 1), 4 * q.ids, 4 * (B + 1), 4 * B, 4 * T, 4 * T, 8 * T};
  PyObject* out[9] = {};  // eight arrays, then the order
  bool ok = true;
  for (int i = 0; i < 8 && ok; ++i) ok = (out[i] = PyByteArray_FromStringAndSize(nullptr, bytes[i]));
  if (ok) ok = (out[8] = PyList_New(B));
  bool read = ok;
  if (ok) {
    const auto words = [&](int i) { return (int32_t*)PyByteArray_AS_STRING(out[i]); };
    int32_t *pos = words(0), *cu = words(1), *ids = words(2), *ptr = words(3), *last = words(4), *bi = words(5);
    int64_t* slots = (int64_t*)PyByteArray_AS_STRING(out[7]);
    int64_t t = 0, at = 0;
    cu[0] = ptr[0] = 0;
    for (int64_t b = 0; b < B && read; ++b) {
      const Requests::One& r = q.in_order[b];
      if (!(read = copy_ids(r.ids, r.num_ids, ids + at))) break;
      const int64_t from = t;
      for (int64_t p = r.filled_len; p < r.context_len;) {
        const int64_t page = p / page_size, end = std::min(r.context_len, (page + 1) * page_size);
        for (int64_t slot = ids[at + page] * page_size + p % page_size; p < end; ++p, ++t) {
          pos[t] = (int32_t)p;
          bi[t] = (int32_t)b;
          slots[t] = slot++;
        }
      }
      cu[b + 1] = cu[b] + (int32_t)(t - from);
      at += r.num_ids;
      ptr[b + 1] = (int32_t)at;
      // of an empty request, (0 - 1) mod page_size + 1
      last[b] = (int32_t)(r.context_len ? (r.context_len - 1) % page_size + 1 : page_size);
    }
    if (read) memcpy(PyByteArray_AS_STRING(out[6]), pos, (size_t)bytes[6]);
    for (int64_t b = 0; b < B && ok; ++b) {
      PyObject* o = PyLong_FromLongLong(q.order[b]);
      if (!(ok = o != nullptr)) break;
      PyList_SET_ITEM(out[8], b, o);
    }
  }
  if (!ok || !read) {
    for (PyObject* o : out) Py_XDECREF(o);
    return ok ? PyLong_FromLong(NOT_FAST) : nullptr;
  }
  return Py_BuildValue("(NNLNNNNNNN)", out[0], out[1], (long long)q.prefill_tokens, out[2], out[3], out[4], out[5],
                       out[6], out[7], out[8]);
  END_HANDLE_TH_ERRORS
}

constexpr int64_t kUploadMost = 4 << 20;  // bytes of index arrays that go through the staging ring

// The dense buffer of a one-dimensional array of native integers, released with the object.
struct HostArray {
  Py_buffer view{};
  bool held = false;
  ~HostArray() {
    if (held) PyBuffer_Release(&view);
  }
  bool open(PyObject* o, Py_ssize_t itemsize) {
    if (PyObject_GetBuffer(o, &view, PyBUF_C_CONTIGUOUS | PyBUF_FORMAT) != 0) {
      PyErr_Clear();
      return false;
    }
    held = true;
    const char* f = view.format;
    return view.ndim == 1 && view.itemsize == itemsize && view.len > 0 && f && f[1] == 0 &&
           (f[0] == 'i' || f[0] == 'l' || f[0] == 'q');
  }
  int64_t size() const { return (int64_t)(view.len / view.itemsize); }
  const int32_t* words() const { return (const int32_t*)view.buf; }
};

/* upload_index(position_ids, cu_seqlens_q, kv_indices, kv_indptr, kv_last_page_len, slots | None, page_size, device,
 * stream) -> 1, a negative kvc_status, or (position_ids, cu_seqlens_q, kv_indices, kv_indptr, kv_last_page_len,
 * batch_indices, positions, slots | None) on the device, in one allocation and one launch: the arrays go through a
 * staging buffer, where a copy of each from pageable memory would wait for all work queued before it. */
PyObject* fast_upload_index(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS  // an allocation that fails is a Python exception
  int64_t page_size, device;
  void* stream;
  if (nargs != 9) {
    PyErr_SetString(PyExc_TypeError, "upload_index takes 9 arguments");
    return nullptr;
  }
  if (!as_i64(args[7], &device) || !as_ptr(args[8], &stream)) return nullptr;
  if (!int_of(args[6], &page_size) || page_size <= 0 || page_size > INT32_MAX || !on_current_device((int)device) ||
      stream_is_capturing(stream))
    return PyLong_FromLong(NOT_FAST);
  const int arrays = args[5] == Py_None ? 5 : 6;
  HostArray a[6];
  for (int i = 0; i < arrays; ++i)
    if (!a[i].open(args[i], i == 5 ? 8 : 4)) return PyLong_FromLong(NOT_FAST);
  const int64_t B = a[4].size(), T = a[1].words()[a[1].size() - 1];
  if (a[1].size() != B + 1 || a[3].size() != B + 1 || T <= 0) return PyLong_FromLong(NOT_FAST);
  const auto up = [](int64_t n) { return (n + 15) / 16 * 16; };
  int64_t at[7] = {};
  for (int i = 0; i < arrays; ++i) at[i + 1] = at[i] + up(a[i].view.len);
  // more is better off with the copy engine, and would leave the ring that large
  if (at[arrays] > kUploadMost) return PyLong_FromLong(NOT_FAST);
  const int64_t staged_bytes = at[arrays], o_bi = staged_bytes, o_pos = o_bi + up(4 * T), end = o_pos + up(4 * T);
  void* staged = nullptr;
  int rc = acquire_staging(staged_bytes, &staged);
  if (rc < 0) return PyLong_FromLong(rc == KVC_ERR_STAGING ? NOT_FAST : rc);
  for (int i = 0; i < arrays; ++i) memcpy((char*)staged + at[i], a[i].view.buf, (size_t)a[i].view.len);
  const at::Tensor buf = device_bytes(end, (int)device);
  char* p = (char*)buf.data_ptr();
  rc = kvc_staging_upload_index(p, staged_bytes, at[1], at[3], at[4], B, page_size, T, (int32_t*)(p + o_bi),
                                (int32_t*)(p + o_pos), stream);
  if (rc < 0) return PyLong_FromLong(rc);
  PyObject* slots;
  if (arrays == 6) slots = piece(buf, at::kLong, a[5].size(), at[5]);
  else Py_INCREF(slots = Py_None);
  return Py_BuildValue("(NNNNNNNN)", piece(buf, at::kInt, a[0].size(), at[0]), piece(buf, at::kInt, B + 1, at[1]),
                       piece(buf, at::kInt, a[2].size(), at[2]), piece(buf, at::kInt, B + 1, at[3]),
                       piece(buf, at::kInt, B, at[4]), piece(buf, at::kInt, T, o_bi), piece(buf, at::kInt, T, o_pos),
                       slots);
  END_HANDLE_TH_ERRORS
}

/* upload_requests(requests, max_requests, max_tokens, max_ids, dst, device, stream) -> an int (1, or a negative
 * kvc_status), or (order, requests, tokens): packed as a KVWriteStep holds them and uploaded to its buffer */
PyObject* fast_upload_requests(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS  // an allocation that fails is a Python exception
  int64_t max_requests, max_tokens, max_ids, device;
  void *dst, *stream;
  if (nargs != 7) {
    PyErr_SetString(PyExc_TypeError, "upload_requests takes 7 arguments");
    return nullptr;
  }
  if (!as_i64(args[1], &max_requests) || !as_i64(args[2], &max_tokens) || !as_i64(args[3], &max_ids) ||
      !as_ptr(args[4], &dst) || !as_i64(args[5], &device) || !as_ptr(args[6], &stream))
    return nullptr;
  Requests q;
  if (!on_current_device((int)device) || stream_is_capturing(stream) || !read_requests(args[0], &q)) return PyLong_FromLong(NOT_FAST);
  const int64_t n = (int64_t)q.in_order.size(), ids_at = 3 * max_requests;
  if (n > max_requests || q.tokens > max_tokens || q.ids > max_ids) return PyLong_FromLong(NOT_FAST);
  void* staged = nullptr;
  const int64_t bytes = (ids_at + q.ids + 3) / 4 * 16;
  if (bytes > kStagingMost) return PyLong_FromLong(NOT_FAST);
  int rc = acquire_staging(bytes, &staged);
  if (rc < 0) return PyLong_FromLong(rc == KVC_ERR_STAGING ? NOT_FAST : rc);
  if (!pack_requests(q, max_requests, ids_at, (int32_t*)staged)) return PyLong_FromLong(NOT_FAST);
  rc = kvc_staging_upload(dst, bytes, stream);
  if (rc < 0) return PyLong_FromLong(rc);
  PyObject* order = PyList_New((Py_ssize_t)q.order.size());
  if (!order) return nullptr;
  for (size_t i = 0; i < q.order.size(); ++i) PyList_SET_ITEM(order, i, PyLong_FromLongLong(q.order[i]));
  return Py_BuildValue("(NLL)", order, (long long)n, (long long)q.tokens);
  END_HANDLE_TH_ERRORS
}

/* copy_blocks(kv_caches, {src: [dst, ...]}, device, stream) -> 0, 1, or a negative kvc_status:
 * kvc_copy_blocks_host_pairs on a contiguous [L, num_blocks, ...] pool */
PyObject* fast_copy_blocks(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS  // an allocation that fails is a Python exception
  int64_t device;
  void* stream;
  if (nargs != 4) {
    PyErr_SetString(PyExc_TypeError, "copy_blocks takes 4 arguments");
    return nullptr;
  }
  if (!as_i64(args[2], &device) || !as_ptr(args[3], &stream)) return nullptr;
  const at::Tensor* c = tensor_of(args[0]);
  if (!c || !PyDict_CheckExact(args[1]) || !c->is_cuda() || c->device().index() != device || c->dim() < 2 ||
      !c->is_contiguous() || c->numel() == 0 || !on_current_device((int)device) || stream_is_capturing(stream))
    return PyLong_FromLong(NOT_FAST);
  std::vector<int64_t> pairs;
  pairs.reserve(2 * (size_t)PyDict_GET_SIZE(args[1]));
  PyObject *key, *value;
  Py_ssize_t at = 0;
  while (PyDict_Next(args[1], &at, &key, &value)) {  // nothing below runs Python code
    int64_t src, dst;
    if (!plain_sequence(value)) return PyLong_FromLong(NOT_FAST);
    const Py_ssize_t n = PySequence_Fast_GET_SIZE(value);
    for (Py_ssize_t i = 0; i < n; ++i) {
      if (!int_of(key, &src) || !int_of(PySequence_Fast_GET_ITEM(value, i), &dst)) {
        PyErr_Clear();
        return PyLong_FromLong(NOT_FAST);
      }
      pairs.push_back(src);
      pairs.push_back(dst);
    }
  }
  const int64_t n = (int64_t)pairs.size() / 2, layers = c->sizes()[0], blocks = c->sizes()[1];
  if (n == 0) return PyLong_FromLong(0);
  const int64_t layer_bytes = c->numel() / layers * (int64_t)c->element_size();
  void* const pool = c->data_ptr();
  int rc = kvc_copy_blocks_host_pairs(pool, pairs.data(), n, nullptr, layers, layer_bytes, layer_bytes / blocks, blocks,
                                      stream);
  if (rc == KVC_ERR_STAGING) {
    const at::Tensor buf =
        at::empty({2 * n}, at::TensorOptions().dtype(at::kLong).device(at::kCUDA, (c10::DeviceIndex)device));
    int64_t* const scratch = (int64_t*)buf.data_ptr();
    Py_BEGIN_ALLOW_THREADS  // may wait for a staging buffer
    rc = kvc_copy_blocks_host_pairs(pool, pairs.data(), n, scratch, layers, layer_bytes, layer_bytes / blocks, blocks,
                                    stream);
    Py_END_ALLOW_THREADS
    if (rc == KVC_ERR_STAGING) return PyLong_FromLong(NOT_FAST);
  }
  return PyLong_FromLong(rc);
  END_HANDLE_TH_ERRORS
}

/* scalar_type_code(tensor) -> the integer the two calls above compare dtypes with */
PyObject* scalar_type_code(PyObject*, PyObject* o) {
  const at::Tensor* t = tensor_of(o);
  if (!t) {
    PyErr_SetString(PyExc_TypeError, "scalar_type_code takes a tensor");
    return nullptr;
  }
  return PyLong_FromLong((long)t->scalar_type());
}

PyMethodDef methods[] = {
    {"write_plan_append", (PyCFunction)(void (*)(void))fast_write_plan_append, METH_FASTCALL,
     "kvc_write_plan_append on (key, value, cache) tensors; 0, 1 = not the fast layout, or a negative kvc_status."},
    {"rotary_plan_run", (PyCFunction)(void (*)(void))fast_rotary_plan_run, METH_FASTCALL,
     "kvc_rotary_plan_run on tensors; 0, 1 = not the fast layout, or a negative kvc_status."},
    {"append_paged", (PyCFunction)(void (*)(void))fast_append_paged, METH_FASTCALL,
     "kvc_append_paged_kv_cache on tensors; 0, 1 = not the fast layout, or a negative kvc_status."},
    {"reshape_and_cache", (PyCFunction)(void (*)(void))fast_reshape_and_cache, METH_FASTCALL,
     "kvc_reshape_and_cache on tensors; 0, 1 = not the fast layout, or a negative kvc_status."},
    {"rotary_pos_emb", (PyCFunction)(void (*)(void))fast_rotary_pos_emb, METH_FASTCALL,
     "kvc_rotary_pos_emb on tensors; 0, 1 = not the fast layout, or a negative kvc_status."},
    {"rotary_append_paged", (PyCFunction)(void (*)(void))fast_rotary_append_paged, METH_FASTCALL,
     "kvc_rotary_pos_emb_and_append_paged on tensors; 0, 1 = not the fast layout, or a negative kvc_status."},
    {"build_index", (PyCFunction)(void (*)(void))fast_build_index, METH_FASTCALL,
     "Requests -> the step's index tensors, one launch; 1 = not what it reads, or a negative kvc_status."},
    {"host_index", (PyCFunction)(void (*)(void))fast_host_index, METH_FASTCALL,
     "Requests -> the step's index arrays in host memory; 1 = not what it reads."},
    {"upload_index", (PyCFunction)(void (*)(void))fast_upload_index, METH_FASTCALL,
     "Index arrays -> device tensors; 1 = not what it reads, or a negative kvc_status."},
    {"upload_requests", (PyCFunction)(void (*)(void))fast_upload_requests, METH_FASTCALL,
     "Requests -> a KVWriteStep's packed buffer; 1 = not what it reads, or a negative kvc_status."},
    {"copy_blocks", (PyCFunction)(void (*)(void))fast_copy_blocks, METH_FASTCALL,
     "kvc_copy_blocks_host_pairs on a pool and a dict; 0, 1 = not what it reads, or a negative kvc_status."},
    {"scalar_type_code", (PyCFunction)scalar_type_code, METH_O, "Integer code of a tensor's dtype."},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_kvc_fast",
                      "Low-overhead calls into libkvcache's per-layer plan entry points.", -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__kvc_fast(void) {
  PyObject* m = PyModule_Create(&module);
  if (m && (PyModule_AddIntConstant(m, "abi_version", KVC_ABI_VERSION) < 0 ||
            PyModule_AddIntConstant(m, "interface", kInterface) < 0 ||
            PyModule_AddIntConstant(m, "NOT_FAST", NOT_FAST) < 0)) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
