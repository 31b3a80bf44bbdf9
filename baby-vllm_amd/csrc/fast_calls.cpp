// The host side of the kernel wrappers' common calls: argument checks, output and
// scratch allocation and the C-ABI call in one native function each. The Python
// wrappers spend 6 to 12 us per call on the same work (attribute reads, ctypes
// argument conversion), more than the GPU needs for a decode step's small kernels.
//
// Every function returns None for a call that is not plainly valid (other types,
// layouts, devices, shapes, tensor subclasses, empty inputs): the Python wrapper then
// runs its own checks and path, so what is accepted, what is refused and with which
// error stays in one place. A call is declined only before the library is called: a
// code the library returns raises here, since the kernel may have run and the in-place
// ones must not run twice. Nothing is kept between calls. The GIL is released
// around allocation and launch, as ctypes and torch's own bindings do.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/pybind.h>

#include <ATen/ops/empty.h>
#include <ATen/ops/empty_like.h>

#include <cstdint>
#include <cstdlib>
#include <cstring>

#include "../../include/babyvllm_amd.h"

namespace {

// C-ABI entry points, bound once by the loader from the library it opened.
struct Entry {
  decltype(&bvllm_rope_kv_append) rope = nullptr;
  decltype(&bvllm_decode_workspace_bytes) decode_bytes = nullptr;
  decltype(&bvllm_paged_decode) decode = nullptr;
  decltype(&bvllm_decode_balanced_workspace_bytes) balanced_bytes = nullptr;
  decltype(&bvllm_paged_decode_balanced) balanced = nullptr;
  decltype(&bvllm_paged_prefill) prefill = nullptr;
  decltype(&bvllm_prefill_split_tiles) split_tiles = nullptr;
  decltype(&bvllm_prefill_balance_rows) balance_rows = nullptr;
  decltype(&bvllm_prefill_ranges) ranges = nullptr;
  decltype(&bvllm_prefill_workspace_bytes) prefill_bytes = nullptr;
  decltype(&bvllm_paged_prefill_split) prefill_split = nullptr;
  decltype(&bvllm_fused_add_rms_norm) norm = nullptr;
  decltype(&bvllm_silu_mul) silu = nullptr;
  decltype(&bvllm_linear_workspace_bytes) linear_bytes = nullptr;
  decltype(&bvllm_linear) linear = nullptr;
} g;

struct BindName {
  const char* name;
  void** slot;
};
const BindName kNames[] = {
    {"bvllm_rope_kv_append", (void**)&g.rope},
    {"bvllm_decode_workspace_bytes", (void**)&g.decode_bytes},
    {"bvllm_paged_decode", (void**)&g.decode},
    {"bvllm_decode_balanced_workspace_bytes", (void**)&g.balanced_bytes},
    {"bvllm_paged_decode_balanced", (void**)&g.balanced},
    {"bvllm_paged_prefill", (void**)&g.prefill},
    {"bvllm_prefill_split_tiles", (void**)&g.split_tiles},
    {"bvllm_prefill_balance_rows", (void**)&g.balance_rows},
    {"bvllm_prefill_ranges", (void**)&g.ranges},
    {"bvllm_prefill_workspace_bytes", (void**)&g.prefill_bytes},
    {"bvllm_paged_prefill_split", (void**)&g.prefill_split},
    {"bvllm_fused_add_rms_norm", (void**)&g.norm},
    {"bvllm_silu_mul", (void**)&g.silu},
    {"bvllm_linear_workspace_bytes", (void**)&g.linear_bytes},
    {"bvllm_linear", (void**)&g.linear},
};

// The wrappers' own error for a return code (babyvllm.kernels._lib.check), bound with the addresses.
PyObject* g_check = nullptr;

PyObject* none() { Py_RETURN_NONE; }

PyObject* failed(int rc, const char* what) {
  PyObject* r = PyObject_CallFunction(g_check, "is", rc, what);
  Py_XDECREF(r);
  return PyErr_Occurred() ? nullptr : PyErr_Format(PyExc_RuntimeError, "%s failed (code %d)", what, rc);
}

// A plain tensor (or parameter) on ROCm device `dev` of type `t`, or nullptr.
const at::Tensor* plain(PyObject* o, at::ScalarType t, int64_t dev) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& x = THPVariable_Unpack(o);
  if (!x.defined() || !x.is_cuda() || x.scalar_type() != t || x.get_device() != dev || x.layout() != at::kStrided ||
      x.is_conj() || x.is_neg())
    return nullptr;
  return &x;
}

bool small(int64_t v) { return v >= 0 && v <= INT32_MAX; }

template <typename F>
PyObject* launch(const at::Tensor& out, const char* what, F&& call) {
  int rc;
  {
    pybind11::gil_scoped_release no_gil;
    rc = call();
  }
  return rc == 0 ? THPVariable_Wrap(out) : failed(rc, what);
}

at::Tensor new_empty(at::IntArrayRef sizes, const at::Tensor& like, at::ScalarType t) {
  pybind11::gil_scoped_release no_gil;
  return at::empty(sizes, like.options().dtype(t).requires_grad(false));
}

// Scratch of a launch that a form without any can stand in for: undefined where there is no
// memory for it, and the caller takes that form.
at::Tensor optional_scratch(int64_t bytes, const at::Tensor& like) {
  try {
    return new_empty({bytes / 4}, like, at::kFloat);
  } catch (const c10::OutOfMemoryError&) {
    return {};
  }
}

void* ptr(const at::Tensor& t) { return const_cast<void*>(t.const_data_ptr()); }
// What a kernel writes: a lazily cloned tensor gets its own storage here, as with data_ptr() in Python.
void* out_ptr(const at::Tensor& t) { return t.mutable_data_ptr(); }

// (input, residual | None, weight, eps, device, stream)
PyObject* fast_norm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 6) return none();
  const int64_t dev = PyLong_AsLongLong(a[4]);
  const at::Tensor* x = plain(a[0], at::kBFloat16, dev);
  if (!x || x->dim() < 1 || !x->is_contiguous() || x->numel() == 0) return none();
  const at::Tensor* res = nullptr;
  const int64_t hidden = x->size(-1), rows = x->numel() / hidden;
  if (a[1] != Py_None) {
    res = plain(a[1], at::kBFloat16, dev);
    if (!res || res->dim() < 1 || !res->is_contiguous() || res->size(-1) != hidden || res->numel() != x->numel())
      return none();
  }
  const at::Tensor* w = plain(a[2], at::kBFloat16, dev);
  const bool w32 = w == nullptr;
  if (w32) w = plain(a[2], at::kFloat, dev);
  if (!w || w->numel() != hidden || !w->is_contiguous() || !small(rows) || !small(hidden)) return none();
  const float eps = (float)PyFloat_AsDouble(a[3]);
  void* stream = PyLong_AsVoidPtr(a[5]);
  if (PyErr_Occurred()) return nullptr;
  at::Tensor out = new_empty(x->sizes(), *x, at::kBFloat16);
  return launch(out, "bvllm_fused_add_rms_norm", [&] {
    return g.norm(ptr(*x), hidden, res ? out_ptr(*res) : nullptr, res ? hidden : 0, ptr(*w), w32 ? 1 : 0, ptr(out),
                  hidden, (int32_t)rows, (int32_t)hidden, eps, stream);
  });
  END_HANDLE_TH_ERRORS
}

// (gate_up, device, stream)
PyObject* fast_silu(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 3) return none();
  const at::Tensor* x = plain(a[0], at::kBFloat16, PyLong_AsLongLong(a[1]));
  if (!x || x->dim() < 1 || !x->is_contiguous() || x->numel() == 0 || x->size(-1) % 2) return none();
  const int64_t d = x->size(-1) / 2, rows = x->numel() / (2 * d);
  void* stream = PyLong_AsVoidPtr(a[2]);
  if (PyErr_Occurred()) return nullptr;
  if (!small(d)) return none();
  std::vector<int64_t> sizes = x->sizes().vec();
  sizes.back() = d;
  at::Tensor out = new_empty(sizes, *x, at::kBFloat16);
  return launch(out, "bvllm_silu_mul", [&] { return g.silu(ptr(*x), rows, (int32_t)d, ptr(out), stream); });
  END_HANDLE_TH_ERRORS
}

// [2, NB, page, Hkv, D] whose halves share a layout with a unit last stride.
bool plain_cache(const at::Tensor* c) {
  return c && c->dim() == 5 && c->size(0) == 2 && c->stride(4) == 1 && small(c->size(1)) && small(c->size(3));
}
// The attention kernels' page size; others (0 among them, which the plan would divide by)
// are for the wrapper to refuse.
constexpr int64_t kPage = 16;
const char* v_half(const at::Tensor& c) { return (const char*)c.const_data_ptr() + c.stride(0) * 2; }

bool rows_of(const at::Tensor* t, int64_t dim) { return t && t->dim() == dim && t->stride(dim - 1) == 1; }

// (q, k, v, cos, sin, kv_cache, slot_mapping, device, stream) -> True or None
PyObject* fast_rope(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 9) return none();
  const int64_t dev = PyLong_AsLongLong(a[7]);
  const at::Tensor* t[6];
  for (int i = 0; i < 6; ++i) t[i] = plain(a[i], at::kBFloat16, dev);
  const at::Tensor *q = t[0], *k = t[1], *v = t[2], *cos = t[3], *sin = t[4], *c = t[5];
  const at::Tensor* slots = plain(a[6], at::kLong, dev);
  if (!rows_of(q, 3) || !rows_of(k, 3) || !rows_of(v, 3) || !rows_of(cos, 2) || !rows_of(sin, 2)) return none();
  const int64_t tokens = q->size(0), heads = q->size(1), d = q->size(2), hkv = k->size(1);
  if (!plain_cache(c) || !c->is_contiguous() || !slots || slots->dim() != 1 || !slots->is_contiguous()) return none();
  if (tokens == 0 || k->size(0) != tokens || k->size(2) != d || v->sizes() != k->sizes()) return none();
  if (cos->size(0) < tokens || cos->size(1) != d || sin->sizes() != cos->sizes()) return none();
  if (c->size(3) != hkv || c->size(4) != d || slots->size(0) < tokens || !small(tokens) || !small(heads)) return none();
  void* stream = PyLong_AsVoidPtr(a[8]);
  if (PyErr_Occurred()) return nullptr;
  int rc;
  {
    pybind11::gil_scoped_release no_gil;
    // The written ones first: where q and k are views of one storage, no pointer is read before it is settled.
    void *qp = out_ptr(*q), *kp = out_ptr(*k), *cp = out_ptr(*c);
    rc = g.rope(qp, q->stride(0), q->stride(1), kp, k->stride(0), k->stride(1), ptr(*v), v->stride(0), v->stride(1),
                ptr(*cos), cos->stride(0), ptr(*sin), sin->stride(0), cp, (char*)cp + c->stride(0) * 2, c->stride(2),
                c->stride(3), c->size(1) * c->size(2), slots->const_data_ptr<int64_t>(), (int32_t)tokens,
                (int32_t)heads, (int32_t)hkv, (int32_t)d, stream);
  }
  if (rc != 0) return failed(rc, "bvllm_rope_kv_append");
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

int64_t cdiv(int64_t a, int64_t b) { return a / b + (a % b > 0); }  // a >= 0: no sum to overflow
// An int of any size: past 64 bits the nearest one, which means the same for a length.
int64_t clamped(PyObject* o) {
  int overflow = 0;
  const long long v = PyLong_AsLongLongAndOverflow(o, &overflow);
  return overflow > 0 ? INT64_MAX : overflow < 0 ? INT64_MIN : v;
}
int64_t pow2_at_least(int64_t n) {
  int64_t p = 1;
  while (p < n) p <<= 1;
  return p;
}

// decode_split_plan's "auto" rules (babyvllm/kernels/decode_split.py).
struct Plan {
  int64_t splits, pages;
};
Plan auto_plan(int64_t batch, int64_t hkv, int64_t page, int64_t width, int64_t max_seq_len, int64_t cus,
               int64_t min_pages) {
  int64_t ctx = max_seq_len < 0 ? width : cdiv(max_seq_len, page);
  ctx = width >= 1 ? std::min(std::max<int64_t>(ctx, 1), width) : 1;
  const int64_t rows = pow2_at_least(batch);
  if (rows * hkv >= cus) return {1, ctx};
  const int64_t pages = std::max(min_pages, rows);
  return {cdiv(ctx, pages), pages};
}

// (batch, hkv, page, width, max_seq_len | -1, cus, min_pages) -> (splits, pages), for tests
PyObject* fast_auto_plan(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 7) return none();
  int64_t v[7];
  for (int i = 0; i < 7; ++i) v[i] = clamped(a[i]);
  if (PyErr_Occurred()) return nullptr;
  if (v[2] < 1) return none();
  const Plan p = auto_plan(v[0], v[1], v[2], v[3], v[4], v[5], v[6]);
  return Py_BuildValue("LL", (long long)p.splits, (long long)p.pages);
}

// balance_pays (babyvllm/kernels/paged_attn.py).
bool balance_pays(int64_t batch, int64_t heads, int64_t hkv, int64_t cus) {
  if (hkv < 1 || heads % hkv != 0) return false;
  return pow2_at_least(batch) * hkv * cdiv(heads / hkv, 16) <= 2 * cus;
}

// (q, kv_cache, block_tables, seq_lens, scale, max_seq_len | None, cus, min_pages, balance_min_pages,
//  partition env name, device, stream): the "auto" plan
PyObject* fast_decode(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 12) return none();
  const int64_t dev = PyLong_AsLongLong(a[10]);
  const at::Tensor* q = plain(a[0], at::kBFloat16, dev);
  const at::Tensor* c = plain(a[1], at::kBFloat16, dev);
  const at::Tensor* bt = plain(a[2], at::kInt, dev);
  const at::Tensor* lens = plain(a[3], at::kInt, dev);
  if (!rows_of(q, 3) || !plain_cache(c) || !bt || bt->dim() != 2 || bt->stride(1) != 1) return none();
  const int64_t batch = q->size(0), heads = q->size(1), d = q->size(2), hkv = c->size(3), width = bt->size(1);
  if (batch == 0 || c->size(4) != d || bt->size(0) < batch) return none();
  if (!lens || lens->dim() != 1 || lens->size(0) < batch || !lens->is_contiguous()) return none();
  if (!small(batch) || !small(heads) || !small(width) || c->size(2) != kPage) return none();
  int64_t max_seq_len = -1;
  if (a[5] != Py_None) {
    if (!PyLong_CheckExact(a[5])) return none();
    max_seq_len = std::max<int64_t>(clamped(a[5]), 0);
  }
  if (!PyFloat_CheckExact(a[4])) return none();
  const float scale = (float)PyFloat_AsDouble(a[4]);
  const int64_t cus = PyLong_AsLongLong(a[6]), min_pages = PyLong_AsLongLong(a[7]);
  const int64_t balance = PyLong_AsLongLong(a[8]);
  const char* env_name = PyUnicode_AsUTF8(a[9]);
  void* stream = PyLong_AsVoidPtr(a[11]);
  if (PyErr_Occurred()) return nullptr;
  const char* env = std::getenv(env_name);
  if (env != nullptr && std::strcmp(env, "auto") != 0) return none();
  const Plan p = auto_plan(batch, hkv, c->size(2), width, max_seq_len, cus, min_pages);
  if (!small(p.splits) || !small(p.pages)) return none();
  bool balanced = p.splits == 1 && p.pages > balance && batch * width <= BVLLM_BALANCED_MAX_PAGES &&
                  balance_pays(batch, heads, hkv, cus);
  at::Tensor out = new_empty({batch, heads, d}, *q, at::kBFloat16), ws;
  if (balanced) {
    const int64_t bytes = g.balanced_bytes((int32_t)batch, (int32_t)heads, (int32_t)hkv, (int32_t)d);
    if (bytes > 0) ws = optional_scratch(bytes, *q);
    balanced = ws.defined();
  }
  if (!balanced) {
    const int64_t bytes =
        g.decode_bytes((int32_t)batch, (int32_t)heads, (int32_t)hkv, (int32_t)d, (int32_t)p.splits, (int32_t)p.pages);
    if (bytes > 0) ws = new_empty({bytes / 4}, *q, at::kFloat);
  }
  void* wp = ws.defined() ? ptr(ws) : nullptr;
  return launch(out, "bvllm_paged_decode", [&] {
    const int32_t* tables = bt->const_data_ptr<int32_t>();
    const int32_t* l = lens->const_data_ptr<int32_t>();
    if (balanced)
      return g.balanced(ptr(*q), q->stride(0), q->stride(1), ptr(*c), v_half(*c), c->stride(1), c->stride(2),
                        c->stride(3), (int32_t)c->size(1), tables, bt->stride(0), (int32_t)width, l, scale, ptr(out),
                        out.stride(0), out.stride(1), wp, (int32_t)batch, (int32_t)heads, (int32_t)hkv, (int32_t)d,
                        (int32_t)c->size(2), stream);
    return g.decode(ptr(*q), q->stride(0), q->stride(1), ptr(*c), v_half(*c), c->stride(1), c->stride(2), c->stride(3),
                    (int32_t)c->size(1), tables, bt->stride(0), (int32_t)width, l, scale, ptr(out), out.stride(0),
                    out.stride(1), wp, (int32_t)p.splits, (int32_t)p.pages, (int32_t)batch, (int32_t)heads,
                    (int32_t)hkv, (int32_t)d, (int32_t)c->size(2), 0, stream);
  });
  END_HANDLE_TH_ERRORS
}

// (q, kv_cache, block_tables, query_start_loc, seq_lens, context_lens, qsl list, seq_lens list, max_query_len,
//  scale, split_min_pages, device, stream)
PyObject* fast_prefill(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 13) return none();
  const int64_t dev = PyLong_AsLongLong(a[11]);
  const at::Tensor* q = plain(a[0], at::kBFloat16, dev);
  const at::Tensor* c = plain(a[1], at::kBFloat16, dev);
  const at::Tensor* bt = plain(a[2], at::kInt, dev);
  const at::Tensor* qsl = plain(a[3], at::kInt, dev);
  const at::Tensor* seq = plain(a[4], at::kInt, dev);
  const at::Tensor* ctx = plain(a[5], at::kInt, dev);
  if (!rows_of(q, 3) || !plain_cache(c) || !bt || bt->dim() != 2 || bt->stride(1) != 1) return none();
  for (const at::Tensor* v : {qsl, seq, ctx})
    if (!v || v->dim() != 1 || !v->is_contiguous()) return none();
  const int64_t tokens = q->size(0), heads = q->size(1), d = q->size(2), hkv = c->size(3), seqs = seq->size(0);
  const int64_t width = bt->size(1);
  if (tokens == 0 || seqs == 0 || c->size(4) != d || hkv == 0 || heads % hkv != 0 || (d & (d - 1)) != 0) return none();
  if (qsl->size(0) != seqs + 1 || ctx->size(0) != seqs || bt->size(0) < seqs) return none();
  if (!small(tokens) || !small(heads) || !small(seqs) || !small(width) || c->size(2) != kPage) return none();
  // Host lists: single-query sequences and their pages, and the key tiles of the
  // others' blocks.
  if (!PyList_CheckExact(a[6]) || PyList_GET_SIZE(a[6]) != seqs + 1) return none();
  const bool lens_known = PyList_CheckExact(a[7]) && PyList_GET_SIZE(a[7]) == seqs;
  const int64_t split_min = PyLong_AsLongLong(a[10]);
  int64_t single = 0, tiles = lens_known ? 0 : -1, prev = 0, longest = 0, pages = 0;
  int64_t longest_tiles = tiles;
  for (int64_t i = 0; i <= seqs; ++i) {
    PyObject* o = PyList_GET_ITEM(a[6], i);
    if (!PyLong_CheckExact(o)) return none();
    const int64_t v = clamped(o);
    if (!small(v)) return none();
    if (i > 0) {
      const int64_t m = v - prev;
      single += m == 1;
      if (lens_known) {
        PyObject* l = PyList_GET_ITEM(a[7], i - 1);
        if (!PyLong_CheckExact(l)) return none();
        const int64_t len = clamped(l);
        if (!small(m) || !small(len)) return none();
        if (m == 1) {
          longest = std::max(longest, cdiv(len, 16));
          pages += cdiv(len, 16);
        } else if (m > 1) {
          tiles += cdiv(m * (heads / hkv), 128) * cdiv(len, 64);
          longest_tiles = std::max(longest_tiles, cdiv(len, 64));
        }
      }
    }
    prev = v;
  }
  if (!PyLong_CheckExact(a[8]) || !PyFloat_CheckExact(a[9])) return none();
  const int64_t max_q = clamped(a[8]);
  const float scale = (float)PyFloat_AsDouble(a[9]);
  void* stream = PyLong_AsVoidPtr(a[12]);
  if (PyErr_Occurred()) return nullptr;
  if (!small(max_q)) return none();
  int32_t split = width < split_min ? 0
                                    : g.split_tiles((int32_t)seqs, (int32_t)tokens, (int32_t)max_q, (int32_t)single,
                                                    (int32_t)heads, (int32_t)hkv, (int32_t)d, (int32_t)width, tiles,
                                                    longest_tiles);
  int32_t balance = 0;
  if (pages > 0 && seqs * width <= BVLLM_BALANCED_MAX_PAGES)
    balance = g.balance_rows((int32_t)heads, (int32_t)hkv, longest, pages,
                             split > 0 ? std::min<int64_t>(split, longest_tiles) : longest_tiles);
  const int32_t ranges = split > 0 ? g.ranges((int32_t)width, split, longest_tiles) : 0;
  at::Tensor out = new_empty({tokens, heads, d}, *q, at::kBFloat16), ws;
  if (split > 0 || balance) {
    ws = optional_scratch(g.prefill_bytes((int32_t)seqs, (int32_t)tokens, (int32_t)heads, (int32_t)hkv, (int32_t)d,
                                          ranges, balance),
                          *q);
    if (!ws.defined()) split = balance = 0;
  }
  return launch(out, "bvllm_paged_prefill", [&] {
    const int32_t *tables = bt->const_data_ptr<int32_t>(), *ql = qsl->const_data_ptr<int32_t>();
    const int32_t *sl = seq->const_data_ptr<int32_t>(), *cl = ctx->const_data_ptr<int32_t>();
    if (split > 0 || balance)
      return g.prefill_split(ptr(*q), q->stride(0), q->stride(1), ptr(*c), v_half(*c), c->stride(1), c->stride(2),
                             c->stride(3), (int32_t)c->size(1), tables, bt->stride(0), (int32_t)width, ql, sl, cl,
                             scale, ptr(out), out.stride(0), out.stride(1), (int32_t)seqs, (int32_t)tokens,
                             (int32_t)max_q, (int32_t)single, (int32_t)heads, (int32_t)hkv, (int32_t)d,
                             (int32_t)c->size(2), ptr(ws), split, ranges, balance, stream);
    return g.prefill(ptr(*q), q->stride(0), q->stride(1), ptr(*c), v_half(*c), c->stride(1), c->stride(2),
                     c->stride(3), (int32_t)c->size(1), tables, bt->stride(0), (int32_t)width, ql, sl, cl, scale,
                     ptr(out), out.stride(0), out.stride(1), (int32_t)seqs, (int32_t)tokens, (int32_t)max_q,
                     (int32_t)single, (int32_t)heads, (int32_t)hkv, (int32_t)d, (int32_t)c->size(2), stream);
  });
  END_HANDLE_TH_ERRORS
}

// (x, weight, bias | None, out | None, gated, eager, device, stream)
PyObject* fast_linear(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 8) return none();
  const int64_t dev = PyLong_AsLongLong(a[6]);
  const at::Tensor* x = plain(a[0], at::kBFloat16, dev);
  const at::Tensor* w = plain(a[1], at::kBFloat16, dev);
  const bool gated = a[4] == Py_True, eager = a[5] == Py_True;
  if (!x || !w || x->dim() != 2 || w->dim() != 2 || x->stride(1) != 1 || !w->is_contiguous()) return none();
  const int64_t m = x->size(0), k = x->size(1), rows = w->size(0), cols = gated ? rows / 2 : rows;
  if (m < 1 || w->size(1) != k || (gated && rows % 2) || !small(m) || !small(k) || !small(rows)) return none();
  const int64_t x_stride = m > 1 ? x->stride(0) : k;
  // (Rows further apart than the kernel's 32-bit offsets reach are the library's.)
  if (x_stride < k || x_stride % 8 || m * x_stride * 2 >= ((int64_t)1 << 31) || ((uintptr_t)ptr(*x) | (uintptr_t)ptr(*w)) % 16) return none();
  const at::Tensor* bias = nullptr;
  if (a[2] != Py_None) {
    bias = plain(a[2], at::kBFloat16, dev);
    if (!bias || gated || bias->dim() != 1 || bias->size(0) != cols || !bias->is_contiguous()) return none();
  }
  void* stream = PyLong_AsVoidPtr(a[7]);
  if (PyErr_Occurred()) return nullptr;
  const int64_t bytes = g.linear_bytes((int32_t)m, (int32_t)cols, (int32_t)k, gated, eager);
  if (bytes < 0) return none();
  at::Tensor out, ws;
  int64_t out_stride = cols;
  if (a[3] != Py_None) {
    const at::Tensor* o = plain(a[3], at::kBFloat16, dev);
    if (!o || o->dim() != 2 || o->size(0) != m || o->size(1) != cols || o->stride(1) != 1 || (uintptr_t)out_ptr(*o) % 8)
      return none();
    if (m > 1) out_stride = o->stride(0);
    if (out_stride < cols || out_stride % 4) return none();
    // An in-place write to autograd, as torch's out= is: what was saved of the old values is
    // stale, and an inference tensor is refused outside inference mode.
    o->unsafeGetTensorImpl()->bump_version();
    out = *o;
  } else {
    out = new_empty({m, cols}, *x, at::kBFloat16);
  }
  if (bytes > 0) {
    ws = optional_scratch(bytes, *x);
    if (!ws.defined()) return none();  // the library's
  }
  return launch(out, "bvllm_linear", [&] {
    return g.linear(ptr(*x), x_stride, ptr(*w), bias ? ptr(*bias) : nullptr, out_ptr(out), out_stride, (int32_t)m,
                    (int32_t)cols, (int32_t)k, gated, eager, bytes > 0 ? ptr(ws) : nullptr, stream);
  });
  END_HANDLE_TH_ERRORS
}

// ({name: address}, check): binds the library's entry points and what raises for a return code.
PyObject* bind(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 2 || !PyDict_Check(a[0]) || !PyCallable_Check(a[1]))
    return PyErr_Format(PyExc_TypeError, "bind({name: address}, check)");
  for (const BindName& b : kNames) {
    PyObject* v = PyDict_GetItemString(a[0], b.name);
    if (v == nullptr) return PyErr_Format(PyExc_KeyError, "no address for %s", b.name);
    *b.slot = PyLong_AsVoidPtr(v);
    if (PyErr_Occurred()) return nullptr;
  }
  Py_INCREF(a[1]);
  Py_XSETREF(g_check, a[1]);
  Py_RETURN_NONE;
}

// The entry points that bind() wants.
PyObject* names(PyObject*, PyObject*) {
  PyObject* l = PyList_New(0);
  if (!l) return nullptr;
  for (const BindName& b : kNames) {
    PyObject* s = PyUnicode_FromString(b.name);
    if (!s || PyList_Append(l, s) != 0) {
      Py_XDECREF(s);
      Py_DECREF(l);
      return nullptr;
    }
    Py_DECREF(s);
  }
  return l;
}

#define FAST(name) {#name, (PyCFunction)(void (*)(void))fast_##name, METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {
    FAST(norm), FAST(silu), FAST(rope), FAST(auto_plan), FAST(decode), FAST(prefill), FAST(linear),
    {"bind", (PyCFunction)(void (*)(void))bind, METH_FASTCALL, nullptr}, {"names", names, METH_NOARGS, nullptr}, {nullptr, nullptr, 0, nullptr},
};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_fast_calls", nullptr, -1, kMethods};

}  // namespace

// ABI_VERSION: that of the header the calls above were compiled against.
PyMODINIT_FUNC PyInit__fast_calls() {
  PyObject* m = PyModule_Create(&kModule);
  if (m != nullptr && PyModule_AddIntConstant(m, "ABI_VERSION", BVLLM_ABI_VERSION) != 0) Py_CLEAR(m);
  return m;
}
