// The Python layer's calls into libcie_attn.so as a CPython extension
// (cie_host.so, built next to it): tensor checks, output and workspace
// allocation and the C ABI call of one operation without interpreter work in
// between. A call through ctypes with its argument conversion, stride arrays
// and device context took 17-24 us of host time per operation, more than most
// of the kernels it launches; here it takes 4-7.
//
// Every function handles exact tensors on one GPU of supported dtypes and
// shapes, making the copies the Python functions make where a kernel cannot
// read an operand in place (misaligned rows, int64 tables, a bias of another
// type: handing those back cost the refused call on top of the Python path,
// Int8Linear of a bf16 model with its fp16 bias 18.9 -> 20.9 us at 16 x 4096 x
// 4096). It returns None for everything else, before any side effect: the
// Python function then raises or converts as the case needs. A non-zero status
// of the library comes back as an int.
//
// The library's functions are bound by address (bind), so the extension works
// with whichever build of the library the package loaded.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/core/grad_mode.h>
#include <c10/core/DeviceGuard.h>
#include <c10/util/Exception.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cmath>
#include <vector>

#include "cie_attn.h"

namespace {

struct Api {
  decltype(&cie_flash_workspace_bytes) flash_ws;
  decltype(&cie_flash_fwd_ex) flash;
  decltype(&cie_flash_paged_workspace_bytes) flash_paged_ws;
  decltype(&cie_flash_paged) flash_paged;
  decltype(&cie_paged_workspace_bytes) paged_ws;
  decltype(&cie_paged_fwd_ex) paged;
  decltype(&cie_kv_append) append;
  decltype(&cie_kv_append_rope) append_rope;
  decltype(&cie_kv_append_seq) append_seq;
  decltype(&cie_kv_gather) gather;
  decltype(&cie_int8_matmul_workspace_bytes) int8_ws;
  decltype(&cie_int8_matmul) int8;
} api;
const char* const kNames[] = {"cie_flash_workspace_bytes", "cie_flash_fwd_ex", "cie_flash_paged_workspace_bytes",
                              "cie_flash_paged", "cie_paged_workspace_bytes", "cie_paged_fwd_ex", "cie_kv_append",
                              "cie_kv_append_rope", "cie_kv_append_seq", "cie_kv_gather", "cie_int8_matmul_workspace_bytes", "cie_int8_matmul"};
constexpr size_t kFns = sizeof(kNames) / sizeof(kNames[0]);
static_assert(sizeof(Api) == kFns * sizeof(void*), "one name per function, in order");

using at::Tensor;

// The tensor behind an object that is exactly a Tensor or Parameter (no
// subclass: those may override what a call does), else nullptr.
const Tensor* tensor(PyObject* o) { return THPVariable_CheckExact(o) ? &THPVariable_Unpack(o) : nullptr; }
// The same, None allowed (*ok false when it is neither).
const Tensor* tensor_or_none(PyObject* o, bool* ok) {
  if (o == Py_None) return nullptr;
  const Tensor* t = tensor(o);
  *ok &= t != nullptr;
  return t;
}

int dtype_code(const Tensor& t) {
  return t.scalar_type() == at::kHalf ? CIE_DTYPE_F16 : t.scalar_type() == at::kBFloat16 ? CIE_DTYPE_BF16 : -1;
}
int any_code(const Tensor& t) { return t.scalar_type() == at::kFloat ? CIE_TABLE_F32 : dtype_code(t); }

bool strided(const Tensor& t) { return t.layout() == at::kStrided && !t.is_conj() && !t.is_neg(); }
bool on_gpu(const Tensor& t) { return t.is_cuda() && strided(t); }

bool head_dim_ok(int64_t D) { return D == 16 || D == 32 || D == 64 || D == 128 || D == 256; }
bool fits(int64_t x) { return x >= 0 && x <= 0x7fffffff; }

// What the kernels read in place: unit last stride, 16-byte aligned rows.
bool kernel_layout(const Tensor& t) {
  const int64_t n = t.dim();
  if (t.stride(n - 1) != 1 || (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15)) return false;
  for (int64_t i = 0; i < n - 1; ++i)
    if (t.size(i) != 1 && (t.stride(i) % 8 || t.stride(i) < 0)) return false;
  return true;
}

// t, or a contiguous copy when the kernels cannot read it in place.
Tensor laid_out(const Tensor& t) { return kernel_layout(t) ? t : t.clone(at::MemoryFormat::Contiguous); }

// Block tables, lengths and the like: int32 or int64 on the device of `like`,
// converted where the kernels need it.
bool index_ok(const Tensor* t, const Tensor& like) {
  return t && on_gpu(*t) && t->device() == like.device() && (t->scalar_type() == at::kInt || t->scalar_type() == at::kLong);
}
Tensor index32(const Tensor& t) {
  return t.scalar_type() == at::kInt && t.is_contiguous() ? t : t.to(at::kInt).contiguous();
}
const int32_t* ip(const Tensor& t) { return static_cast<const int32_t*>(t.data_ptr()); }

struct Strides {
  int64_t s[4];
  explicit Strides(const Tensor& t) {  // a size-1 dimension's stride is never multiplied: 0
    const int64_t n = t.dim();
    for (int64_t i = 0; i < n; ++i) s[i] = i < n - 1 && t.size(i) == 1 ? 0 : t.stride(i);
  }
};

struct Rope {
  const void *cos = nullptr, *sin = nullptr;
  int rows = 0, dt = 0;
  bool ok = true;
  Rope(PyObject* c, PyObject* s, int64_t D, const Tensor& like) {
    const Tensor* ct = tensor_or_none(c, &ok);
    const Tensor* st = tensor_or_none(s, &ok);
    ok = ok && (ct == nullptr) == (st == nullptr);
    if (!ok || !ct) return;
    for (const Tensor* t : {ct, st})
      ok = ok && on_gpu(*t) && t->device() == like.device() && t->dim() == 2 && t->size(1) == D / 2 &&
           t->is_contiguous() && any_code(*t) >= 0 && !(reinterpret_cast<uintptr_t>(t->data_ptr()) & 15);
    ok = ok && ct->sizes() == st->sizes() && ct->size(0) >= 1 && fits(ct->size(0)) &&
         ct->scalar_type() == st->scalar_type();
    if (!ok) return;
    cos = ct->data_ptr();
    sin = st->data_ptr();
    rows = (int)ct->size(0);
    dt = any_code(*ct);
  }
};

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

Tensor bytes_like(size_t n, const Tensor& t) { return at::empty({(int64_t)n}, t.options().dtype(at::kByte)); }

// The partial states of a launch with key splits. When memory for them is short
// the launch goes without splits, which needs none (*splits 0: the library's
// rule, 1: none).
Tensor split_workspace(size_t* nbytes, int* splits, const Tensor& like) {
  *splits = 0;
  if (!*nbytes) return Tensor();
  try {
    return bytes_like(*nbytes, like);
  } catch (const c10::OutOfMemoryError&) {
    *nbytes = 0;
    *splits = 1;
    return Tensor();
  }
}

// Runs f without the GIL (as ctypes does); f returns a status.
template <typename F>
int launch(F&& f) {
  struct Released {
    PyThreadState* s = PyEval_SaveThread();
    ~Released() { PyEval_RestoreThread(s); }
  } released;
  return f();
}

PyObject* result(int rc, const Tensor& out) { return rc ? PyLong_FromLong(rc) : THPVariable_Wrap(out); }

bool number(PyObject* o, double* v) {
  *v = PyFloat_AsDouble(o);
  if (!PyErr_Occurred()) return true;
  PyErr_Clear();
  return false;
}

// flash(q, k, v, causal, scale | None, cos | None, sin | None, q_pos0 | None, out | None)
PyObject* flash(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS  // torch's own translation: an allocator failure is torch.OutOfMemoryError
  if (n != 9) Py_RETURN_NONE;
  const Tensor *q = tensor(a[0]), *k = tensor(a[1]), *v = tensor(a[2]);
  bool ok = q && k && v;
  const Tensor* pos = tensor_or_none(a[7], &ok);
  const Tensor* o = tensor_or_none(a[8], &ok);
  if (!ok || !on_gpu(*q) || !on_gpu(*k) || !on_gpu(*v) || q->dim() != 4 || k->dim() != 4 || v->dim() != 4) Py_RETURN_NONE;
  const int dt = dtype_code(*q);
  const int64_t B = q->size(0), H = q->size(1), M = q->size(2), D = q->size(3), Hk = k->size(1), N = k->size(2);
  if (dt < 0 || k->scalar_type() != q->scalar_type() || v->scalar_type() != q->scalar_type() ||
      k->device() != q->device() || v->device() != q->device() || !head_dim_ok(D) || v->sizes() != k->sizes() ||
      k->size(0) != B || k->size(3) != D || Hk < 1 || H % Hk || !fits(B) || !fits(H) || !fits(M) || !fits(N))
    Py_RETURN_NONE;
  if (o && (!on_gpu(*o) || o->sizes() != q->sizes() || o->scalar_type() != q->scalar_type() ||
            o->device() != q->device() || !kernel_layout(*o)))
    Py_RETURN_NONE;
  const Rope rope(a[5], a[6], D, *q);
  if (!rope.ok || (pos && (!rope.cos || !on_gpu(*pos) || pos->device() != q->device() ||
                           pos->scalar_type() != at::kInt || pos->dim() != 1 || pos->size(0) != B ||
                           !pos->is_contiguous())))
    Py_RETURN_NONE;
  double scale = 1.0 / std::sqrt((double)D);
  if (a[4] != Py_None && !number(a[4], &scale)) Py_RETURN_NONE;
  const int causal = PyObject_IsTrue(a[3]);
  if (causal < 0) return nullptr;
  const c10::OptionalDeviceGuard guard(q->device());
  const Tensor out = o ? *o : at::empty({B, H, M, D}, q->options());
  size_t nbytes = api.flash_ws((int)B, (int)H, (int)Hk, (int)M, (int)N, (int)D, causal, 0);
  int splits;
  const Tensor ws = split_workspace(&nbytes, &splits, *q);
  const Tensor qc = laid_out(*q), kc = laid_out(*k), vc = laid_out(*v);
  const Strides sq(qc), sk(kc), sv(vc), so(out);
  void* stream = stream_of(*q);
  const int rc = launch([&] {
    return api.flash(qc.data_ptr(), kc.data_ptr(), vc.data_ptr(), out.data_ptr(), sq.s, sk.s, sv.s, so.s, (int)B,
                     (int)H, (int)Hk, (int)M, (int)N, (int)D, (float)scale, causal, dt, rope.cos, rope.sin, rope.rows,
                     rope.dt, pos ? static_cast<const int32_t*>(pos->data_ptr()) : nullptr, splits,
                     nbytes ? ws.data_ptr() : nullptr, nbytes, stream);
  });
  return result(rc, out);
  END_HANDLE_TH_ERRORS
}

// A launch over one layer's pools.
struct Pools {
  const Tensor *kc, *vc, *bt, *lens;  // block table and lengths as given; index32() of them for a kernel
  int64_t num_blocks = 0, block_size = 0, Hk = 0, width = 0;
  bool ok;
  Pools(PyObject* k, PyObject* v, PyObject* t, PyObject* l, const Tensor& like, int64_t B, int64_t D)
      : kc(tensor(k)), vc(tensor(v)), bt(tensor(t)), lens(tensor(l)) {
    ok = kc && vc && bt && lens;
    if (!ok) return;
    for (const Tensor* x : {kc, vc})
      ok = ok && on_gpu(*x) && x->device() == like.device() && x->dim() == 4 && x->scalar_type() == like.scalar_type() &&
           x->size(3) == D && kernel_layout(*x);
    for (const Tensor* x : {bt, lens}) ok = ok && index_ok(x, like);
    ok = ok && kc->sizes() == vc->sizes() && bt->dim() == 2 && bt->size(0) == B && lens->dim() == 1 && lens->size(0) == B;
    if (!ok) return;
    num_blocks = kc->size(0), block_size = kc->size(1), Hk = kc->size(2), width = bt->size(1);
    ok = Hk >= 1 && fits(num_blocks) && fits(block_size) && fits(Hk) && fits(width);
  }
};

// The plan of a launch (PagedPlan.data, .split, .key): none, or one built for
// exactly this launch.
struct Plan {
  const Tensor* data = nullptr;
  int split = -1;
  bool ok = true;
  Plan(PyObject* d, PyObject* s, PyObject* key, std::initializer_list<int64_t> want, const Tensor& like) {
    data = tensor_or_none(d, &ok);
    if (!ok || !data) return;
    ok = PyLong_Check(s) && PyTuple_Check(key) && PyTuple_GET_SIZE(key) == (Py_ssize_t)want.size() && on_gpu(*data) &&
         data->device() == like.device() && data->is_contiguous();
    if (!ok) return;
    split = (int)PyLong_AsLong(s);
    Py_ssize_t i = 0;
    for (int64_t w : want) {
      const int64_t x = PyLong_AsLongLong(PyTuple_GET_ITEM(key, i++));
      ok = ok && x == w;
    }
    if (PyErr_Occurred()) {
      PyErr_Clear();
      ok = false;
    }
  }
};

// Launches paged attention (kn: with the new rows appended) or, prefill, the
// prefill kernels over the pools.
int paged_launch(const Tensor& q, const Pools& P, const Tensor& out, const Rope& rope, const Plan& plan, int64_t mc,
                 double scale, int causal, const void* kn, const void* vn, const int64_t* kns, const int64_t* vns,
                 bool prefill) {
  const int B = (int)q.size(0), Hq = (int)q.size(1), Lq = (int)q.size(2), D = (int)q.size(3), dt = dtype_code(q);
  const int nb = (int)P.num_blocks, bs = (int)P.block_size, Hk = (int)P.Hk, w = (int)P.width, m = (int)mc;
  size_t nbytes = 0;
  int splits = 0;
  if (prefill) nbytes = api.flash_paged_ws(B, Hq, Hk, Lq, D, m, bs, w, 0);
  else if (!plan.data || plan.split) nbytes = api.paged_ws(B, Hq, Hk, Lq, D, m, bs, w);
  const Tensor ws = prefill ? split_workspace(&nbytes, &splits, q) : nbytes ? bytes_like(nbytes, q) : Tensor();
  const Strides sq(q), sk(*P.kc), sv(*P.vc), so(out);
  void* const wp = nbytes ? ws.data_ptr() : nullptr;
  void* stream = stream_of(q);
  // (a plan carries both)
  const Tensor bt_c = plan.data ? Tensor() : index32(*P.bt), lens_c = plan.data ? Tensor() : index32(*P.lens);
  const int32_t *bt = plan.data ? nullptr : ip(bt_c), *lens = plan.data ? nullptr : ip(lens_c);
  return launch([&] {
    if (prefill)
      return api.flash_paged(q.data_ptr(), P.kc->data_ptr(), P.vc->data_ptr(), bt, lens, out.data_ptr(), sq.s, sk.s,
                             sv.s, so.s, B, Hq, Hk, Lq, D, nb, bs, w, m, (float)scale, causal, dt, rope.cos, rope.sin,
                             rope.rows, rope.dt, splits, wp, nbytes, stream);
    return api.paged(q.data_ptr(), kn, vn, P.kc->data_ptr(), P.vc->data_ptr(), bt, lens, plan.data ? plan.data->data_ptr() : nullptr,
                     plan.data ? (size_t)plan.data->nbytes() : 0, plan.split, out.data_ptr(), wp, nbytes, sq.s, kns, vns,
                     sk.s, sv.s, so.s, B, Hq, Hk, Lq, D, nb, bs, w, m, (float)scale, causal, dt, rope.cos, rope.sin,
                     rope.rows, rope.dt, stream);
  });
}

// paged(prefill, q, k_cache, v_cache, block_tables, context_lens, causal, scale | None, max_context, cos, sin, out | None)
PyObject* paged(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 12) Py_RETURN_NONE;
  const bool prefill = a[0] == Py_True;
  const Tensor* q = tensor(a[1]);
  bool ok = q != nullptr;
  const Tensor* o = tensor_or_none(a[11], &ok);
  if (!ok || !on_gpu(*q) || q->dim() != 4 || dtype_code(*q) < 0 || !head_dim_ok(q->size(3))) Py_RETURN_NONE;
  const int64_t B = q->size(0), Hq = q->size(1), Lq = q->size(2), D = q->size(3);
  const Pools P(a[2], a[3], a[4], a[5], *q, B, D);
  const int64_t mc = PyLong_Check(a[8]) ? PyLong_AsLongLong(a[8]) : -1;
  if (!P.ok || Hq % P.Hk || !fits(mc) || !fits(B) || !fits(Hq) || !fits(Lq)) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  if (o && (!on_gpu(*o) || o->sizes() != q->sizes() || o->scalar_type() != q->scalar_type() ||
            o->device() != q->device() || !kernel_layout(*o)))
    Py_RETURN_NONE;
  const Rope rope(a[9], a[10], D, *q);
  double scale = 1.0 / std::sqrt((double)D);
  if (!rope.ok || (a[7] != Py_None && !number(a[7], &scale))) Py_RETURN_NONE;
  const int causal = PyObject_IsTrue(a[6]);
  if (causal < 0) return nullptr;
  const c10::OptionalDeviceGuard guard(q->device());
  const Tensor out = o ? *o : at::empty({B, Hq, Lq, D}, q->options());
  const int64_t none3[3] = {0, 0, 1};
  const Plan no_plan(Py_None, Py_None, Py_None, {}, *q);
  return result(paged_launch(laid_out(*q), P, out, rope, no_plan, mc, scale, causal, nullptr, nullptr, none3, none3, prefill), out);
  END_HANDLE_TH_ERRORS
}

// One layer's fused decode / verify section:
// section(q, k, v, k_cache, v_cache, block_tables, context_lens, max_context, cos, sin, plan data | None, split, key)
// with q (B, Hq, L, D), k / v (B, Hk, L, D); returns (B, L, Hq * D).
PyObject* section(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 13) Py_RETURN_NONE;
  const Tensor *q = tensor(a[0]), *k = tensor(a[1]), *v = tensor(a[2]);
  if (!q || !k || !v || !on_gpu(*q) || !on_gpu(*k) || !on_gpu(*v) || q->dim() != 4 || k->dim() != 4 ||
      v->sizes() != k->sizes() || dtype_code(*q) < 0 || !head_dim_ok(q->size(3)))
    Py_RETURN_NONE;
  const int64_t B = q->size(0), Hq = q->size(1), L = q->size(2), D = q->size(3);
  const Pools P(a[3], a[4], a[5], a[6], *q, B, D);
  const int64_t mc = PyLong_Check(a[7]) ? PyLong_AsLongLong(a[7]) : -1;
  if (!P.ok || Hq % P.Hk || !fits(mc) || !fits(B) || !fits(Hq) || !fits(L) || B * L == 0) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  for (const Tensor* t : {k, v})
    if (t->size(0) != B || t->size(1) != P.Hk || t->size(2) != L || t->size(3) != D ||
        t->scalar_type() != q->scalar_type() || t->device() != q->device())
      Py_RETURN_NONE;
  const Rope rope(a[8], a[9], D, *q);
  const Plan plan(a[10], a[11], a[12], {B, Hq, P.Hk, L, D, P.num_blocks, P.block_size, P.width, mc, 1}, *q);
  if (!rope.ok || !plan.ok) Py_RETURN_NONE;
  const c10::OptionalDeviceGuard guard(q->device());
  Tensor kv[2];
  int64_t st[2][3];  // token row b * L + i of k / v: one stride over all of them, else copied
  for (int x = 0; x < 2; ++x) {
    Tensor& t = kv[x];
    t = x ? *v : *k;
    if (!kernel_layout(t) || (B > 1 && L > 1 && t.stride(0) != L * t.stride(2)))
      t = t.transpose(1, 2).clone(at::MemoryFormat::Contiguous).transpose(1, 2);
    st[x][0] = L > 1 ? t.stride(2) : B > 1 ? t.stride(0) : 0;
    st[x][1] = P.Hk > 1 ? t.stride(1) : 0;
    st[x][2] = 1;
  }
  const Tensor rows = at::empty({B, L, Hq, D}, q->options());
  const Tensor out = rows.transpose(1, 2);
  const int rc = paged_launch(laid_out(*q), P, out, rope, plan, mc, 1.0 / std::sqrt((double)D), 1, kv[0].data_ptr(),
                              kv[1].data_ptr(), st[0], st[1], false);
  return result(rc, rows.view({B, L, Hq * D}));
  END_HANDLE_TH_ERRORS
}

// append(k_new, v_new, k_cache, v_cache, block_tables, cu_new, start, max_new, status | None, cos, sin, k_out | None);
// returns True when done.
PyObject* append(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 12) Py_RETURN_NONE;
  const Tensor *k = tensor(a[0]), *v = tensor(a[1]), *cu = tensor(a[5]);
  bool ok = k && v && cu;
  const Tensor* status = tensor_or_none(a[8], &ok);
  const Tensor* ko = tensor_or_none(a[11], &ok);
  if (!ok || !on_gpu(*k) || !on_gpu(*v) || k->dim() != 3 || v->sizes() != k->sizes() || dtype_code(*k) < 0 ||
      v->scalar_type() != k->scalar_type() || v->device() != k->device() || !kernel_layout(*k) || !kernel_layout(*v))
    Py_RETURN_NONE;
  const int64_t Hk = k->size(1), D = k->size(2), max_new = PyLong_Check(a[7]) ? PyLong_AsLongLong(a[7]) : -1;
  if (!head_dim_ok(D) || cu->dim() != 1 || cu->size(0) < 2 || !fits(max_new)) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  const int64_t B = cu->size(0) - 1, T = k->size(0);
  const Pools P(a[2], a[3], a[4], a[6], *k, B, D);
  const Rope rope(a[9], a[10], D, *k);
  if (!P.ok || P.Hk != Hk || !fits(B) || !fits(T) || !rope.ok || !index_ok(cu, *k)) Py_RETURN_NONE;
  if (status && (!on_gpu(*status) || status->device() != k->device() || status->numel() < 1 ||
                 (status->scalar_type() != at::kInt && status->scalar_type() != at::kUInt32)))
    Py_RETURN_NONE;
  if (ko && (!rope.cos || !on_gpu(*ko) || ko->sizes() != k->sizes() || ko->scalar_type() != k->scalar_type() ||
             ko->device() != k->device() || !kernel_layout(*ko)))
    Py_RETURN_NONE;
  const c10::OptionalDeviceGuard guard(k->device());
  const Strides sn(*k), sm(*v), sk(*P.kc), sv(*P.vc), so(ko ? *ko : *k);
  void* stream = stream_of(*k);
  const Tensor bt = index32(*P.bt), cu_new = index32(*cu), start = index32(*P.lens);
  uint32_t* const sp = status ? static_cast<uint32_t*>(status->data_ptr()) : nullptr;
  const int dt = dtype_code(*k);
  const int rc = launch([&] {
    if (!rope.cos)
      return api.append(k->data_ptr(), v->data_ptr(), P.kc->data_ptr(), P.vc->data_ptr(), sn.s, sm.s, sk.s, sv.s,
                        ip(bt), ip(cu_new), ip(start), sp, (int)B, (int)T, (int)max_new, (int)Hk, (int)D,
                        (int)P.num_blocks, (int)P.block_size, (int)P.width, dt, stream);
    return api.append_rope(k->data_ptr(), v->data_ptr(), P.kc->data_ptr(), P.vc->data_ptr(), sn.s, sm.s, sk.s, sv.s,
                           ip(bt), ip(cu_new), ip(start), sp, (int)B, (int)T, (int)max_new, (int)Hk, (int)D,
                           (int)P.num_blocks, (int)P.block_size, (int)P.width, dt, rope.cos, rope.sin, rope.rows,
                           rope.dt, ko ? ko->data_ptr() : nullptr, ko ? so.s : nullptr, stream);
  });
  if (rc) return PyLong_FromLong(rc);
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

// Block ids of a BlockTable's list.
bool id_list(PyObject* o, std::vector<int32_t>* ids) {
  if (!PyList_CheckExact(o)) return false;
  const Py_ssize_t n = PyList_GET_SIZE(o);
  ids->resize((size_t)n);
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject* x = PyList_GET_ITEM(o, i);
    const long long v = PyLong_CheckExact(x) ? PyLong_AsLongLong(x) : -2;
    if (v < 0 || v > 0x7fffffff) {
      PyErr_Clear();
      return false;
    }
    (*ids)[(size_t)i] = (int32_t)v;
  }
  return true;
}

// The two pools of a layer, (num_blocks, block_size, heads, D) of any element
// type, head rows of a multiple of 16 bytes, 16-byte aligned.
struct SeqPools {
  int64_t strides[6];
  int64_t head_bytes = 0;
  bool ok;
  SeqPools(const Tensor* k, const Tensor* v) {
    ok = k && v && on_gpu(*k) && on_gpu(*v) && k->dim() == 4 && k->sizes() == v->sizes() && k->device() == v->device() &&
         k->scalar_type() == v->scalar_type() && k->numel() > 0;
    if (!ok) return;
    const int64_t e = k->element_size();
    head_bytes = k->size(3) * e;
    ok = head_bytes % 16 == 0;
    for (const Tensor* t : {k, v}) {
      ok = ok && t->stride(3) == 1 && !(reinterpret_cast<uintptr_t>(t->data_ptr()) & 15);
      for (int i = 0; i < 3; ++i) {
        const int64_t st = t->size(i) == 1 ? 0 : t->stride(i) * e;
        strides[(t == v ? 3 : 0) + i] = st;
        ok = ok && st >= 0 && st % 16 == 0;
      }
      ok = ok && fits(t->size(0)) && fits(t->size(1)) && fits(t->size(2));
    }
  }
};

// A graph captured from either of the two below would replay with the block ids
// and the position of the capture: handed back, to be refused like the copies
// of the Python path.
bool capturing() {
  return c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None;
}

// append_seq(k_new, v_new, k_cache, v_cache, blocks, start): (L, heads, D) rows
// to positions start ..; True when done.
PyObject* append_seq(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 6) Py_RETURN_NONE;
  const Tensor *k = tensor(a[0]), *v = tensor(a[1]), *kc = tensor(a[2]), *vc = tensor(a[3]);
  // (the engine's 16-bit caches only, as the append through device tables)
  if (!k || !v || !on_gpu(*k) || !on_gpu(*v) || k->dim() != 3 || v->sizes() != k->sizes() || dtype_code(*k) < 0 ||
      k->size(0) < 1 || !PyLong_Check(a[5]))
    Py_RETURN_NONE;
  const SeqPools P(kc, vc);
  if (!P.ok || !head_dim_ok(k->size(2)) || kc->size(2) != k->size(1) || kc->size(3) != k->size(2) ||
      kc->device() != k->device() || v->device() != k->device() || kc->scalar_type() != k->scalar_type() ||
      v->scalar_type() != k->scalar_type() || !kernel_layout(*k) || !kernel_layout(*v))
    Py_RETURN_NONE;
  std::vector<int32_t> ids;
  if (!id_list(a[4], &ids)) Py_RETURN_NONE;
  const int64_t start = PyLong_AsLongLong(a[5]), L = k->size(0);
  if (PyErr_Occurred() || start < 0 || start + L > (int64_t)ids.size() * kc->size(1)) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  const c10::OptionalDeviceGuard guard(k->device());
  if (capturing()) Py_RETURN_NONE;
  const Strides sk(*k), sv(*v);
  const int64_t dense[4] = {2 * sk.s[0], 2 * sk.s[1], 2 * sv.s[0], 2 * sv.s[1]};
  void* stream = stream_of(*k);
  const int rc = launch([&] {
    return api.append_seq(k->data_ptr(), v->data_ptr(), kc->data_ptr(), vc->data_ptr(), dense, P.strides, ids.data(),
                          (int)ids.size(), start, L, (int)kc->size(2), P.head_bytes, (int)kc->size(0),
                          (int)kc->size(1), stream);
  });
  if (rc) return PyLong_FromLong(rc);
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

// gather(k_cache, v_cache, blocks, L): dense (L, heads, D) copies of both
PyObject* gather(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 4) Py_RETURN_NONE;
  const Tensor *kc = tensor(a[0]), *vc = tensor(a[1]);
  const SeqPools P(kc, vc);
  std::vector<int32_t> ids;
  if (!P.ok || !PyLong_Check(a[3]) || !id_list(a[2], &ids)) Py_RETURN_NONE;
  const int64_t L = PyLong_AsLongLong(a[3]);
  if ( PyErr_Occurred() || L < 1 || !fits(L) || L > (int64_t)ids.size() * kc->size(1)) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  const c10::OptionalDeviceGuard guard(kc->device());
  if (capturing()) Py_RETURN_NONE;
  const int64_t heads = kc->size(2);
  const Tensor k = at::empty({L, heads, kc->size(3)}, kc->options()), v = at::empty_like(k);
  const int64_t dense[4] = {heads * P.head_bytes, P.head_bytes, heads * P.head_bytes, P.head_bytes};
  void* stream = stream_of(*kc);
  const int rc = launch([&] {
    return api.gather(kc->data_ptr(), vc->data_ptr(), k.data_ptr(), v.data_ptr(), dense, P.strides, ids.data(),
                      (int)ids.size(), L, (int)heads, P.head_bytes, (int)kc->size(0), (int)kc->size(1), stream);
  });
  if (rc) return PyLong_FromLong(rc);
  PyObject *pk = THPVariable_Wrap(k), *pv = THPVariable_Wrap(v);
  return pk && pv ? Py_BuildValue("(NN)", pk, pv) : nullptr;
  END_HANDLE_TH_ERRORS
}

// t (rows, K) itself when its rows start 16-byte aligned (a row stride of a
// multiple of `elems` elements), else a copy with padded rows.
Tensor aligned_rows(const Tensor& t, int64_t elems) {
  const int64_t K = t.size(1);
  if (t.stride(1) == 1 && t.stride(0) % elems == 0 && t.stride(0) >= K && !(reinterpret_cast<uintptr_t>(t.data_ptr()) & 15))
    return t;
  const Tensor rows = at::empty({t.size(0), (K + elems - 1) / elems * elems}, t.options()).narrow(1, 0, K);
  rows.copy_(t);
  return rows;
}

// int8(x, w_int8, scales, bias | None)
PyObject* int8(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 4) Py_RETURN_NONE;
  const Tensor *x = tensor(a[0]), *w = tensor(a[1]), *s = tensor(a[2]);
  bool ok = x && w && s;
  const Tensor* b = tensor_or_none(a[3], &ok);
  if (!ok || !on_gpu(*x) || !on_gpu(*w) || !on_gpu(*s) || x->dim() < 1 || w->dim() != 2 || s->dim() != 1 ||
      w->scalar_type() != at::kChar || dtype_code(*x) < 0 || w->device() != x->device() || s->device() != x->device() ||
      (any_code(*s) < 0 && s->scalar_type() != at::kDouble))
    Py_RETURN_NONE;
  const int64_t N = w->size(0), K = w->size(1);
  if (K < 1 || N < 1 || x->size(-1) != K || x->numel() < 1 || s->size(0) != N || !fits(N) || !fits(K) ||
      !fits(x->numel() / K))
    Py_RETURN_NONE;
  if (b && (!on_gpu(*b) || b->dim() != 1 || b->size(0) != N || b->device() != x->device() || any_code(*b) < 0))
    Py_RETURN_NONE;
  const c10::OptionalDeviceGuard guard(x->device());
  const at::NoGradGuard no_grad;  // (the copies of a Parameter need no graph)
  const Tensor xr = aligned_rows(x->dim() == 2 ? *x : x->reshape({-1, K}), 8), wr = aligned_rows(*w, 16);
  const Tensor sr = (any_code(*s) < 0 ? s->to(at::kFloat) : *s).contiguous();
  const Tensor br = b ? b->to(x->scalar_type()).contiguous() : Tensor();
  const int64_t M = xr.size(0);
  at::DimVector shape(x->sizes().begin(), x->sizes().end());
  shape.back() = N;
  const Tensor y = at::empty(shape, x->options());
  const size_t nbytes = api.int8_ws((int)M, (int)N, (int)K);
  const Tensor ws = nbytes ? bytes_like(nbytes, *x) : Tensor();
  void* stream = stream_of(*x);
  const int rc = launch([&] {
    return api.int8(xr.data_ptr(), static_cast<const int8_t*>(wr.data_ptr()), sr.data_ptr(), b ? br.data_ptr() : nullptr,
                    y.data_ptr(), xr.stride(0), wr.stride(0), N, (int)M, (int)N, (int)K, dtype_code(*x), any_code(sr),
                    nbytes ? ws.data_ptr() : nullptr, nbytes, stream);
  });
  return result(rc, y);
  END_HANDLE_TH_ERRORS
}

// bind({name: address}): the library's entry points.
PyObject* bind(PyObject*, PyObject* d) {
  void** out = reinterpret_cast<void**>(&api);
  for (size_t i = 0; i < kFns; ++i) {
    PyObject* v = PyDict_GetItemString(d, kNames[i]);
    if (!v) return PyErr_Format(PyExc_KeyError, "%s", kNames[i]);
    out[i] = PyLong_AsVoidPtr(v);
    if (PyErr_Occurred()) return nullptr;
  }
  Py_RETURN_NONE;
}

PyObject* names(PyObject*, PyObject*) {
  PyObject* l = PyList_New(0);
  for (const char* s : kNames) {
    PyObject* u = PyUnicode_FromString(s);
    PyList_Append(l, u);
    Py_DECREF(u);
  }
  return l;
}

#define CIE_FAST(f) {#f, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {CIE_FAST(flash), CIE_FAST(paged), CIE_FAST(section), CIE_FAST(append), CIE_FAST(append_seq),
                         CIE_FAST(gather), CIE_FAST(int8),
                         {"bind", bind, METH_O, nullptr},
                         {"names", names, METH_NOARGS, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "cie_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_cie_host() { return PyModule_Create(&module); }
