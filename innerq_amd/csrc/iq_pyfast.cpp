// Native front of the per-token calls: the argument checks, segment structures
// and launches of ops.decode_attention, ops.qk_gemv, ops.av_gemv and
// ops.window_append for the ordinary case, without Python between them.
//
// The Python wrappers build ~40 ctypes fields and ~30 small objects per call,
// and short calls waited for them: a decode of one sequence over 1000 tokens
// took 21.7 us (15.4 through here, its kernels' time), a QK^T GEMV over 8192
// tokens 12.2 (5.0), a layer's append() + attend() at 4 x 8 heads x 500 tokens
// 72 (24).  Each function here
// returns None when anything is out of the ordinary (a shape, type, stride or
// state that the wrapper converts or refuses, a buffer that has to grow, an
// argument that the entry point refuses): no window or store has been changed
// then, and the wrapper's general path runs and decides, so results and errors
// are its own.  A failed launch (IQ_ERR_HIP, which an earlier call's error also
// gives) is raised from here as the general path raises it: the kernel may have
// run, and an append run twice would quantize the rows that it left in the
// window in place of the tokens.
//
// A CPython extension over libtorch's tensors; the kernels are entered through
// the C ABI's function addresses, handed in by bind().
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/ATen.h>

#include "../../include/innerq_abi.h"

namespace {

typedef size_t (*decode_ws_t)(int, int, int, int);
typedef int (*decode_t)(const void*, int64_t, int64_t, const void*, const iq_segment*, const iq_segment*, int, int, int,
                        int, int, float, void*, int64_t, int64_t, void*, size_t, void*);
typedef size_t (*qk_ws_t)(int, int, int);
typedef int (*qk_t)(const void*, int64_t, int64_t, const void*, const uint32_t*, const uint16_t*, int64_t, int, int,
                    int, int, int, int, int, int, int, float, float*, int64_t, int64_t, void*, size_t, void*);
typedef size_t (*av_ws_t)(int, int, int, int, int);
typedef int (*av_t)(const void*, int64_t, int64_t, const uint32_t*, const uint16_t*, int64_t, int, int, int, int, int,
                    int, int, int, int, float*, void*, int64_t, int64_t, int, void*, size_t, void*);
typedef int (*append_t)(const iq_window*, const iq_window*, int, int, int, void*);

struct Bound {
  decode_ws_t decode_ws;
  decode_t decode;
  qk_ws_t qk_ws;
  qk_t qk;
  av_ws_t av_ws;
  av_t av;
  append_t append;
  PyObject* workspaces;  // ops._WS: (device index, stream) -> uint8 tensor
  PyObject* raw_stream;  // device index -> the current stream's handle
} fn{};

PyObject *S_codes, *S_meta, *S_t_cap, *S_length, *S_bits, *S_group, *S_mode, *S_dtype, *S_axis, *S_B, *S_H, *S_D, *S_buf,
    *S_start, *S_n, *S_deq_rows, *S_shadow;

// an attribute as an integer; false (no Python error) when it is none
bool get_int(PyObject* o, PyObject* name, int64_t* v) {
  PyObject* a = PyObject_GetAttr(o, name);
  if (!a) { PyErr_Clear(); return false; }
  const bool ok = PyLong_Check(a);
  if (ok) *v = PyLong_AsLongLong(a);
  Py_DECREF(a);
  if (ok && *v == -1 && PyErr_Occurred()) { PyErr_Clear(); return false; }
  return ok;
}
// a plain device tensor (no subclass, wrapper or lazy tensor), or null
const at::Tensor* tensor_of(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || !t.has_storage() || t.layout() != at::kStrided || t.is_conj() || t.is_neg())
    return nullptr;
  return &t;
}
bool act_dtype(at::ScalarType d) { return d == at::kHalf || d == at::kBFloat16; }
int act_flag(at::ScalarType d) { return d == at::kBFloat16 ? IQ_MODE_BF16 : 0; }

// a PackedStore's fields.  The tensors are held here: while the kernels are
// enqueued another thread may run, grow the store and drop them
struct Store {
  at::Tensor codes_t, meta_t;
  const uint32_t* codes;
  uint16_t* meta;
  int64_t B, H, D, t_cap, length, bits, group, mode;
  at::ScalarType dtype;
  int device;
  bool channel;
};
bool store_of(PyObject* o, Store* s) {
  if (!get_int(o, S_B, &s->B) || !get_int(o, S_H, &s->H) || !get_int(o, S_D, &s->D) || !get_int(o, S_t_cap, &s->t_cap) ||
      !get_int(o, S_length, &s->length) || !get_int(o, S_bits, &s->bits) || !get_int(o, S_group, &s->group) ||
      !get_int(o, S_mode, &s->mode))
    return false;
  PyObject *c = PyObject_GetAttr(o, S_codes), *m = PyObject_GetAttr(o, S_meta), *d = PyObject_GetAttr(o, S_dtype),
           *ax = PyObject_GetAttr(o, S_axis);
  bool ok = c && m && d && ax && THPDtype_Check(d) && PyUnicode_Check(ax);
  if (ok) {
    const at::Tensor *ct = tensor_of(c), *mt = tensor_of(m);
    ok = ct && mt && ct->scalar_type() == at::kInt && mt->scalar_type() == at::kShort && ct->is_contiguous() &&
         mt->is_contiguous();
    if (ok) {
      s->codes_t = *ct;
      s->meta_t = *mt;
      s->codes = (const uint32_t*)ct->data_ptr();
      s->meta = (uint16_t*)mt->data_ptr();
      s->device = ct->get_device();
      s->dtype = ((THPDtype*)d)->scalar_type;
      s->channel = PyUnicode_CompareWithASCIIString(ax, "channel") == 0;
      ok = act_dtype(s->dtype);
    }
  }
  Py_XDECREF(c); Py_XDECREF(m); Py_XDECREF(d); Py_XDECREF(ax);
  if (!ok) PyErr_Clear();
  return ok;
}

bool stream_of(int device, void** stream, PyObject** key) {  // key: new reference, a (device, stream) tuple
  PyObject* d = PyLong_FromLong(device);
  PyObject* s = d ? PyObject_CallOneArg(fn.raw_stream, d) : nullptr;
  if (!s) { Py_XDECREF(d); PyErr_Clear(); return false; }
  *stream = PyLong_AsVoidPtr(s);
  *key = PyTuple_Pack(2, d, s);
  Py_DECREF(d); Py_DECREF(s);
  if (!*key || PyErr_Occurred()) { Py_XDECREF(*key); PyErr_Clear(); return false; }
  return true;
}
// the stream's workspace where it is large enough (the wrapper makes or grows
// it), held in *hold: a thread that needs a larger one replaces it
bool workspace_of(PyObject* key, size_t need, at::Tensor* hold, void** ws, size_t* bytes) {
  PyObject* w = PyDict_GetItemWithError(fn.workspaces, key);
  if (!w) { PyErr_Clear(); return false; }
  const at::Tensor* t = tensor_of(w);
  if (!t || size_t(t->numel()) < need) return false;
  *hold = *t;
  *ws = t->data_ptr();
  *bytes = size_t(t->numel());
  return true;
}

// rows [r0, r0 + n) of a dense K or V segment [B, H, >= r0 + n, D] (None: n = 0)
bool dense_segment(PyObject* o, int64_t r0, int64_t n, int64_t B, int64_t H, int64_t D, at::ScalarType dt, int device,
                   iq_segment* g) {
  g->n = 0;
  if (o == Py_None) return n <= 0;
  const at::Tensor* t = tensor_of(o);
  if (!t || t->dim() != 4 || t->size(0) != B || t->size(1) != H || t->size(3) != D || t->scalar_type() != dt ||
      t->get_device() != device)
    return false;
  if (n < 0) n = t->size(2) - r0;  // the rest
  if (r0 < 0 || n < 0 || r0 + n > t->size(2)) return false;
  g->n = int(n);
  if (!n) return true;
  if (t->stride(3) != 1) return false;
  g->mode = act_flag(dt);
  g->s_b = t->stride(0); g->s_h = t->stride(1); g->s_t = t->stride(2);
  g->dense = (const char*)t->data_ptr() + r0 * g->s_t * 2;
  return true;
}
// tokens [t0, len) of a store (its fields, and the hold on its tensors, in s)
bool packed_segment(PyObject* o, int64_t t0, int64_t len, bool channel, int64_t B, int64_t* H, int64_t D,
                    at::ScalarType dt, int device, Store& s, iq_segment* g) {
  g->n = 0;
  if (o == Py_None) return t0 == 0;
  if (!store_of(o, &s)) return false;
  if (len < 0) len = s.length;
  if (s.channel != channel || s.B != B || s.D != D || s.dtype != dt || s.device != device || (*H >= 0 && s.H != *H) ||
      t0 < 0 || t0 > len || len > s.length)
    return false;
  *H = s.H;
  g->n = int(len - t0);
  if (!g->n) return true;
  g->codes = s.codes; g->meta = s.meta; g->t_cap = s.t_cap; g->t0 = int(t0);
  g->bits = int(s.bits); g->group = int(s.group); g->mode = int(s.mode) | act_flag(dt);
  return true;
}

// norm: None, or numel values of dtype dt, contiguous
bool norm_of(PyObject* o, int64_t numel, at::ScalarType dt, int device, const void** p) {
  *p = nullptr;
  if (o == Py_None) return true;
  const at::Tensor* t = tensor_of(o);
  if (!t || t->numel() != numel || t->scalar_type() != dt || !t->is_contiguous() || t->get_device() != device)
    return false;
  *p = t->data_ptr();
  return true;
}

// what a call returns whose entry point returned status st (not IQ_OK)
PyObject* not_ok(const char* name, int st) {
  if (st != IQ_ERR_HIP) Py_RETURN_NONE;
  PyObject* m = PyImport_ImportModule("innerq_amd._lib");
  PyObject* e = m ? PyObject_CallMethod(m, "IQError", "si", name, st) : nullptr;
  if (e) PyErr_SetObject((PyObject*)Py_TYPE(e), e);
  Py_XDECREF(e);
  Py_XDECREF(m);
  return nullptr;
}

bool ints(PyObject* const* a, std::initializer_list<int> at, int64_t* v) {
  for (int i : at) {
    if (!PyLong_Check(a[i])) return false;
    *v = PyLong_AsLongLong(a[i]);
    if (*v == -1 && PyErr_Occurred()) { PyErr_Clear(); return false; }
    ++v;
  }
  return true;
}

// the token count T of a GEMV from t0 on (None: to the store's end); a negative one stays negative
bool tokens_of(PyObject* o, int64_t t0, const Store& s, int64_t* T) {
  if (o == Py_None) { *T = s.length - t0; return true; }
  return ints(&o, {0}, T);
}

// decode(q, k_sink, k_sink0, k_store, k_t0, k_len, k_recent, k_r0, k_rn, v_sink, v_sink0, v_store, v_t0, v_len,
//        v_recent, v_r0, v_rn, scale, norm, out, nd): q [B,Hq,D] (nd = 3) or [B,Hq,1,D] (nd = 4); the sinks' rows from
// *_sink0 on, the stores' tokens [t0, len) (len -1: all), the recents' rows [r0, r0 + rn) (rn -1: the rest).  Returns
// the output (of q's shape) or None.
PyObject* decode(PyObject*, PyObject* const* a, Py_ssize_t na) {
  if (na != 21) Py_RETURN_NONE;
  int64_t v[11];  // sink0, t0, len, r0, rn of K, then of V; nd
  if (!ints(a, {2, 4, 5, 7, 8, 10, 12, 13, 15, 16, 20}, v)) Py_RETURN_NONE;
  const at::Tensor* q = tensor_of(a[0]);
  if (!q || !act_dtype(q->scalar_type()) || (v[10] != 3 && v[10] != 4) || q->dim() != v[10] ||
      (q->dim() == 4 && q->size(2) != 1) || q->stride(q->dim() - 1) != 1)
    Py_RETURN_NONE;
  const int64_t B = q->size(0), Hq = q->size(1), D = q->size(q->dim() - 1);
  const at::ScalarType dt = q->scalar_type();
  const int dev = q->get_device();
  iq_segment ks[3] = {}, vs[3] = {};
  Store kst, vst;
  int64_t H = -1;
  if (!packed_segment(a[3], v[1], v[2], true, B, &H, D, dt, dev, kst, &ks[1]) ||
      !packed_segment(a[11], v[6], v[7], false, B, &H, D, dt, dev, vst, &vs[1]) || H <= 0 || Hq % H ||
      !dense_segment(a[1], v[0], a[1] == Py_None ? 0 : -1, B, H, D, dt, dev, &ks[0]) ||
      !dense_segment(a[6], v[3], a[6] == Py_None ? 0 : v[4], B, H, D, dt, dev, &ks[2]) ||
      !dense_segment(a[9], v[5], a[9] == Py_None ? 0 : -1, B, H, D, dt, dev, &vs[0]) ||
      !dense_segment(a[14], v[8], a[14] == Py_None ? 0 : v[9], B, H, D, dt, dev, &vs[2]))
    Py_RETURN_NONE;
  const int64_t T = int64_t(ks[0].n) + ks[1].n + ks[2].n;
  if (T != int64_t(vs[0].n) + vs[1].n + vs[2].n || T <= 0 || T > INT32_MAX || B <= 0) Py_RETURN_NONE;
  const void* norm;
  if (!norm_of(a[18], B * H * D, dt, dev, &norm)) Py_RETURN_NONE;
  const double scale = PyFloat_AsDouble(a[17]);
  if (scale == -1.0 && PyErr_Occurred()) { PyErr_Clear(); Py_RETURN_NONE; }
  const at::Tensor* given = nullptr;
  if (a[19] != Py_None) {
    given = tensor_of(a[19]);
    if (!given || given->sizes() != q->sizes() || given->scalar_type() != dt || given->get_device() != dev ||
        given->stride(given->dim() - 1) != 1)
      Py_RETURN_NONE;
  }
  void *stream, *ws;
  size_t wsb;
  at::Tensor hold;
  PyObject* key;
  if (!stream_of(dev, &stream, &key)) Py_RETURN_NONE;
  const bool have = workspace_of(key, fn.decode_ws(int(B), int(Hq), int(T), int(D)), &hold, &ws, &wsb);
  Py_DECREF(key);
  if (!have) Py_RETURN_NONE;
  at::Tensor out;
  try {
    out = given ? *given : at::empty(q->sizes(), q->options().requires_grad(false));
  } catch (...) {
    Py_RETURN_NONE;
  }
  int st;
  Py_BEGIN_ALLOW_THREADS
  st = fn.decode(q->data_ptr(), q->stride(0), q->stride(1), norm, ks, vs, int(B), int(Hq), int(H), int(T), int(D),
                 float(scale), out.data_ptr(), out.stride(0), out.stride(1), ws, wsb, stream);
  Py_END_ALLOW_THREADS
  if (st != IQ_OK) return not_ok("iq_decode_attention", st);
  if (given) { Py_INCREF(a[19]); return a[19]; }
  return THPVariable_Wrap(std::move(out));
}

// qk(q, store, scale, norm, t0, T, out): T None: to the store's end
PyObject* qk(PyObject*, PyObject* const* a, Py_ssize_t na) {
  if (na != 7) Py_RETURN_NONE;
  int64_t t0, T;
  const at::Tensor* q = tensor_of(a[0]);
  Store s;
  if (!ints(a, {4}, &t0) || !q || q->dim() != 3 || q->scalar_type() != at::kHalf || q->stride(2) != 1 ||
      !store_of(a[1], &s) || !tokens_of(a[5], t0, s, &T))
    Py_RETURN_NONE;
  const int64_t B = q->size(0), Hq = q->size(1), D = q->size(2);
  const int dev = q->get_device();
  const void* norm;
  if (!s.channel || s.dtype != at::kHalf || s.device != dev || s.B != B || s.D != D || s.H <= 0 || Hq % s.H || t0 < 0 ||
      T <= 0 || t0 > s.length || T > s.length - t0 || B <= 0 || !norm_of(a[3], B * s.H * D, at::kHalf, dev, &norm))
    Py_RETURN_NONE;
  const double scale = PyFloat_AsDouble(a[2]);
  if (scale == -1.0 && PyErr_Occurred()) { PyErr_Clear(); Py_RETURN_NONE; }
  const at::Tensor* given = nullptr;
  if (a[6] != Py_None) {
    given = tensor_of(a[6]);
    if (!given || given->dim() != 3 || given->size(0) != B || given->size(1) != Hq || given->size(2) != T ||
        given->scalar_type() != at::kFloat || given->get_device() != dev || given->stride(2) != 1)
      Py_RETURN_NONE;
  }
  void *stream, *ws;
  size_t wsb;
  at::Tensor hold;
  PyObject* key;
  if (!stream_of(dev, &stream, &key)) Py_RETURN_NONE;
  const bool have = workspace_of(key, fn.qk_ws(int(B), int(Hq), int(D)), &hold, &ws, &wsb);
  Py_DECREF(key);
  if (!have) Py_RETURN_NONE;
  at::Tensor out;
  try {
    out = given ? *given : at::empty({B, Hq, T}, q->options().dtype(at::kFloat).requires_grad(false));
  } catch (...) {
    Py_RETURN_NONE;
  }
  int st;
  Py_BEGIN_ALLOW_THREADS
  st = fn.qk(q->data_ptr(), q->stride(0), q->stride(1), norm, s.codes, s.meta, s.t_cap, int(B), int(Hq), int(s.H),
             int(t0), int(T), int(D), int(s.group), int(s.bits), int(s.mode), float(scale), (float*)out.data_ptr(),
             out.stride(0), out.stride(1), ws, wsb, stream);
  Py_END_ALLOW_THREADS
  if (st != IQ_OK) return not_ok("iq_qk_gemv", st);
  if (given) { Py_INCREF(a[6]); return a[6]; }
  return THPVariable_Wrap(std::move(out));
}

// av(p, store, t0, T, out): the fp16 output alone, written (not accumulated); T None: to the store's end
PyObject* av(PyObject*, PyObject* const* a, Py_ssize_t na) {
  if (na != 5) Py_RETURN_NONE;
  int64_t t0, T;
  const at::Tensor* p = tensor_of(a[0]);
  Store s;
  if (!ints(a, {2}, &t0) || !p || p->dim() != 3 || p->scalar_type() != at::kHalf || p->stride(2) != 1 ||
      !store_of(a[1], &s) || !tokens_of(a[3], t0, s, &T))
    Py_RETURN_NONE;
  const int64_t B = p->size(0), Hq = p->size(1);
  const int dev = p->get_device();
  if (s.channel || s.dtype != at::kHalf || s.device != dev || s.B != B || s.H <= 0 || Hq % s.H || t0 < 0 || T <= 0 ||
      t0 > s.length || T > s.length - t0 || p->size(2) < T || B <= 0)
    Py_RETURN_NONE;
  const at::Tensor* given = nullptr;
  if (a[4] != Py_None) {
    given = tensor_of(a[4]);
    if (!given || given->dim() != 3 || given->size(0) != B || given->size(1) != Hq || given->size(2) != s.D ||
        given->scalar_type() != at::kHalf || given->get_device() != dev || given->stride(2) != 1)
      Py_RETURN_NONE;
  }
  void *stream, *ws;
  size_t wsb;
  at::Tensor hold;
  PyObject* key;
  if (!stream_of(dev, &stream, &key)) Py_RETURN_NONE;
  const bool have = workspace_of(key, fn.av_ws(int(B), int(Hq), int(T), int(s.D), int(s.group)), &hold, &ws, &wsb);
  Py_DECREF(key);
  if (!have) Py_RETURN_NONE;
  at::Tensor out;
  try {
    out = given ? *given : at::empty({B, Hq, s.D}, p->options().requires_grad(false));
  } catch (...) {
    Py_RETURN_NONE;
  }
  int st;
  Py_BEGIN_ALLOW_THREADS
  st = fn.av(p->data_ptr(), p->stride(0), p->stride(1), s.codes, s.meta, s.t_cap, int(B), int(Hq), int(s.H), int(t0),
             int(T), int(s.D), int(s.group), int(s.bits), int(s.mode), nullptr, out.data_ptr(), out.stride(0),
             out.stride(1), 0, ws, wsb, stream);
  Py_END_ALLOW_THREADS
  if (st != IQ_OK) return not_ok("iq_av_gemv", st);
  if (given) { Py_INCREF(a[4]); return a[4]; }
  return THPVariable_Wrap(std::move(out));
}

// one role of a window append: its iq_window, and the state after it
struct Role {
  iq_window w{};
  at::Tensor buf;  // the window's and the store's tensors, held through the launch
  Store s;
  PyObject *win = nullptr, *store = nullptr;
  int64_t start, n, shadow, length, flush;
  bool deq;
};
bool set_int(PyObject* o, PyObject* name, int64_t v) {
  PyObject* x = PyLong_FromLongLong(v);
  const bool ok = x && PyObject_SetAttr(o, name, x) == 0;
  Py_XDECREF(x);
  return ok;
}
bool role_of(PyObject* win, PyObject* x, PyObject* flush, PyObject* store, PyObject* norm, Role* r, int64_t* B,
             int64_t* H, int64_t* D, int* dev) {
  if (!PyLong_Check(flush)) return false;
  r->win = win;
  r->flush = PyLong_AsLongLong(flush);
  PyObject* bo = PyObject_GetAttr(win, S_buf);
  PyObject* dq = PyObject_GetAttr(win, S_deq_rows);
  const at::Tensor* bt = bo ? tensor_of(bo) : nullptr;
  if (bt) r->buf = *bt;
  const at::Tensor* buf = bt ? &r->buf : nullptr;
  r->deq = dq == Py_True;
  Py_XDECREF(bo);
  Py_XDECREF(dq);
  const at::Tensor* t = tensor_of(x);
  if (PyErr_Occurred()) { PyErr_Clear(); return false; }
  if (!buf || !t || buf->dim() != 4 || t->dim() != 4 || t->scalar_type() != buf->scalar_type() ||
      !act_dtype(t->scalar_type()) || t->stride(3) != 1 || t->size(0) != buf->size(0) || t->size(1) != buf->size(1) ||
      t->size(3) != buf->size(3) || t->get_device() != buf->get_device() || !get_int(win, S_start, &r->start) ||
      !get_int(win, S_n, &r->n) || !get_int(win, S_shadow, &r->shadow))
    return false;
  if (*B < 0) { *B = t->size(0); *H = t->size(1); *D = t->size(3); *dev = t->get_device(); }
  else if (*B != t->size(0) || *H != t->size(1) || *D != t->size(3) || *dev != t->get_device()) return false;
  const int64_t m = t->size(2), cap = buf->size(2);
  if (r->start + r->n + m > cap || r->flush < 0 || r->flush > r->n + m) return false;  // the window has to move first
  iq_window& w = r->w;
  w.buf = buf->data_ptr();
  w.s_b = buf->stride(0); w.s_h = buf->stride(1); w.s_t = buf->stride(2);
  w.cap = int(cap); w.start = int(r->start); w.n = int(r->n);
  w.x = t->data_ptr();
  w.sx_b = t->stride(0); w.sx_h = t->stride(1); w.sx_t = t->stride(2);
  w.m = int(m); w.flush = int(r->flush);
  if (r->flush) {
    Store& s = r->s;
    if (store == Py_None || !store_of(store, &s) || s.dtype != t->scalar_type() || s.device != *dev || s.B != *B ||
        s.H != *H || s.D != *D || s.length + r->flush > s.t_cap || (!s.channel && r->flush % s.group))
      return false;
    r->store = store;
    r->length = s.length;
    w.codes = const_cast<uint32_t*>(s.codes); w.meta = s.meta;
    w.t_cap = s.t_cap; w.t_off = s.length;
    w.bits = int(s.bits); w.group = int(s.group); w.mode = int(s.mode) | act_flag(s.dtype);
    w.axis = s.channel ? 0 : 1;
    w.deq_rows = r->deq ? 1 : 0;
    const void* np;
    if (norm != Py_None && !s.channel) return false;
    if (!norm_of(norm, *B * *H * *D, t->scalar_type(), *dev, &np)) return false;
    w.norm = np;
  }
  return true;
}
// window_append(kwin, knew, kflush, kstore, knorm, vwin, vnew, vflush, vstore): True, or None
PyObject* window_append(PyObject*, PyObject* const* a, Py_ssize_t na) {
  if (na != 9 || a[0] == Py_None || a[5] == Py_None) Py_RETURN_NONE;
  Role r[2];
  int64_t B = -1, H = -1, D = -1;
  int dev = 0;
  if (!role_of(a[0], a[1], a[2], a[3], a[4], &r[0], &B, &H, &D, &dev) ||
      !role_of(a[5], a[6], a[7], a[8], Py_None, &r[1], &B, &H, &D, &dev))
    Py_RETURN_NONE;
  void* stream;
  PyObject* key;
  if (!stream_of(dev, &stream, &key)) Py_RETURN_NONE;
  Py_DECREF(key);
  int st;
  Py_BEGIN_ALLOW_THREADS
  st = fn.append(&r[0].w, &r[1].w, int(B), int(H), int(D), stream);
  Py_END_ALLOW_THREADS
  if (st != IQ_OK) return not_ok("iq_window_append", st);
  for (Role& x : r) {
    if (!set_int(x.win, S_start, x.start + x.flush) || !set_int(x.win, S_n, x.n + x.w.m - x.flush)) return nullptr;
    if (x.flush) {  // the flushed rows now hold their dequantized values (deq_rows)
      if (!set_int(x.win, S_shadow, x.deq ? x.shadow + x.flush : 0) || !set_int(x.store, S_length, x.length + x.flush))
        return nullptr;
    }
  }
  Py_RETURN_TRUE;
}

// bind(addresses, workspaces, raw_stream)
PyObject* bind(PyObject*, PyObject* const* a, Py_ssize_t na) {
  if (na != 3 || !PyTuple_Check(a[0]) || PyTuple_Size(a[0]) != 7 || !PyDict_Check(a[1]) || !PyCallable_Check(a[2])) {
    PyErr_SetString(PyExc_TypeError, "bind(seven addresses, workspaces, raw_stream)");
    return nullptr;
  }
  void* p[7];
  for (int i = 0; i < 7; ++i) p[i] = PyLong_AsVoidPtr(PyTuple_GetItem(a[0], i));
  if (PyErr_Occurred()) return nullptr;
  fn.decode_ws = (decode_ws_t)p[0]; fn.decode = (decode_t)p[1]; fn.qk_ws = (qk_ws_t)p[2]; fn.qk = (qk_t)p[3];
  fn.av_ws = (av_ws_t)p[4]; fn.av = (av_t)p[5]; fn.append = (append_t)p[6];
  Py_INCREF(a[1]); Py_INCREF(a[2]);
  fn.workspaces = a[1];
  fn.raw_stream = a[2];
  Py_RETURN_NONE;
}

#define FAST(name) {#name, (PyCFunction)(void (*)(void))name, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {FAST(bind), FAST(decode), FAST(qk), FAST(av), FAST(window_append), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_iqfast", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__iqfast() {
  struct { PyObject** s; const char* n; } names[] = {
      {&S_codes, "codes"}, {&S_meta, "meta"}, {&S_t_cap, "t_cap"}, {&S_length, "length"}, {&S_bits, "bits"},
      {&S_group, "group"}, {&S_mode, "mode"}, {&S_dtype, "dtype"}, {&S_axis, "axis"}, {&S_B, "B"}, {&S_H, "H"},
      {&S_D, "D"}, {&S_buf, "buf"}, {&S_start, "start"}, {&S_n, "n"}, {&S_deq_rows, "deq_rows"}, {&S_shadow, "shadow"}};
  for (auto& x : names)
    if (!(*x.s = PyUnicode_InternFromString(x.n))) return nullptr;
  return PyModule_Create(&module);
}
