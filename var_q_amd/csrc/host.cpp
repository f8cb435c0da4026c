// The host side of a call in native code: tensor checks, output and workspace allocation and the call
// of the C ABI, for the entry points of ops.py, pack_unpack.py, kv_cache.py and quant.py.
//
// A step of a few tokens is bound by its host work, not by its kernels: attributes of a dozen
// tensors, assertions, allocations and thirty ctypes conversions took 14-20 us per call from Python
// where the launch itself takes 3.  Functions take positional arguments only (METH_FASTCALL); the
// Python wrappers above them carry the names, the defaults and the documentation.
// Exceptions are those of the Python layer: AssertionError for arguments that do not fit together,
// VarqError for tensors off the GPU and for statuses of the library.
#include <Python.h>

#include <array>
#include <optional>

#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/varq.h"

namespace {

PyObject *g_varq_error = nullptr;

[[noreturn]] void raise(PyObject *type, const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  PyErr_FormatV(type, fmt, ap);
  va_end(ap);
  throw python_error();
}
#define ASSERT(cond, ...)                                  \
  do {                                                     \
    if (!(cond)) raise(PyExc_AssertionError, __VA_ARGS__); \
  } while (0)

void check(int rc, const char *what) {
  if (rc != VARQ_OK) raise(g_varq_error, "%s failed (status %d): %s", what, rc, varq_last_error());
}

// The interpreter's lock is given back while device memory is taken and launches are made: an allocation may wait
// for the device and a launch for room in a full queue, and neither is a reason for the program's other threads to wait.
// Once per call, around everything behind the reading of the arguments: inside, no Python object is touched and
// nothing is raised that is not a C++ exception.
struct NoGil {
  PyThreadState *const state = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(state); }
};
template <class F> int status_unlocked(F &&f) {
  const NoGil unlocked;
  return f();
}
template <class F> void unlocked(const char *what, F &&f) { check(status_unlocked(f), what); }

// ---- arguments ------------------------------------------------------------------------------
const at::Tensor &gpu(PyObject *o, const char *name) {
  if (!THPVariable_Check(o)) raise(g_varq_error, "%s must be a GPU tensor (got %s); the VAR-Q HIP path has no CPU fallback", name, Py_TYPE(o)->tp_name);
  const at::Tensor &t = THPVariable_Unpack(o);
  if (!t.is_cuda())
    raise(g_varq_error, "%s must be a GPU tensor (got %s); the VAR-Q HIP path has no CPU fallback", name, t.device().str().c_str());
  return t;
}
// None or a GPU tensor
const at::Tensor *maybe(PyObject *o, const char *name) { return o == Py_None ? nullptr : &gpu(o, name); }

int64_t integer(PyObject *o) {
  const long long v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) {
    // (numpy integers and the like)
    PyErr_Clear();
    PyObject *i = PyNumber_Index(o);
    if (!i) throw python_error();
    const long long w = PyLong_AsLongLong(i);
    Py_DECREF(i);
    if (w == -1 && PyErr_Occurred()) throw python_error();
    return w;
  }
  return v;
}
double real(PyObject *o) {
  const double v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) throw python_error();
  return v;
}
bool truth(PyObject *o) { return PyObject_IsTrue(o) == 1; }

int dtype_code(const at::Tensor &t) {
  switch (t.scalar_type()) {
    case at::kFloat: return VARQ_F32;
    case at::kBFloat16: return VARQ_BF16;
    case at::kHalf: return VARQ_F16;
    default: raise(g_varq_error, "unsupported dtype %s; expected float32, bfloat16 or float16", toString(t.scalar_type()));
  }
}
at::ScalarType dtype_of(int code) { return code == VARQ_F32 ? at::kFloat : code == VARQ_BF16 ? at::kBFloat16 : at::kHalf; }

template <typename T> T *ptr(const at::Tensor &t) { return reinterpret_cast<T *>(t.data_ptr()); }
template <typename T> T *ptr(const at::Tensor *t) { return t ? reinterpret_cast<T *>(t->data_ptr()) : nullptr; }

void *stream_of(const at::Tensor &t) { return (void *)c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

at::Tensor empty(at::IntArrayRef shape, at::ScalarType dt, const at::Tensor &like) { return at::empty(shape, like.options().dtype(dt)); }

PyObject *wrap(const at::Tensor &t) { return THPVariable_Wrap(t); }
PyObject *triple(const at::Tensor &a, const at::Tensor &b, const at::Tensor &c) {
  PyObject *t = PyTuple_New(3);
  PyTuple_SET_ITEM(t, 0, wrap(a));
  PyTuple_SET_ITEM(t, 1, wrap(b));
  if (c.defined()) PyTuple_SET_ITEM(t, 2, wrap(c));
  else { Py_INCREF(Py_None); PyTuple_SET_ITEM(t, 2, Py_None); }
  return t;
}

void need_args(Py_ssize_t n, Py_ssize_t want, const char *name) {
  if (n != want) raise(PyExc_TypeError, "%s takes %zd arguments (%zd given)", name, want, n);
}

// ---- quantize + pack --------------------------------------------------------------------------
// quant_rows(x, group, bits, asym, eps) -> (words, scale, zp | None)
PyObject *quant_rows(PyObject *const *a) {
  const at::Tensor &x0 = gpu(a[0], "x");
  const int64_t group = integer(a[1]), bits = integer(a[2]);
  const bool asym = truth(a[3]);
  const float eps = (float)real(a[4]);
  const int64_t c = x0.dim() ? x0.size(-1) : 0, rows = c ? x0.numel() / c : 0;
  ASSERT(x0.dim() >= 1 && group != 0, "quant_pack_rows: a tensor of rows and a group size are needed");
  const int dt = dtype_code(x0);
  const c10::DeviceGuard guard(x0.device());
  at::Tensor words, scale, zp;
  unlocked("varq_quant_pack_rows", [&] {
    const at::Tensor x = x0.contiguous();
    c10::DimVector shape(x.sizes().begin(), x.sizes().end());
    shape.back() = c * bits / 32;
    words = empty(shape, at::kInt, x);
    shape.back() = c / group;
    scale = empty(shape, at::kFloat, x);
    if (asym) zp = empty(shape, at::kFloat, x);
    return varq_quant_pack_rows(x.data_ptr(), dt, rows, (int)c, (int)group, (int)bits, asym, eps, nullptr, nullptr, ptr<int32_t>(words),
                                ptr<float>(scale), asym ? ptr<float>(zp) : nullptr, stream_of(x));
  });
  return triple(words, scale, zp);
}

struct Shared {   // shapes of a quantization with groups that span rows
  int64_t sh[4], sshape[4], last;
  Shared(const at::Tensor &x, int mask, int64_t bits, bool pack) {
    for (int d = 0; d < 4; ++d) {
      sh[d] = x.size(d);
      sshape[d] = mask >> d & 1 ? 1 : sh[d];
    }
    const int64_t vals = 32 / bits;
    last = pack ? (sh[3] + vals - 1) / vals : sh[3];
  }
};

// quant_shared(x, mask, bits, asym, eps, pack) -> (words | codes, scale, zp | None)
PyObject *quant_shared(PyObject *const *a) {
  const at::Tensor &x0 = gpu(a[0], "x");
  ASSERT(x0.dim() == 4, "expected a 4-D [B,L,H,c] / [B,H,L,c] tensor");
  const int mask = (int)integer(a[1]);
  const int64_t bits = integer(a[2]);
  const bool asym = truth(a[3]), pack = truth(a[5]);
  const float eps = (float)real(a[4]);
  ASSERT(bits > 0 && bits <= 32, "bits must be in 2..8");
  const Shared s(x0, mask, bits, pack);
  const int dt = dtype_code(x0);
  const c10::DeviceGuard guard(x0.device());
  at::Tensor q, scale, zp;
  unlocked("varq_quant_pack", [&] {
    const at::Tensor x = x0.contiguous();
    q = empty({s.sh[0], s.sh[1], s.sh[2], s.last}, pack ? at::kInt : at::kChar, x);
    scale = empty(at::IntArrayRef(s.sshape, 4), at::kFloat, x);
    if (asym) zp = empty(at::IntArrayRef(s.sshape, 4), at::kFloat, x);
    const size_t ws_bytes = std::max<size_t>(varq_quant_workspace_bytes(s.sh, mask), 8);
    const at::Tensor ws = empty({(int64_t)ws_bytes}, at::kByte, x);
    return varq_quant_pack(x.data_ptr(), dt, s.sh, mask, (int)bits, asym, eps, pack ? ptr<int32_t>(q) : nullptr, pack ? nullptr : ptr<int8_t>(q),
                           ptr<float>(scale), asym ? ptr<float>(zp) : nullptr, nullptr, ws.data_ptr(), ws_bytes, stream_of(x));
  });
  return triple(q, scale, zp);
}

// x and, in the same launches, x1 (or null), which is like it
int pack_rows(const at::Tensor &x, const void *x1, int dt, const int64_t *sh, int mask, int bits, bool asym, float eps, int32_t *w0, int32_t *w1,
              float *const *s, float *const *z, const int64_t *map) {
  const size_t one = std::max<size_t>(varq_quant_workspace_bytes(sh, mask), 8), ws_bytes = x1 ? 2 * one : one;
  const at::Tensor ws = empty({(int64_t)ws_bytes}, at::kByte, x);
  if (x1)
    return varq_quant_pack2(x.data_ptr(), x1, dt, sh, mask, bits, asym, eps, w0, nullptr, s[0], z[0], w1, nullptr, s[1], z[1], map, ws.data_ptr(), ws_bytes, stream_of(x));
  return varq_quant_pack(x.data_ptr(), dt, sh, mask, bits, asym, eps, w0, nullptr, s[0], z[0], map, ws.data_ptr(), ws_bytes, stream_of(x));
}

// ---- pack / unpack of int8 codes ----------------------------------------------------------------
int64_t codes_per_word(int64_t bits) {
  ASSERT(bits == 2 || bits == 4 || bits == 8, "bits must be 2, 4 or 8 (got %lld)", (long long)bits);
  return 32 / bits;
}
// pack(codes, bits) -> words
PyObject *pack(PyObject *const *a) {
  const at::Tensor &codes0 = gpu(a[0], "q_int8");
  const int64_t bits = integer(a[1]), c = codes0.size(-1), vals = codes_per_word(bits), rows = c ? codes0.numel() / c : 0;
  c10::DimVector shape(codes0.sizes().begin(), codes0.sizes().end());
  shape.back() = (c + vals - 1) / vals;
  const c10::DeviceGuard guard(codes0.device());
  at::Tensor words;
  unlocked("varq_pack", [&] {
    const at::Tensor codes = codes0.contiguous();
    words = empty(shape, at::kInt, codes);
    return varq_pack(ptr<int8_t>(codes), rows, (int)c, (int)bits, ptr<int32_t>(words), stream_of(codes));
  });
  return wrap(words);
}
// unpack(words, c, bits) -> codes
PyObject *unpack(PyObject *const *a) {
  const at::Tensor &words0 = gpu(a[0], "packed");
  const int64_t c = integer(a[1]), bits = integer(a[2]), w = words0.size(-1), rows = w ? words0.numel() / w : 0, vals = codes_per_word(bits);
  ASSERT(rows == 0 || w == (c + vals - 1) / vals, "unpack: rows of %lld words do not hold %lld codes of %lld bits", (long long)w, (long long)c, (long long)bits);
  c10::DimVector shape(words0.sizes().begin(), words0.sizes().end());
  shape.back() = c;
  const c10::DeviceGuard guard(words0.device());
  at::Tensor codes;
  unlocked("varq_unpack", [&] {
    const at::Tensor words = words0.contiguous();
    codes = empty(shape, at::kChar, words);
    return varq_unpack(ptr<int32_t>(words), rows, (int)c, (int)bits, ptr<int8_t>(codes), stream_of(words));
  });
  return wrap(codes);
}

// ---- dequantize ---------------------------------------------------------------------------------
// One scale per (i2, channel) whatever i0 and i1, the n2 rows of an (i0, i1) pair next to each other: the
// same bytes read as [1, n0, n1, n2 * c] (see ops._rows_as_channels, which states when and why).
void rows_as_channels(bool packed, int64_t (&sh)[4], int64_t (&ss)[4], int64_t group, int64_t bits, int64_t *map) {
  const int64_t n0 = sh[0], n1 = sh[1], n2 = sh[2], c = sh[3], c8 = n2 * c / 8;
  if (!packed || group != 1 || n2 <= 1 || c % 8 || c * bits % 32 || ss[0] || ss[1] || ss[2] != c || ss[3] != 1 || c8 > 256 || (c8 & (c8 - 1))) return;
  if (map) {
    if (map[5] != 1 || map[7] >= 0 || map[3] % n2 || map[4] % n2 || map[6] % n2) return;
    const int64_t m[8] = {1, n0, n1, 0, map[3] / n2, map[4] / n2, map[6] / n2, -1};
    std::copy(m, m + 8, map);
  }
  sh[0] = 1; sh[1] = n0; sh[2] = n1; sh[3] = n2 * c;
  ss[0] = ss[1] = ss[2] = 0;
}

// dequant(q, scale, zp | None, c, bits, out dtype code) -> [n0,n1,n2,c].  q: rows of words or codes, dense
// inside (a window of a cache buffer is read where it lies).
PyObject *dequant(PyObject *const *a) {
  at::Tensor q = gpu(a[0], "q"), scale = gpu(a[1], "scale"), zp;
  if (a[2] != Py_None) zp = gpu(a[2], "zp");
  const int64_t c = integer(a[3]), bits = integer(a[4]), code = integer(a[5]);
  ASSERT(q.dim() == 4 && scale.dim() == 4, "dequant: 4-D codes and scale");
  const bool packed = q.scalar_type() == at::kInt;
  ASSERT(packed || q.scalar_type() == at::kChar, "dequant: int32 words or int8 codes");
  const int64_t wq = q.size(3), s3 = scale.size(3);
  const int64_t vals = packed ? codes_per_word(bits) : 1;
  ASSERT(!q.numel() || wq == (c + vals - 1) / vals, "dequant: rows of %lld entries do not hold %lld channels", (long long)wq, (long long)c);
  ASSERT(s3 > 0 && c % s3 == 0, "scale last dim %lld does not divide c=%lld", (long long)s3, (long long)c);
  int64_t sh[4] = {q.size(0), q.size(1), q.size(2), c}, ss[4], map[8];
  for (int d = 0; d < 4; ++d)
    ASSERT(d == 3 || scale.size(d) == 1 || scale.size(d) == q.size(d), "scale dim %d = %lld vs %lld", d, (long long)scale.size(d), (long long)q.size(d));
  const c10::DeviceGuard guard(q.device());
  at::Tensor out;
  unlocked("varq_dequant", [&] {
    if (!q.is_contiguous() && (q.stride(3) != 1 || !wq || q.stride(0) % wq || q.stride(1) % wq || q.stride(2) % wq)) q = q.contiguous();
    if (zp.defined() && (zp.sizes() != scale.sizes() || zp.strides() != scale.strides())) {
      zp = zp.expand_as(scale).contiguous();
      scale = scale.contiguous();
    }
    for (int d = 0; d < 4; ++d) ss[d] = scale.size(d) == 1 ? 0 : scale.stride(d);
    out = empty(at::IntArrayRef(sh, 4), dtype_of((int)code), q);
    bool mapped = false;
    if (q.is_contiguous()) {
      // (leading dims that the scale does not depend on collapse: fuller blocks)
      if (!ss[0] && !ss[1] && !ss[2]) { sh[2] = sh[0] * sh[1] * sh[2]; sh[0] = sh[1] = 1; }
    } else {
      const int64_t m[8] = {sh[0], sh[1], sh[2], q.stride(0) / wq, q.stride(1) / wq, q.stride(2) / wq, 0, -1};
      std::copy(m, m + 8, map);
      mapped = true;
    }
    rows_as_channels(packed, sh, ss, c / s3, bits, mapped ? map : nullptr);
    return varq_dequant(packed ? ptr<int32_t>(q) : nullptr, packed ? nullptr : ptr<int8_t>(q), ptr<float>(scale), zp.defined() ? ptr<float>(zp) : nullptr,
                        sh, ss, (int)(c / s3), (int)bits, mapped ? map : nullptr, out.data_ptr(), (int)code, stream_of(q));
  });
  return wrap(out);
}

// dequant_steps(buf, seg_ends, tab, ztab | None, c, bits, out dtype code, token_dim) -> the tokens cached so far
PyObject *dequant_steps(PyObject *const *a) {
  const at::Tensor &buf = gpu(a[0], "buffer"), &tab = gpu(a[2], "scale table");
  const at::Tensor *ztab = maybe(a[3], "zero-point table");
  const int64_t c = integer(a[4]), bits = integer(a[5]), code = integer(a[6]), d = integer(a[7]);
  int32_t ends[16];
  ASSERT(PyList_Check(a[1]) && PyList_GET_SIZE(a[1]) >= 1 && PyList_GET_SIZE(a[1]) <= 16, "dequant_steps: 1..16 segments");
  const int nseg = (int)PyList_GET_SIZE(a[1]);
  for (int i = 0; i < nseg; ++i) ends[i] = (int32_t)integer(PyList_GET_ITEM(a[1], i));
  ASSERT(buf.dim() == 4 && buf.is_contiguous() && buf.scalar_type() == at::kInt && buf.size(3) * 32 == c * bits && (d == 1 || d == 2), "dequant_steps: buffer");
  const int64_t B = buf.size(0), H = buf.size(3 - d);
  ASSERT(tab.is_contiguous() && tab.scalar_type() == at::kFloat && tab.numel() >= nseg * H * c && (!ztab || ztab->sizes() == tab.sizes()), "dequant_steps: tables");
  const c10::DeviceGuard guard(buf.device());
  at::Tensor out;
  unlocked("varq_dequant_steps", [&] {
    out = d == 1 ? empty({B, ends[nseg - 1], H, c}, dtype_of((int)code), buf) : empty({B, H, ends[nseg - 1], c}, dtype_of((int)code), buf);
    return varq_dequant_steps(ptr<int32_t>(buf), ptr<float>(tab), ptr<float>(ztab), nseg, ends, (int)B, (int)H, buf.size(d), (int)c, (int)bits, d == 1,
                              out.data_ptr(), (int)code, stream_of(buf));
  });
  return wrap(out);
}

// ---- attention ----------------------------------------------------------------------------------
struct AttnShape {
  int64_t B, Hq, Lq, D, Hkv, Lstride;
  int layout;   // of the call, out included
  int64_t out_size[4];
  at::Tensor out;
  void new_out(const at::Tensor &q) {
    if (!out.defined()) out = empty(at::IntArrayRef(out_size, 4), q.scalar_type(), q);
  }
};

int layout_code(PyObject *o) {
  const char *s = PyUnicode_Check(o) ? PyUnicode_AsUTF8(o) : "";
  if (!strcmp(s, "BHLc")) return VARQ_LAYOUT_BHLC;
  ASSERT(!strcmp(s, "BLHc"), "layout must be one of ['BHLc', 'BLHc']");
  return VARQ_LAYOUT_BLHC;
}

// the layout of the call and its result tensor; s.out is not there yet (see new_out) unless the caller brought one
void make_out(AttnShape &s, const at::Tensor &q, PyObject *out, int lay, int olay) {
  s.layout = lay;
  if (olay != lay) {
    ASSERT(lay == VARQ_LAYOUT_BHLC, "out_layout: only tokens-first out of a heads-first call");
    s.layout = VARQ_LAYOUT_BHLC_OUT_BLHC;
  }
  const int64_t n[4] = {s.B, olay == VARQ_LAYOUT_BHLC ? s.Hq : s.Lq, olay == VARQ_LAYOUT_BHLC ? s.Lq : s.Hq, s.D};
  std::copy(n, n + 4, s.out_size);
  if (out != Py_None) {
    s.out = gpu(out, "out");
    ASSERT(s.out.scalar_type() == q.scalar_type() && s.out.sizes() == at::IntArrayRef(n, 4) && s.out.is_contiguous(),
           "out must be contiguous, of the dtype of q and of the shape its layout implies");
  }
}

// (the checks that both attention calls share; a: q, k_words, out, layout, out_layout)
AttnShape attn_shape(const at::Tensor &q, const at::Tensor &kw, PyObject *out, int lay, int out_lay) {
  AttnShape s;
  ASSERT((q.scalar_type() == at::kBFloat16 || q.scalar_type() == at::kHalf) && q.dim() == 4, "q must be bf16 or fp16");
  ASSERT(kw.dim() == 4, "k_words must be 4-D");
  const int h = lay == VARQ_LAYOUT_BHLC ? 1 : 2, t = 3 - h;
  s.B = q.size(0); s.Hq = q.size(h); s.Lq = q.size(t); s.D = q.size(3);
  s.Hkv = kw.size(h); s.Lstride = kw.size(t);
  ASSERT(kw.size(0) == s.B, "batch sizes of q and the cache differ");
  make_out(s, q, out, lay, out_lay);
  return s;
}
const at::Tensor &dense(PyObject *o, const char *name) {
  const at::Tensor &t = gpu(o, name);
  ASSERT(t.is_contiguous(), "%s must be contiguous", name);
  return t;
}
void check_limit_and_map(const at::Tensor *limit, const at::Tensor *map, const AttnShape &s) {
  if (limit) ASSERT(limit->scalar_type() == at::kInt && limit->numel() == s.Lq && limit->is_contiguous(), "kv_limit must be contiguous int32 [Lq]");
  if (map) ASSERT(map->scalar_type() == at::kInt && map->numel() == s.Hkv && map->is_contiguous(), "head_map must be int32 [Hkv]");
  else ASSERT(s.Hkv == s.Hq, "Hkv != Hq needs a head map");
}
int io_code(const at::Tensor &q) { return q.scalar_type() == at::kHalf ? VARQ_F16 : VARQ_BF16; }

// Device memory for a launch that shares keys out or expands them (undefined: neither).  Expanding takes more the longer the
// cache is; where the device has no room for it the call does without.  expands: the default operand form.
at::Tensor workspace(const AttnShape &s, const at::Tensor &q, int64_t Lk, int nseg, int64_t splits, bool limits, bool expands = true) {
  const size_t shared = expands ? varq_fused_attn_workspace_bytes_call((int)s.B, (int)s.Hkv, (int)s.Lq, (int)Lk, (int)s.D, nseg, (int)splits, limits)
                                : varq_fused_attn_workspace_bytes((int)s.B, (int)s.Hkv, (int)s.Lq, (int)Lk, (int)s.D, nseg, (int)splits);
  const auto bytes = limits ? varq_fused_attn_expand_bytes_limits : varq_fused_attn_expand_bytes;
  const size_t expanded = expands && splits <= 1 ? bytes((int)s.B, (int)s.Hkv, (int)s.Lq, (int)Lk, (int)s.D) : 0;
  if (expanded > shared) {
    try {
      return empty({(int64_t)expanded}, at::kByte, q);
    } catch (const c10::OutOfMemoryError &) {
    }
  }
  return shared ? empty({(int64_t)shared}, at::kByte, q) : at::Tensor();
}
void *bytes_of(const at::Tensor &ws) { return ws.defined() ? ws.data_ptr() : nullptr; }
size_t size_of(const at::Tensor &ws) { return ws.defined() ? (size_t)ws.numel() : 0; }

// Attention over the packed rows of one bit-width with scales per key.
struct KeyScales {
  const at::Tensor &kw, &ks, &vw, &vs;
  const at::Tensor *kz, *vz;
  int64_t k_bits, v_bits;
};
PyObject *attend_rows(const at::Tensor &q, const KeyScales &r, int64_t Lk, float softmax_scale, const at::Tensor *limit, const at::Tensor *map, PyObject *out,
                      int64_t splits, int lay, int out_lay, bool exact) {
  const at::Tensor &kw = r.kw, &ks = r.ks, &vw = r.vw, &vs = r.vs;
  const c10::DeviceGuard guard(q.device());
  AttnShape s = attn_shape(q, kw, out, lay, out_lay);
  ASSERT(vw.dim() == 4 && ks.dim() == 4 && vs.dim() == 4, "4-D cache tensors");
  for (int d = 0; d < 3; ++d)
    ASSERT(vw.size(d) == kw.size(d) && ks.size(d) == kw.size(d) && vs.size(d) == kw.size(d), "words and scales must agree in batch, heads and tokens");
  ASSERT(kw.size(3) * 32 == s.D * r.k_bits && vw.size(3) * 32 == s.D * r.v_bits, "words per row do not match the head dim and the bit-width");
  ASSERT(ks.size(3) > 0 && vs.size(3) > 0, "empty scales");
  for (const auto &[z, sc, n] : {std::tuple(r.kz, &ks, "k_zp"), std::tuple(r.vz, &vs, "v_zp")})
    ASSERT(!z || (z->sizes() == sc->sizes() && z->scalar_type() == at::kFloat && z->is_contiguous()), "%s must look like its scale", n);
  ASSERT(ks.scalar_type() == at::kFloat && vs.scalar_type() == at::kFloat && kw.scalar_type() == at::kInt && vw.scalar_type() == at::kInt,
         "scales must be fp32 and words int32");
  ASSERT(0 <= Lk && Lk <= s.Lstride, "Lk=%lld outside the cache of %lld tokens", (long long)Lk, (long long)s.Lstride);
  check_limit_and_map(limit, map, s);
  unlocked("varq_fused_attn", [&] {
    s.new_out(q);
    const at::Tensor ws = workspace(s, q, Lk, 1, splits, limit != nullptr, !exact || io_code(q) == VARQ_F16);
    return varq_fused_attn(q.data_ptr(), s.out.data_ptr(), ptr<int32_t>(kw), ptr<float>(ks), ptr<float>(r.kz), (int)r.k_bits, (int)(s.D / ks.size(3)),
                           ptr<int32_t>(vw), ptr<float>(vs), ptr<float>(r.vz), (int)r.v_bits, (int)(s.D / vs.size(3)), (int)s.B, (int)s.Hq, (int)s.Hkv,
                           ptr<int32_t>(map), (int)s.Lq, (int)Lk, (int)s.Lstride, (int)s.D, ptr<int32_t>(limit), softmax_scale, s.layout, io_code(q),
                           exact, bytes_of(ws), size_of(ws), (int)splits, stream_of(q));
  });
  return wrap(s.out);
}

// attn(q, k_words, k_scale, k_zp, v_words, v_scale, v_zp, k_bits, v_bits, Lk, softmax_scale, kv_limit, head_map, out, splits,
//      layout, exact_codes, out_layout) -> out
PyObject *attn(PyObject *const *a) {
  const at::Tensor &q = dense(a[0], "q");
  const KeyScales r = {dense(a[1], "k_words"), dense(a[2], "k_scale"), dense(a[4], "v_words"), dense(a[5], "v_scale"), maybe(a[3], "k_zp"), maybe(a[6], "v_zp"),
                       integer(a[7]), integer(a[8])};
  const at::Tensor *limit = maybe(a[11], "kv_limit"), *map = maybe(a[12], "head_map");
  const int lay = layout_code(a[15]);
  return attend_rows(q, r, integer(a[9]), (float)real(a[10]), limit, map, a[13], integer(a[14]), lay, a[17] == Py_None ? lay : layout_code(a[17]), truth(a[16]));
}

// attn_channel(q, k_words, k_scale, k_zp, v_words, v_scale, v_zp, bits, Lk, softmax_scale, kv_limit, head_map, out, seg_ends, splits,
//              layout, out_layout) -> out
PyObject *attn_channel(PyObject *const *a) {
  const at::Tensor &q = dense(a[0], "q"), &kw = dense(a[1], "k_words"), &ks = dense(a[2], "k_chan_scale"), &vw = dense(a[4], "v_words"), &vs = dense(a[5], "v_chan_scale");
  const at::Tensor *kz = maybe(a[3], "k_chan_zp"), *vz = maybe(a[6], "v_chan_zp"), *limit = maybe(a[10], "kv_limit"), *map = maybe(a[11], "head_map");
  const int64_t bits = integer(a[7]), Lk = integer(a[8]), splits = integer(a[14]);
  const c10::DeviceGuard guard(q.device());
  const int lay = layout_code(a[15]);
  AttnShape s = attn_shape(q, kw, a[12], lay, a[16] == Py_None ? lay : layout_code(a[16]));
  ASSERT(vw.sizes() == kw.sizes() && kw.size(3) * 32 == s.D * bits, "K and V words must agree and match the head dim and the bit-width");
  int32_t ends[16];
  int nseg = 1;
  const bool seg = a[13] != Py_None;
  if (seg) {
    PyObject *f = PySequence_Fast(a[13], "seg_ends must be a sequence");
    if (!f) throw python_error();
    const Py_ssize_t n = PySequence_Fast_GET_SIZE(f);
    bool fine = n >= 1 && n <= 16;
    if (fine) {
      nseg = (int)n;
      for (int i = 0; i < nseg; ++i) ends[i] = (int32_t)integer(PySequence_Fast_GET_ITEM(f, i));
      fine = ends[nseg - 1] == Lk;
    }
    Py_DECREF(f);
    ASSERT(fine, "seg_ends: 1..16 entries, the last one equal to Lk");
  }
  for (const auto &[t, n] : {std::pair(&ks, "k_chan_scale"), std::pair(kz, "k_chan_zp"), std::pair(&vs, "v_chan_scale"), std::pair(vz, "v_chan_zp")})
    ASSERT(!t || (t->scalar_type() == at::kFloat && t->numel() >= nseg * s.Hkv * s.D && t->is_contiguous()),
           "%s must be fp32 [nseg, Hkv, D] (more tables than segments are allowed)", n);
  ASSERT(kw.scalar_type() == at::kInt && vw.scalar_type() == at::kInt, "words must be int32");
  ASSERT(0 <= Lk && Lk <= s.Lstride, "Lk=%lld outside the cache of %lld tokens", (long long)Lk, (long long)s.Lstride);
  check_limit_and_map(limit, map, s);
  const float softmax_scale = (float)real(a[9]);
  unlocked("varq_fused_attn_channel", [&] {
    s.new_out(q);
    const at::Tensor ws = workspace(s, q, Lk, nseg, splits, limit != nullptr);
    return varq_fused_attn_channel(q.data_ptr(), s.out.data_ptr(), ptr<int32_t>(kw), ptr<float>(ks), ptr<float>(kz), ptr<int32_t>(vw), ptr<float>(vs),
                                   ptr<float>(vz), nseg, seg ? ends : nullptr, (int)bits, (int)s.B, (int)s.Hq, (int)s.Hkv, ptr<int32_t>(map), (int)s.Lq,
                                   (int)Lk, (int)s.Lstride, (int)s.D, ptr<int32_t>(limit), softmax_scale, s.layout, io_code(q),
                                   bytes_of(ws), size_of(ws), (int)splits, stream_of(q));
  });
  return wrap(s.out);
}

// ---- packed cache -------------------------------------------------------------------------------
// A PackedKVCache as its attributes say at the time of the call: a caller may have replaced buffers, or set others of them.
// attribute `name` (an interned string) of o: out of the instance's own dictionary where it has one and the name is there, which
// takes a third of the general way's time
PyObject *attribute(PyObject *o, PyObject *name) {   // (a new reference)
  PyObject **const d = _PyObject_GetDictPtr(o);
  PyObject *v = d && *d ? PyDict_GetItemWithError(*d, name) : nullptr;
  if (v) {
    Py_INCREF(v);
    return v;
  }
  if (PyErr_Occurred() || !(v = PyObject_GetAttr(o, name))) throw python_error();
  return v;
}
struct Ref {   // owns the reference it is given
  PyObject *const o;
  explicit Ref(PyObject *owned) : o(owned) { if (!o) throw python_error(); }
  Ref(const Ref &) = delete;
  ~Ref() { Py_DECREF(o); }
};
#define NAME(id) ([]() { static PyObject *const name = PyUnicode_InternFromString(#id); return name; }())

// A tensor of a cache: held through its Python object, which is free under the interpreter's lock, as every place of use is
// made and dropped.
struct Held {
  PyObject *o = nullptr;
  const at::Tensor *t = nullptr;
  Held() = default;
  Held(const Held &) = delete;
  ~Held() { Py_XDECREF(o); }
  const at::Tensor *operator->() const { return t; }
};
template <typename T> T *ptr(const Held &h) { return h.t ? reinterpret_cast<T *>(h.t->data_ptr()) : nullptr; }

struct CacheClass {
  int64_t bits, heads;
  Held k_words, k_scale, k_zp, v_words, v_scale, v_zp, slot, head_map;

  // field i of a class, whose Python object is a list of its fields (another object: by name)
  static PyObject *field(PyObject *of, int i, PyObject *name) {
    if (!PyList_Check(of) || PyList_GET_SIZE(of) != 10) return attribute(of, name);
    PyObject *const v = PyList_GET_ITEM(of, i);
    Py_INCREF(v);
    return v;
  }
  static void dense(Held &h, PyObject *of, int i, PyObject *name, at::ScalarType dt) {
    h.o = field(of, i, name);
    h.t = &gpu(h.o, "cache buffer");
    ASSERT(h.t->scalar_type() == dt && h.t->is_contiguous(), "cache buffer %U must be contiguous and of type %s", name, toString(dt));
  }
  void read(PyObject *o, int64_t H, bool asym) {
    bits = integer(Ref(field(o, 0, NAME(bits))).o);
    const Py_ssize_t n = PyObject_Size(Ref(field(o, 1, NAME(heads))).o);
    if (n < 0) throw python_error();
    heads = n;
    dense(k_words, o, 2, NAME(k_words), at::kInt);
    dense(k_scale, o, 3, NAME(k_scale), at::kFloat);
    if (asym) dense(k_zp, o, 4, NAME(k_zp), at::kFloat);
    dense(v_words, o, 5, NAME(v_words), at::kInt);
    dense(v_scale, o, 6, NAME(v_scale), at::kFloat);
    if (asym) dense(v_zp, o, 7, NAME(v_zp), at::kFloat);
    dense(slot, o, 8, NAME(slot), at::kInt);
    dense(head_map, o, 9, NAME(head_map), at::kInt);
    ASSERT(heads > 0 && slot->numel() == H && head_map->numel() == heads, "cache class of %lld bits: slot and head_map do not fit its heads", (long long)bits);
  }
  // the kernels trust the sizes: rows as long as the call implies, and the last one it reaches inside
  void check(int64_t D, int64_t group, int64_t last) const {
    const int64_t W = D * bits / 32, ng = D / group;
    for (const auto &[w, sc, z] : {std::tuple(&k_words, &k_scale, &k_zp), std::tuple(&v_words, &v_scale, &v_zp)}) {
      const auto &ws = (*w)->sizes(), &ss = (*sc)->sizes();
      if (ws.empty() || ss.empty() || ws.back() != W || ss.back() != ng || (z->t && (*z)->sizes() != ss))
        raise(g_varq_error, "cache class of %lld bits: rows of words, scales and zero-points must have %lld, %lld and %lld entries", (long long)bits, (long long)W, (long long)ng, (long long)ng);
      const int64_t rows = std::min((*w)->numel() / W, (*sc)->numel() / ng);
      if (last >= rows)
        raise(g_varq_error, "cache class of %lld bits: the call reaches row %lld of buffers that hold %lld rows", (long long)bits, (long long)last, (long long)rows);
    }
  }
};
struct Cache {
  int64_t B, H, Lmax, D, group;
  bool asym;
  float eps;
  int n = 0;
  CacheClass classes[3];
  explicit Cache(PyObject *o) {
    auto number = [&](PyObject *name) { return integer(Ref(attribute(o, name)).o); };
    B = number(NAME(B)); H = number(NAME(H)); Lmax = number(NAME(Lmax)); D = number(NAME(D)); group = number(NAME(group));
    asym = !truth(Ref(attribute(o, NAME(symmetric))).o);
    eps = (float)real(Ref(attribute(o, NAME(eps))).o);
    ASSERT(B > 0 && H > 0 && D >= 16 && group > 0 && D % group == 0, "cache sizes");
    const Ref list(attribute(o, NAME(classes))), seq(PySequence_Fast(list.o, "classes must be a sequence"));
    const Py_ssize_t count = PySequence_Fast_GET_SIZE(seq.o);
    ASSERT(count >= 1 && count <= 3, "a cache has 1..3 bit-width classes");
    for (; n < count; ++n) {
      classes[n].read(PySequence_Fast_GET_ITEM(seq.o, n), H, asym);
      ASSERT(classes[n].bits == 2 || classes[n].bits == 4 || classes[n].bits == 8, "a class has 2, 4 or 8 bits");
    }
  }
  // every class holds tokens 0..len-1 (token j of a head lies Lmax rows from that of the next)
  void check(int64_t len) const {
    for (int i = 0; i < n; ++i) classes[i].check(D, group, (B * classes[i].heads - 1) * Lmax + len - 1);
  }
};

// the classes of a cache as the C ABI takes them
int class_table(const Cache &c, varq_kv_class (&t)[3]) {
  for (int i = 0; i < c.n; ++i) {
    const CacheClass &k = c.classes[i];
    t[i] = {(int)k.bits, (int)k.heads, ptr<int32_t>(k.head_map), ptr<int32_t>(k.slot), ptr<int32_t>(k.k_words), ptr<int32_t>(k.v_words),
            ptr<float>(k.k_scale), c.asym ? ptr<float>(k.k_zp) : nullptr, ptr<float>(k.v_scale), c.asym ? ptr<float>(k.v_zp) : nullptr};
  }
  return c.n;
}

// cache_attend(cache, len, q, softmax_scale, kv_limit, out, splits, out_layout, exact_codes) -> out: all classes in one call
// (exact codes: of a cache of one class only)
PyObject *cache_attend(PyObject *const *a) {
  const Cache c(a[0]);
  const int64_t len = integer(a[1]), splits = integer(a[6]);
  const at::Tensor &q = dense(a[2], "q");
  const at::Tensor *limit = maybe(a[4], "kv_limit");
  const bool exact = truth(a[8]);
  if (c.n == 1) {
    const CacheClass &k = c.classes[0];
    const KeyScales r = {*k.k_words.t, *k.k_scale.t, *k.v_words.t, *k.v_scale.t, k.k_zp.t, k.v_zp.t, k.bits, k.bits};
    return attend_rows(q, r, len, (float)real(a[3]), limit, nullptr, a[5], splits, VARQ_LAYOUT_BHLC, layout_code(a[7]), exact);
  }
  ASSERT(!exact, "exact codes: one class at a time");
  ASSERT((q.scalar_type() == at::kBFloat16 || q.scalar_type() == at::kHalf) && q.dim() == 4, "q must be bf16 or fp16");
  ASSERT(q.size(0) == c.B && q.size(1) == c.H && q.size(3) == c.D, "attend: q does not fit the cache");
  ASSERT(0 < len && len <= c.Lmax, "attend: the cache holds no such token");
  c.check(len);
  const c10::DeviceGuard guard(q.device());
  AttnShape s;
  s.B = c.B; s.Hq = s.Hkv = c.H; s.Lq = q.size(2); s.D = c.D; s.Lstride = c.Lmax;
  make_out(s, q, a[5], VARQ_LAYOUT_BHLC, layout_code(a[7]));
  check_limit_and_map(limit, nullptr, s);
  varq_kv_class t[3];
  const int n = class_table(c, t);
  const float softmax_scale = (float)real(a[3]);
  unlocked("varq_fused_attn_classes", [&] {
    s.new_out(q);
    const at::Tensor ws = workspace(s, q, len, 1, splits, limit != nullptr);
    return varq_fused_attn_classes(q.data_ptr(), s.out.data_ptr(), t, n, (int)c.group, (int)c.B, (int)c.H, (int)s.Lq, (int)len, (int)c.Lmax, (int)c.D,
                                   ptr<int32_t>(limit), softmax_scale, s.layout, io_code(q), bytes_of(ws), size_of(ws), (int)splits,
                                   stream_of(q));
  });
  return wrap(s.out);
}

// cache_append(cache, len, k, v, layout) -> tokens appended
PyObject *cache_append(PyObject *const *a) {
  const Cache c(a[0]);
  const int64_t len = integer(a[1]);
  ASSERT(THPVariable_Check(a[2]) && THPVariable_Check(a[3]), "append: tensors");
  at::Tensor k = THPVariable_Unpack(a[2]), v = THPVariable_Unpack(a[3]);
  const int lay = layout_code(a[4]), h = lay == VARQ_LAYOUT_BHLC ? 1 : 2;
  ASSERT(k.dim() == 4 && k.size(0) == c.B && k.size(h) == c.H && k.size(3) == c.D && v.sizes() == k.sizes(), "append: the step does not fit the cache");
  const int64_t n = k.size(3 - h);
  ASSERT(len >= 0 && len + n <= c.Lmax, "cache overflow");
  c.check(len + n);
  gpu(a[2], "k"); gpu(a[3], "v");
  const c10::DeviceGuard guard(k.device());
  const int kd = dtype_code(k), vd = dtype_code(v);
  const char *what = "varq_quant_pack_classes";
  const int rc = status_unlocked([&] {
    k = k.contiguous(); v = v.contiguous();
    void *const st = stream_of(k);
    const int64_t rows = c.B * c.H * n;
    if (c.n > 1) {   // (one launch for all classes, where the sizes allow it)
      varq_kv_class t[3];
      const int nc = class_table(c, t);
      auto classes = [&](const void *kp, const void *vp, int dt) {
        return varq_quant_pack_classes(kp, vp, dt, lay, (int)c.B, (int)c.H, n, (int)c.D, (int)c.group, c.asym, c.eps, t, nc, c.Lmax, len, st);
      };
      int rc = kd == vd ? classes(k.data_ptr(), v.data_ptr(), kd) : classes(k.data_ptr(), nullptr, kd);
      if (kd != vd && rc == VARQ_OK) rc = classes(nullptr, v.data_ptr(), vd);
      if (rc != VARQ_ERR_UNSUPPORTED) return rc;
    }
    for (int i = 0; i < c.n; ++i) {
      const CacheClass &cl = c.classes[i];
      // input rows in memory order -> output row b*hc*Lmax + slot(h)*Lmax + len + l
      const int64_t bs = cl.heads * c.Lmax;
      const int64_t bhlc[8] = {c.B, c.H, n, bs, c.Lmax, 1, len, 1}, blhc[8] = {c.B, n, c.H, bs, 1, c.Lmax, len, 2};
      const int64_t *map = lay == VARQ_LAYOUT_BHLC ? bhlc : blhc;
      float *kz = c.asym ? ptr<float>(cl.k_zp) : nullptr, *vz = c.asym ? ptr<float>(cl.v_zp) : nullptr;
      int rc;
      if (kd == vd && 2 * c.B <= 65535) {
        what = "varq_quant_pack_rows2";
        rc = varq_quant_pack_rows2(k.data_ptr(), v.data_ptr(), kd, rows, (int)c.D, (int)c.group, (int)cl.bits, c.asym, c.eps, map, ptr<int32_t>(cl.slot),
                                   ptr<int32_t>(cl.k_words), ptr<float>(cl.k_scale), kz, ptr<int32_t>(cl.v_words), ptr<float>(cl.v_scale), vz, st);
      } else {   // K and V of different dtypes (Infinity: fp32 K after cos-norm, bf16 V)
        what = "varq_quant_pack_rows";
        rc = varq_quant_pack_rows(k.data_ptr(), kd, rows, (int)c.D, (int)c.group, (int)cl.bits, c.asym, c.eps, map, ptr<int32_t>(cl.slot),
                                  ptr<int32_t>(cl.k_words), ptr<float>(cl.k_scale), kz, st);
        if (rc == VARQ_OK)
          rc = varq_quant_pack_rows(v.data_ptr(), vd, rows, (int)c.D, (int)c.group, (int)cl.bits, c.asym, c.eps, map, ptr<int32_t>(cl.slot),
                                    ptr<int32_t>(cl.v_words), ptr<float>(cl.v_scale), vz, st);
      }
      if (rc != VARQ_OK) return rc;
    }
    return (int)VARQ_OK;
  });
  check(rc, what);
  return PyLong_FromLongLong(n);
}

// cache_prepare(cache, len, qkv, q_scale_mul | None, l2norm, norm_eps, cos | None, sin | None, token_start) -> q
PyObject *cache_prepare(PyObject *const *a) {
  const Cache c(a[0]);
  const int64_t len = integer(a[1]), start = integer(a[8]);
  at::Tensor qkv = gpu(a[2], "qkv");
  ASSERT(qkv.dim() == 5 && qkv.size(2) == 3 && qkv.size(0) == c.B && qkv.size(3) == c.H && qkv.size(4) == c.D, "append_from_qkv: qkv [B,n,3,H,D] of the cache's sizes");
  const int64_t n = qkv.size(1);
  ASSERT(len >= 0 && len + n <= c.Lmax, "cache overflow");
  c.check(len + n);
  const at::Tensor *mul = maybe(a[3], "q_scale_mul"), *cs = maybe(a[6], "rope cos"), *sn = maybe(a[7], "rope sin");
  if (cs || sn) {
    ASSERT(cs && sn && cs->dim() == 2 && cs->scalar_type() == at::kFloat && sn->scalar_type() == at::kFloat && cs->is_contiguous() && sn->is_contiguous(), "rope tables must be contiguous fp32");
    ASSERT(cs->sizes() == sn->sizes() && cs->size(1) == c.D / 2 && cs->size(0) >= start + n, "rope tables are too small");
  }
  if (mul) ASSERT(mul->scalar_type() == at::kFloat && mul->numel() == c.H && mul->is_contiguous(), "q_scale_mul must be contiguous fp32 [H]");
  const c10::DeviceGuard guard(qkv.device());
  const int dt = dtype_code(qkv);
  const bool l2norm = truth(a[4]);
  const float norm_eps = (float)real(a[5]);
  at::Tensor q;
  const char *what = "varq_qkv_prepare_classes";
  const int rc = status_unlocked([&] {
    qkv = qkv.contiguous();
    q = empty({c.B, c.H, n, c.D}, at::kBFloat16, qkv);
    if (c.n > 1) {
      varq_kv_class t[3];
      const int nc = class_table(c, t);
      const int rc = varq_qkv_prepare_classes(qkv.data_ptr(), dt, (int)c.B, (int)n, (int)c.H, (int)c.D, ptr<float>(mul), l2norm, norm_eps, ptr<float>(cs),
                                              ptr<float>(sn), (int)start, q.data_ptr(), (int)c.group, c.asym, c.eps, t, nc, c.Lmax, len, stream_of(qkv));
      if (rc != VARQ_ERR_UNSUPPORTED) return rc;
    }
    what = "varq_qkv_prepare_append";
    for (int i = 0; i < c.n; ++i) {
      const CacheClass &cl = c.classes[i];
      const int64_t map[8] = {c.B, n, c.H, cl.heads * c.Lmax, 1, c.Lmax, len, 2};
      const int rc = varq_qkv_prepare_append(qkv.data_ptr(), dt, (int)c.B, (int)n, (int)c.H, (int)c.D, ptr<float>(mul), l2norm, norm_eps, ptr<float>(cs),
                                             ptr<float>(sn), (int)start, q.data_ptr(), (int)c.group, (int)cl.bits, c.asym, c.eps, map, ptr<int32_t>(cl.slot),
                                             ptr<int32_t>(cl.k_words), ptr<float>(cl.k_scale), c.asym ? ptr<float>(cl.k_zp) : nullptr,
                                             ptr<int32_t>(cl.v_words), ptr<float>(cl.v_scale), c.asym ? ptr<float>(cl.v_zp) : nullptr, stream_of(qkv));
      if (rc != VARQ_OK) return rc;
    }
    return (int)VARQ_OK;
  });
  check(rc, what);
  return wrap(q);
}

// ---- drop-in quantizers -------------------------------------------------------------------------
// A step of VAR_Q (quant.py) and the attention over two of them, with their state read from and left in the Python objects'
// attributes: what quant() followed by cache() leaves.  Anything out of the ordinary -- other rules, no room yet, a tensor of
// another kind -- is refused with nothing done, and the Python methods take the call.
enum class Rule { kHeadDim, kScale, kHead, kToken, kTokenHead, kOtherTable, kOtherToken, kNone };
Rule rule_of(PyObject *m) {
  const std::pair<PyObject *, Rule> rules[] = {{NAME(G_SCALE_HEAD_DIM), Rule::kHeadDim}, {NAME(G_SCALE), Rule::kScale}, {NAME(G_HEAD), Rule::kHead},
                                               {NAME(G_TOKEN), Rule::kToken}, {NAME(G_TOKEN_HEAD), Rule::kTokenHead}, {NAME(G_HEAD_DIM), Rule::kOtherTable},
                                               {NAME(G_TENSOR), Rule::kOtherTable}, {NAME(G_GROUP), Rule::kOtherToken}};
  for (const auto &[name, rule] : rules)
    if (m == name) return rule;
  for (const auto &[name, rule] : rules)
    if (PyUnicode_Check(m) && PyUnicode_Compare(m, name) == 0) return rule;
  return Rule::kNone;
}
bool per_token(Rule r) { return r == Rule::kToken || r == Rule::kTokenHead || r == Rule::kOtherToken; }
void set_attribute(PyObject *o, PyObject *name, PyObject *v) {   // (takes the reference)
  const Ref value(v);
  if (PyObject_SetAttr(o, name, v)) throw python_error();
}
int64_t number_of(PyObject *o, PyObject *name) { return integer(Ref(attribute(o, name)).o); }

// a dense GPU tensor of that type in attribute `name`, or an empty place
bool tensor_of(Held &h, PyObject *o, PyObject *name, at::ScalarType dt) {
  PyObject *const v = attribute(o, name);
  if (THPVariable_Check(v)) {
    const at::Tensor &t = THPVariable_Unpack(v);
    if (t.is_cuda() && t.scalar_type() == dt && t.is_contiguous()) {
      h.o = v;
      h.t = &t;
      return true;
    }
  }
  Py_DECREF(v);
  return false;
}

struct Quantizer {
  PyObject *const o;
  Rule rule;
  int64_t bits, d, k = 0, len, c;      // token dim, cached steps, cached tokens, channels
  bool asym, packed;
  Held buf, scale, zp;                 // codes; the step tables or the scales per token
  Ref item, ends;
  Held tok, tokz;                      // (the growable buffers of the scales per token, as objects)
  bool ready = false;                  // everything above is there, and of the kinds that the kernels read

  explicit Quantizer(PyObject *obj)
      : o(obj), rule(rule_of(Ref(attribute(obj, NAME(quant_method))).o)), bits(number_of(obj, NAME(quant_bits))), d(number_of(obj, NAME(dim_cat))),
        asym(!truth(Ref(attribute(obj, NAME(symmetric))).o)), packed(truth(Ref(attribute(obj, NAME(pack_to_int32))).o)),
        item(attribute(obj, NAME(_c_item))), ends(attribute(obj, NAME(_seg_ends))) {
    if (rule == Rule::kNone || !packed || (bits != 2 && bits != 4 && bits != 8) || (d != 1 && d != 2) || !PyList_Check(ends.o)) return;
    len = number_of(item.o, NAME(len));
    if (number_of(item.o, NAME(dim)) != d || !tensor_of(buf, item.o, NAME(buf), at::kInt) || buf->dim() != 4) return;
    const Ref meta(attribute(o, NAME(_pack_meta)));
    if (!PyDict_Check(meta.o)) return;
    PyObject *const oc = PyDict_GetItem(meta.o, NAME(orig_c)), *const ob = PyDict_GetItem(meta.o, NAME(bits));
    if (!oc || !ob || integer(ob) != bits) return;
    c = integer(oc);
    if (buf->size(3) * 32 != c * bits) return;
    k = PyList_GET_SIZE(ends.o);
    if (per_token(rule)) {
      tok.o = attribute(o, NAME(_tok_scale));
      tokz.o = attribute(o, NAME(_tok_zp));
      if (number_of(tok.o, NAME(dim)) != d || number_of(tok.o, NAME(len)) != len || !tensor_of(scale, tok.o, NAME(buf), at::kFloat) || scale->dim() != 4) return;
      if (asym ? number_of(tokz.o, NAME(len)) != len || !tensor_of(zp, tokz.o, NAME(buf), at::kFloat) || zp->sizes() != scale->sizes()
               : Ref(attribute(tokz.o, NAME(buf))).o != Py_None)
        return;
      if (scale->size(0) != buf->size(0) || scale->size(1) != buf->size(1) || scale->size(2) != buf->size(2)) return;
    } else {
      if (!tensor_of(scale, o, NAME(_tab_scale), at::kFloat) || scale->dim() != 3 || scale->size(1) != buf->size(3 - d) || scale->size(2) != c) return;
      if (asym ? !tensor_of(zp, o, NAME(_tab_zp), at::kFloat) || zp->sizes() != scale->sizes() : Ref(attribute(o, NAME(_tab_zp))).o != Py_None) return;
    }
    ready = len >= 0 && len <= buf->size(d);
  }
  int64_t heads() const { return buf->size(3 - d); }
  int64_t last_end() const { return k ? integer(PyList_GET_ITEM(ends.o, k - 1)) : 0; }

  // whether a step can go behind the cached ones as it is
  bool takes(PyObject *x) const {
    if (!ready || rule == Rule::kOtherTable || rule == Rule::kOtherToken || !THPVariable_Check(x)) return false;
    const at::Tensor &t = THPVariable_Unpack(x);
    if (!t.is_cuda() || t.device() != buf->device() || t.dim() != 4 || !t.is_contiguous() || t.numel() == 0 || (c % 8 != 0 && rule != Rule::kHeadDim)) return false;
    if (t.scalar_type() != at::kFloat && t.scalar_type() != at::kBFloat16 && t.scalar_type() != at::kHalf) return false;
    if (t.size(0) != buf->size(0) || t.size(3 - d) != heads() || t.size(3) != c || len + t.size(d) > buf->size(d)) return false;
    return per_token(rule) ? scale->size(3) == 1 : k < 16 && k < scale->size(0);
  }
  int mask() const {   // the dims that the rule reduces (VAR_Q/quant.py:78-95)
    switch (rule) {
      case Rule::kHeadDim: return d == 1 ? 0b0011 : 0b0101;
      case Rule::kScale: return 0b1111;
      case Rule::kHead: return d == 1 ? 0b1011 : 0b1101;
      case Rule::kToken: return d == 1 ? 0b1101 : 0b1011;
      default: return 0b1001;
    }
  }
  // Where the scales of a step of n tokens go (see varq_quant_pack_spread): into the step's row of the tables, or to its tokens
  // of the scales per token, [B, H, cap, 1] or [B, cap, H, 1], of every batch entry (and head).
  void spread(int64_t n, int64_t (&m)[7]) const {
    const int64_t B = buf->size(0), H = heads(), cap = buf->size(d);
    auto set = [&](int64_t gi, int64_t go, int64_t ge, int64_t off, int64_t r_in, int64_t r_out, int64_t s_out) {
      const int64_t v[7] = {gi, go, ge, off, r_in, r_out, s_out};
      std::copy(v, v + 7, m);
    };
    if (rule == Rule::kScale) set(1, 0, 0, k * H * c, H * c, 1, 0);
    else if (rule == Rule::kHead) set(1, c, 0, k * H * c, c, 1, 0);
    else if (rule == Rule::kTokenHead) {
      if (d == 2) set(n, cap, 1, len, 1, B, H * cap);
      else set(1, 1, 0, len * H, 1, B, cap * H);
    } else if (d == 2) set(1, 1, 0, len, 1, B * H, cap);
    else set(1, H, 0, len * H, H, B, cap * H);
  }
  // the shape of the scale of a step of n tokens
  std::array<int64_t, 4> scale_shape(int64_t n) const {
    const int64_t H = heads(), s1 = d == 1 ? n : H, s2 = d == 1 ? H : n;
    const bool tokens = per_token(rule);
    return {1, rule == Rule::kTokenHead || (tokens && d == 1) || (!tokens && d == 2 && rule != Rule::kScale) ? s1 : 1,
            rule == Rule::kTokenHead || (tokens && d == 2) || (!tokens && d == 1 && rule != Rule::kScale) ? s2 : 1, rule == Rule::kHeadDim ? c : 1};
  }
  // Where the scale (and `half` behind it the zero-point) of a step of n tokens goes by itself, which is a caller's to change where the
  // cache's copies are not: its stretch of a buffer with one for every token, or step, that the cache has room for (see VAR_Q._own_room).
  // (A tensor for each took 0.9 us of the host apiece, of a step of 20.)
  struct Own {
    Held buf;
    int64_t at, half;
    float *data() const { return ptr<float>(buf) + at; }
  };
  bool own_place(Own &w, int64_t n) const {
    const bool tokens = per_token(rule);
    const int64_t per = rule == Rule::kTokenHead || rule == Rule::kHead ? heads() : 1, slots = tokens ? buf->size(d) : 16;
    if (!tensor_of(w.buf, o, NAME(_own_scales), at::kFloat) || w.buf->device() != buf->device() || w.buf->numel() < slots * per * (asym ? 2 : 1)) return false;
    w.at = (tokens ? len : k) * per;
    w.half = w.buf->numel() / 2;
    return true;
  }
  // the state that quant() followed by cache() leaves, the kernels having written codes and scales in place; own: where the step's
  // scale and zero-point are by themselves (null: its row of the step tables is they)
  void commit(int64_t n, const Own *own = nullptr) const {
    const bool tokens = per_token(rule);
    const auto shape = scale_shape(n);
    const Ref sshape(Py_BuildValue("(LLLL)", (long long)shape[0], (long long)shape[1], (long long)shape[2], (long long)shape[3]));
    set_attribute(o, NAME(_window), Py_BuildValue("(OLLLOOLO)", buf.o, (long long)d, (long long)len, (long long)n, own ? own->buf.o : scale.o,
                                                  !asym ? Py_None : own ? own->buf.o : zp.o, (long long)(own ? -1 - own->at : k), sshape.o));
    Py_INCREF(Py_None);
    set_attribute(o, NAME(_staged), Py_None);
    if (c % 8) {   // (rows that are no whole octets are not dequantized through the tables: see _keep_scales)
      const Ref tokens_n(PyLong_FromLongLong(n)), channels(PyLong_FromLongLong(c));
      Ref(PyObject_CallMethodObjArgs(o, NAME(_keep_scales), tokens_n.o, channels.o, nullptr));
    }
    Py_INCREF(sshape.o);
    set_attribute(o, NAME(_scale_shape), sshape.o);
    set_attribute(item.o, NAME(len), PyLong_FromLongLong(len + n));
    if (tokens) {
      set_attribute(tok.o, NAME(len), PyLong_FromLongLong(len + n));
      if (asym) set_attribute(tokz.o, NAME(len), PyLong_FromLongLong(len + n));
    } else {
      const Ref end(PyLong_FromLongLong(last_end() + n));
      if (PyList_Append(ends.o, end.o)) throw python_error();
    }
  }
};

// quantizer_step(k_quant, k, v_quant | None, v | None) -> whether the step was taken: quant and cache, K and V of a step in the same launches.
// One call with the scales written where the cache keeps them took a step of the rules with scales per token from 72 us of host work
// (two quantizers: reductions, expand, copies into the growing buffers) to that of the shipped rule.
bool take_step(const Quantizer &kq, PyObject *const *a) {
  const bool two = a[2] != Py_None;
  if (!kq.takes(a[1])) return false;
  std::optional<Quantizer> vq;
  const at::Tensor &k = THPVariable_Unpack(a[1]);
  const double eps = real(Ref(attribute(a[0], NAME(eps))).o);
  if (two) {
    vq.emplace(a[2]);
    if (a[0] == a[2] || !vq->takes(a[3])) return false;
    const at::Tensor &v = THPVariable_Unpack(a[3]);
    // (one window of two buffers, one row of two tables)
    if (kq.rule != vq->rule || kq.bits != vq->bits || kq.asym != vq->asym || kq.d != vq->d || kq.len != vq->len || kq.k != vq->k || v.sizes() != k.sizes() ||
        v.scalar_type() != k.scalar_type() || v.device() != k.device() || kq.buf->sizes() != vq->buf->sizes() || eps != real(Ref(attribute(a[2], NAME(eps))).o))
      return false;
  }
  const int64_t sh[4] = {k.size(0), k.size(1), k.size(2), k.size(3)}, d = kq.d, n = sh[d], per_tok = d == 1 ? sh[2] : 1, row = kq.k * kq.heads() * kq.c;
  const int64_t map[3] = {n * per_tok, (kq.buf->size(d) - n) * per_tok, kq.len * per_tok};
  const c10::DeviceGuard guard(k.device());
  const int dt = dtype_code(k), mask = kq.mask(), bits = (int)kq.bits;
  const bool asym = kq.asym, rows = kq.rule == Rule::kHeadDim;
  auto at_row = [&](const Held &h) { return h.t ? ptr<float>(h) + (rows ? row : 0) : nullptr; };
  const void *const x1 = two ? THPVariable_Unpack(a[3]).data_ptr() : nullptr;
  int32_t *const w0 = ptr<int32_t>(kq.buf), *const w1 = two ? ptr<int32_t>(vq->buf) : nullptr;
  float *const s[2] = {at_row(kq.scale), two ? at_row(vq->scale) : nullptr}, *const z[2] = {at_row(kq.zp), two ? at_row(vq->zp) : nullptr};
  int64_t spread[7];
  if (!rows) kq.spread(n, spread);
  Quantizer::Own own[2];
  if (!rows && (!kq.own_place(own[0], n) || (two && !vq->own_place(own[1], n)))) return false;
  const int rc = status_unlocked([&] {
    if (rows) return pack_rows(k, x1, dt, sh, mask, bits, asym, (float)eps, w0, w1, s, z, map);
    float *const s0 = own[0].data(), *const s1 = two ? own[1].data() : nullptr;
    auto step = [&](void *ws, size_t ws_bytes) {
      return varq_quant_pack_spread_room(k.data_ptr(), x1, dt, sh, mask, bits, asym, (float)eps, w0, s[0], z[0], w1, s[1], z[1], s0, asym ? s0 + own[0].half : nullptr, s1,
                                         asym && two ? s1 + own[1].half : nullptr, map, spread, ws, ws_bytes, stream_of(k));
    };
    const int rc = step(nullptr, 0);   // (most steps take one launch, which needs none)
    if (rc != VARQ_ERR_UNSUPPORTED) return rc;
    const size_t ws_bytes = std::max<size_t>(varq_quant_workspace_bytes(sh, mask), 8) * (two ? 2 : 1);
    const at::Tensor ws = empty({(int64_t)ws_bytes}, at::kByte, k);
    return step(ws.data_ptr(), ws_bytes);
  });
  if (!rows && rc == VARQ_ERR_UNSUPPORTED) return false;
  check(rc, "varq_quant_pack");
  kq.commit(n, rows ? nullptr : &own[0]);
  if (two) vq->commit(n, rows ? nullptr : &own[1]);
  return true;
}
PyObject *quantizer_step(PyObject *const *a) {
  const Quantizer kq(a[0]);
  return PyBool_FromLong(take_step(kq, a));
}

// quantizer_use(quantizer, x, out dtype code) -> the dequantized cache with the step behind the earlier ones, or None (nothing done)
PyObject *quantizer_use(PyObject *const *a) {
  const Quantizer z(a[0]);
  const bool tokens = per_token(z.rule), rows = z.rule == Rule::kHeadDim;
  if (!z.takes(a[1]) || z.c % 8 != 0 || (!tokens && z.last_end() != z.len)) Py_RETURN_NONE;
  const at::Tensor &x = THPVariable_Unpack(a[1]);
  const int64_t d = z.d, n = x.size(d), B = x.size(0), H = z.heads(), c = z.c, code = integer(a[2]), len = z.len + n;
  if ((rows && (uintptr_t)x.data_ptr() & 15) || (!tokens && len * (d == 1 ? H : 1) * (c / 8) >= (1ll << 31) - 2048)) Py_RETURN_NONE;
  int32_t ends[16];
  for (int i = 0; i < z.k; ++i) ends[i] = (int32_t)integer(PyList_GET_ITEM(z.ends.o, i));
  ends[z.k] = (int32_t)(z.len + n);
  const int64_t sh[4] = {B, x.size(1), x.size(2), c};
  const float eps = (float)real(Ref(attribute(a[0], NAME(eps))).o);
  const c10::DeviceGuard guard(x.device());
  const int dt = dtype_code(x);
  at::Tensor out;
  auto new_out = [&] { return d == 1 ? empty({B, len, H, c}, dtype_of((int)code), x) : empty({B, H, len, c}, dtype_of((int)code), x); };
  if (!rows) {   // the rules whose scales are not a row of the tables: the step, and the launch that dequantizes what they read
    // (what that launch would refuse, and a result that there is no room for, before the step is in the cache: a caller may try it again)
    if (B > 65535 || (d == 2 ? H : tokens ? len : 1) > 65535)
      raise(g_varq_error, "use_var_q: shape [%lld,%lld,%lld,%lld] exceeds the grid limits", (long long)B, (long long)(d == 1 ? len : H), (long long)(d == 1 ? H : len), (long long)c);
    status_unlocked([&] { out = new_out(); return (int)VARQ_OK; });
    PyObject *const step[4] = {a[0], a[1], Py_None, Py_None};
    if (!take_step(z, step)) Py_RETURN_NONE;
    unlocked("varq_dequant", [&] {
      const int64_t cap = z.buf->size(d);
      if (!tokens)
        return varq_dequant_steps(ptr<int32_t>(z.buf), ptr<float>(z.scale), ptr<float>(z.zp), (int)z.k + 1, ends, (int)B, (int)H, cap, (int)c, (int)z.bits, d == 1,
                                  out.data_ptr(), (int)code, stream_of(x));
      const int64_t heads = z.rule == Rule::kTokenHead;   // (the scales of batch entry 0, and of head 0, serve the others)
      const int64_t shape[4] = {B, d == 1 ? len : H, d == 1 ? H : len, c}, ss[4] = {0, d == 1 ? H : heads * cap, d == 1 ? heads : 1, 0};
      const int64_t in[8] = {shape[0], shape[1], shape[2], H * cap, d == 1 ? H : cap, 1, 0, -1};
      return varq_dequant(ptr<int32_t>(z.buf), nullptr, ptr<float>(z.scale), ptr<float>(z.zp), shape, ss, (int)c, (int)z.bits, in, out.data_ptr(), (int)code, stream_of(x));
    });
    return wrap(out);
  }
  unlocked("varq_quant_step_dequant", [&] {
    const size_t ws_bytes = std::max<size_t>(varq_quant_workspace_bytes(sh, z.mask()), 8);
    const at::Tensor ws = empty({(int64_t)ws_bytes}, at::kByte, x);
    out = new_out();
    return varq_quant_step_dequant(x.data_ptr(), dt, (int)B, (int)H, (int)n, (int)c, d == 1, (int)z.bits, z.asym, eps, ptr<int32_t>(z.buf), z.buf->size(d),
                                   ptr<float>(z.scale), ptr<float>(z.zp), (int)z.k + 1, ends, out.data_ptr(), (int)code, ws.data_ptr(), ws_bytes, stream_of(x));
  });
  z.commit(n);
  return wrap(out);
}

// quantizer_attend(q, k_quant, v_quant, softmax_scale, kv_limit, out) -> out, or None where fused_attention has to look closer
PyObject *quantizer_attend(PyObject *const *a) {
  const Quantizer k(a[1]), v(a[2]);
  if (!k.ready || !v.ready || k.len == 0 || k.d != v.d || k.bits != v.bits || k.len != v.len || k.c != v.c || (k.c != 64 && k.c != 128) || per_token(k.rule) != per_token(v.rule) ||
      k.buf->sizes() != v.buf->sizes() || !THPVariable_Check(a[0]))
    Py_RETURN_NONE;
  const at::Tensor &q = THPVariable_Unpack(a[0]);
  if (!q.is_cuda() || q.dim() != 4 || !q.is_contiguous() || !((q.scalar_type() == at::kHalf && k.c == 64) || q.scalar_type() == at::kBFloat16) ||
      q.size(0) != k.buf->size(0) || q.size(3 - k.d) != k.heads() || q.size(3) != k.c)
    Py_RETURN_NONE;
  const Ref bits(PyLong_FromLongLong(k.bits)), len(PyLong_FromLongLong(k.len)), zero(PyLong_FromLong(0));
  PyObject *const kz = k.asym ? k.zp.o : Py_None, *const vz = v.asym ? v.zp.o : Py_None, *const layout = k.d == 1 ? NAME(BLHc) : NAME(BHLc);
  if (per_token(k.rule)) {
    PyObject *const args[18] = {a[0], k.buf.o, k.scale.o, kz, v.buf.o, v.scale.o, vz, bits.o, bits.o, len.o, a[3], a[4], Py_None, a[5], zero.o, layout, Py_False, Py_None};
    return attn(args);
  }
  const int same = PyObject_RichCompareBool(k.ends.o, v.ends.o, Py_EQ);
  if (same < 0) throw python_error();
  if (!same || k.k == 0 || k.k > 16 || k.last_end() != k.len) Py_RETURN_NONE;
  PyObject *const args[17] = {a[0], k.buf.o, k.scale.o, kz, v.buf.o, v.scale.o, vz, bits.o, len.o, a[3], a[4], Py_None, a[5], k.ends.o, zero.o, layout, Py_None};
  return attn_channel(args);
}

// ---- module -------------------------------------------------------------------------------------
template <PyObject *(*F)(PyObject *const *), int N> PyObject *fixed(PyObject *, PyObject *const *a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  need_args(n, N, "native call");
  return F(a);
  END_HANDLE_TH_ERRORS
}
PyObject *set_error(PyObject *, PyObject *e) {
  Py_INCREF(e);
  Py_XDECREF(g_varq_error);
  g_varq_error = e;
  Py_RETURN_NONE;
}

#define FIXED(name, n) {#name, (PyCFunction)(void (*)(void))fixed<name, n>, METH_FASTCALL, nullptr}
PyMethodDef g_methods[] = {
    FIXED(quant_rows, 5), FIXED(quant_shared, 6), FIXED(pack, 2), FIXED(unpack, 3), FIXED(dequant, 6), FIXED(dequant_steps, 8), FIXED(attn, 18), FIXED(attn_channel, 17),
    FIXED(cache_attend, 9), FIXED(cache_append, 5), FIXED(cache_prepare, 9),
    FIXED(quantizer_step, 4), FIXED(quantizer_use, 3), FIXED(quantizer_attend, 6),
    {"set_error", set_error, METH_O, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) { return PyModule_Create(&g_module); }
