// The Python side's calls, in native code: tensors to descriptors, outputs and workspaces from torch's
// allocator, the current stream, the C ABI call.  svod_amd/ops.py holds the functions a program calls (their
// signatures, option classes and exceptions); each hands its arguments to one function here.
//
// Why native: an op of a short call (a query of a few tokens, a decoder step) takes 3-6 us on the device, and
// the same work done through ctypes objects took 11-17 us of host time an op.
//
// The C ABI is not linked: bind() takes the addresses of its functions from the library ops.load_library() has
// loaded, so a build of it named there is the one that runs.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/EmptyTensor.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <atomic>
#include <cstdint>

#include "../../include/svodk.h"

namespace {

struct Abi {
  decltype(&svodk_attention) attention;
  decltype(&svodk_attention_noalloc) attention_noalloc;
  decltype(&svodk_attention_packed) attention_packed;
  decltype(&svodk_attention_workspace) attention_workspace;
  decltype(&svodk_heads) heads;
  decltype(&svodk_linear) linear;
  decltype(&svodk_layer_norm) layer_norm;
  decltype(&svodk_add_layer_norm) add_layer_norm;
  decltype(&svodk_rms_norm) rms_norm;
  decltype(&svodk_add_rms_norm) add_rms_norm;
  decltype(&svodk_order_rows) order_rows;
};
Abi abi;
PyObject *op_error;  // ops.OpError
PyObject *finish;    // ops._finish(op, status): raises what a status other than 0 stands for
PyObject *dtypes[6];  // torch's dtype objects, by svodk_dtype (for ops._fresh)

// A Python error is set: unwinds to the entry point.
struct Raised {};

// An owned reference.
struct Ref {
  PyObject *p;
  explicit Ref(PyObject *x) : p(x) {
    if (p == nullptr) throw Raised();
  }
  Ref(const Ref &) = delete;
  ~Ref() { Py_XDECREF(p); }
  void take(PyObject *x) {  // `x`'s reference in place of the one held
    if (x == nullptr) throw Raised();
    Py_XDECREF(p);
    p = x;
  }
  operator PyObject *() const { return p; }
};

// The owned references of a call's operands, to its end: an option may be computed when it is asked for, and its tensor's
// memory is the call's until the launch is in the stream.
struct Kept {
  c10::SmallVector<PyObject *, 16> all;
  Kept() = default;
  Kept(const Kept &) = delete;
  ~Kept() {
    for (PyObject *p : all) Py_DECREF(p);
  }
  PyObject *operator()(PyObject *x) {
    if (x == nullptr) throw Raised();
    all.push_back(x);
    return x;
  }
};

[[noreturn]] void op_failed(const char *kind, const char *message) {
  if (PyObject *e = PyObject_CallFunction(op_error, "ss", kind, message)) {
    PyErr_SetObject(op_error, e);
    Py_DECREF(e);
  }
  throw Raised();
}

// Attribute names, interned once.
#define SVODK_NAMES(X)                                                                                              \
  X(causal) X(keys) X(kind) X(tensor) X(window) X(chunk) X(seg_start) X(cache) X(head_start) X(kv_heads) X(row_map) \
  X(appended) X(app_lens) X(bias) X(splits) X(scale) X(batch_live) X(row_order) X(heads) X(head_dim) X(q_norm)      \
  X(k_norm) X(eps) X(rope) X(cos) X(sin) X(act) X(gated) X(residual) X(into)
struct Names {
#define SVODK_NAME(n) PyObject *n;
  SVODK_NAMES(SVODK_NAME)
#undef SVODK_NAME
} names;

PyObject *get(PyObject *o, PyObject *name) { return PyObject_GetAttr(o, name); }

int64_t as_int(PyObject *o) {
  if (PyLong_CheckExact(o)) {
    const long long x = PyLong_AsLongLong(o);
    if (x == -1 && PyErr_Occurred()) throw Raised();
    return x;
  }
  Ref i(PyNumber_Index(o));
  const long long x = PyLong_AsLongLong(i);
  if (x == -1 && PyErr_Occurred()) throw Raised();
  return x;
}
double as_double(PyObject *o) {
  const double x = PyFloat_AsDouble(o);
  if (x == -1.0 && PyErr_Occurred()) throw Raised();
  return x;
}
// `value or 0`, and int(flag).
int32_t int_or_zero(PyObject *o) { return o == Py_None ? 0 : (int32_t)as_int(o); }
int32_t truth(PyObject *o) {
  const int x = PyObject_IsTrue(o);
  if (x < 0) throw Raised();
  return x;
}

const at::Tensor &tensor(PyObject *o) {
  if (!THPVariable_Check(o)) {
    PyErr_Format(PyExc_TypeError, "expected a torch.Tensor, got %.100s", Py_TYPE(o)->tp_name);
    throw Raised();
  }
  return THPVariable_Unpack(o);
}

int dtype_of(at::ScalarType t) {
  switch (t) {
    case at::kBFloat16: return SVODK_BF16;
    case at::kHalf: return SVODK_F16;
    case at::kFloat: return SVODK_F32;
    case at::kInt: return SVODK_I32;
    case at::kLong: return SVODK_I64;
    case at::kBool: return SVODK_BOOL;
    default: return -1;
  }
}

void describe(PyObject *o, svodk_tensor &d) {
  const at::Tensor &t = tensor(o);
  d.dtype = dtype_of(t.scalar_type());
  if (d.dtype < 0) {
    Ref dt(PyObject_GetAttrString(o, "dtype"));
    Ref text(PyUnicode_FromFormat("unsupported element type %S", (PyObject *)dt));
    op_failed("Dtype", PyUnicode_AsUTF8(text));
  }
  const auto sizes = t.sizes();
  if (sizes.size() > 4) {
    Ref text(PyUnicode_FromFormat("rank %zd tensor", (Py_ssize_t)sizes.size()));
    op_failed("Shape", PyUnicode_AsUTF8(text));
  }
  if (!t.is_contiguous()) op_failed("Argument", "operands must be dense row-major (call .contiguous())");
  d.data = t.data_ptr();
  d.rank = (int32_t)sizes.size();
  for (size_t i = 0; i < sizes.size(); i++) d.shape[i] = sizes[i];
}

// A tensor or None.
const svodk_tensor *maybe(PyObject *o, svodk_tensor &d) {
  if (o == Py_None) return nullptr;
  describe(o, d);
  return &d;
}
const svodk_tensor *maybe_attr(Kept &kept, PyObject *o, PyObject *name, svodk_tensor &d) {
  return maybe(kept(get(o, name)), d);
}

void *stream_of(const at::Tensor &t) {
  return t.is_cuda() ? (void *)c10::hip::getCurrentHIPStream(t.device().index()).stream() : nullptr;
}

// at::empty next to `like`.  On its device's own turf without the dispatcher, which is more than half of an
// allocation's 0.7 us: torch's allocator (asked for once, by an at::empty) and the same empty tensor around it.
at::Tensor empty_beside(const at::Tensor &like, at::IntArrayRef shape, at::ScalarType type) {
  static std::atomic<c10::Allocator *> own{nullptr};
  c10::Allocator *allocator = own.load(std::memory_order_acquire);
  if (like.is_cuda() && allocator != nullptr && like.device().index() == c10::hip::current_device() &&
      !at::globalContext().deterministicAlgorithms())
    return at::detail::empty_generic(shape, allocator, c10::DispatchKeySet(c10::DispatchKey::CUDA), type, c10::nullopt);
  at::Tensor t = at::empty(shape, like.options().dtype(type).requires_grad(false).memory_format(c10::nullopt));
  if (t.is_cuda() && allocator == nullptr) own.store(t.storage().allocator(), std::memory_order_release);
  return t;
}

// A new tensor of `shape`: torch's allocator, or ops._fresh where the caller hands that in (`fresh`; it fills what
// it allocates, so that an element a kernel leaves unwritten shows).
PyObject *allocate(PyObject *fresh, at::IntArrayRef shape, at::ScalarType type, PyObject *like) {
  const at::Tensor &t = tensor(like);
  if (fresh == Py_None) return THPVariable_Wrap(empty_beside(t, shape, type));
  Ref sizes(PyTuple_New((Py_ssize_t)shape.size()));
  for (size_t i = 0; i < shape.size(); i++) PyTuple_SET_ITEM((PyObject *)sizes, i, PyLong_FromLongLong(shape[i]));
  Ref device(PyObject_GetAttrString(like, "device"));
  PyObject *dtype = type == at::kByte ? nullptr : dtypes[dtype_of(type)];
  if (dtype == nullptr) {
    Ref torch(PyImport_ImportModule("torch"));
    Ref u8(PyObject_GetAttrString(torch, "uint8"));
    return PyObject_CallFunctionObjArgs(fresh, (PyObject *)sizes, (PyObject *)u8, (PyObject *)device, nullptr);
  }
  return PyObject_CallFunctionObjArgs(fresh, (PyObject *)sizes, dtype, (PyObject *)device, nullptr);
}
PyObject *allocate_like(PyObject *fresh, PyObject *like) {
  const at::Tensor &t = tensor(like);
  return allocate(fresh, t.sizes(), t.scalar_type(), like);
}

// The answer of a call: `out` (whose reference passes to the caller), or the exception of its status.
PyObject *answer(const char *op, int status, Ref &out) {
  if (status != 0) {
    Ref none(PyObject_CallFunction(finish, "si", op, status));
  }
  PyObject *p = out.p;
  out.p = nullptr;
  return p;
}

PyObject *held(PyObject *o) {
  Py_INCREF(o);
  return o;
}

// A tensor's device, the current one while this lives: torch's default stream has the same handle on every device.
class OnDeviceOf {
 public:
  explicit OnDeviceOf(const at::Tensor &t) {
    if (!t.is_cuda()) return;
    static const bool several = c10::hip::device_count() > 1;
    if (!several) return;
    const c10::DeviceIndex now = c10::hip::current_device();
    if (t.device().index() == now) return;
    c10::hip::set_device(t.device().index());
    back_ = now;
  }
  OnDeviceOf(const OnDeviceOf &) = delete;
  ~OnDeviceOf() {
    if (back_ >= 0) (void)c10::hip::SetDevice(back_);
  }

 private:
  c10::DeviceIndex back_ = -1;
};

// The launch itself runs without the interpreter lock, as a ctypes call does: it waits when the device's queue is full.
template <typename F>
int unlocked(const at::Tensor &on, F f) {
  const OnDeviceOf device(on);
  int status;
  Py_BEGIN_ALLOW_THREADS status = f();
  Py_END_ALLOW_THREADS return status;
}

// An Attn's fields as the ABI's struct, with the descriptors that it points to.
struct AttnCall {
  svodk_attn a{};
  svodk_cache c{};
  svodk_tensor keys, seg_start, bias, row_order, row_map, k_app, v_app, app_lens;
  Kept kept;

  explicit AttnCall(PyObject *opts) {
    if (opts == Py_None) return;
    {
      Ref x(get(opts, names.causal));
      a.causal = truth(x);
    }
    {
      Ref mask(get(opts, names.keys));
      Ref kind(get(mask, names.kind));
      a.key_kind = (int32_t)as_int(kind);
      a.keys = maybe_attr(kept, mask, names.tensor, keys);
    }
    {
      Ref w(get(opts, names.window));
      if (w != Py_None) {
        Ref left(PySequence_GetItem(w, 0)), right(PySequence_GetItem(w, 1));
        a.has_window = 1, a.window_left = as_int(left), a.window_right = as_int(right);
      }
    }
    {
      Ref ch(get(opts, names.chunk));
      if (ch != Py_None) {
        Ref size(PySequence_GetItem(ch, 0)), left(PySequence_GetItem(ch, 1)), right(PySequence_GetItem(ch, 2));
        a.has_chunk = 1, a.chunk_size = as_int(size), a.chunk_right = as_int(right);
        if (left != Py_None) a.chunk_has_left = 1, a.chunk_left = as_int(left);
      }
    }
    a.seg_start = maybe_attr(kept, opts, names.seg_start, seg_start);
    {
      Ref cache(get(opts, names.cache));
      if (cache != Py_None) {
        Ref head_start(get(cache, names.head_start)), kv_heads(get(cache, names.kv_heads));
        c.head_start = as_int(head_start), c.kv_heads = as_int(kv_heads);
        c.row_map = maybe_attr(kept, cache, names.row_map, row_map);
        Ref app(get(cache, names.appended));
        if (app != Py_None) {
          c.k_app = maybe(kept(PySequence_GetItem(app, 0)), k_app);
          c.v_app = maybe(kept(PySequence_GetItem(app, 1)), v_app);
        }
        c.app_lens = maybe_attr(kept, cache, names.app_lens, app_lens);
        a.cache = &c;
      }
    }
    a.bias = maybe_attr(kept, opts, names.bias, bias);
    {
      Ref x(get(opts, names.splits));
      a.splits = int_or_zero(x);
    }
    {
      Ref x(get(opts, names.scale));
      if (x != Py_None) a.has_scale = 1, a.scale = (float)as_double(x);
    }
    {
      Ref x(get(opts, names.batch_live));
      a.batch_live = int_or_zero(x);
    }
    a.row_order = maybe_attr(kept, opts, names.row_order, row_order);
  }
};

// The partial tensors of a split call, which the reference op allocates itself
// (tk/src/ops/attention.rs:285-293): here the call's own unless the caller lends them.
struct Workspace {
  PyObject *own = nullptr;
  ~Workspace() { Py_XDECREF(own); }
  void lend(svodk_attn &a, const svodk_tensor &q, const svodk_tensor &k, PyObject *like, PyObject *lent, PyObject *fresh) {
    if (a.splits == 1) return;
    if (lent == Py_None) {
      int64_t need = abi.attention_workspace(&q, &k, &a);
      if (need <= 0) return;
      // Twice that for a decoder step that names no count, which may take more splits then, and the words with which it merges
      // them (svodk.h).
      const int64_t kv_heads = a.cache != nullptr ? a.cache->kv_heads : k.shape[2];
      if (a.splits <= 0 && q.shape[1] * q.shape[2] <= 4 * kv_heads) need *= 2;
      need += 128 * (a.batch_live > 0 ? a.batch_live : q.shape[0]) * kv_heads;
      own = allocate(fresh, {need}, at::kByte, like);
      if (own == nullptr) throw Raised();
      lent = own;
    }
    const at::Tensor &t = tensor(lent);
    a.workspace = t.data_ptr(), a.workspace_bytes = (int64_t)t.numel() * (int64_t)t.element_size();
  }
};

// An entry point's body: C++ exceptions become Python's.
#define SVODK_BEGIN \
  HANDLE_TH_ERRORS  \
  try {
#define SVODK_END          \
  }                        \
  catch (const Raised &) { \
    return nullptr;        \
  }                        \
  END_HANDLE_TH_ERRORS

#define SVODK_ARGS(n, name)                                                          \
  if (nargs != n) {                                                                  \
    PyErr_Format(PyExc_TypeError, name " takes %d arguments, got %zd", n, nargs);    \
    return nullptr;                                                                  \
  }

// (q, k, v, opts, out, workspace, fresh)
PyObject *py_attention(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  SVODK_ARGS(7, "attention")
  SVODK_BEGIN
  PyObject *q = args[0], *fresh = args[6];
  // The op allocates its output at capacity (tk/src/ops/mod.rs:423-429).
  Ref out(args[4] == Py_None ? allocate_like(fresh, q) : held(args[4]));
  AttnCall call(args[3]);
  svodk_tensor qd, kd, vd, od;
  describe(q, qd), describe(args[1], kd), describe(args[2], vd), describe(out, od);
  Workspace ws;
  ws.lend(call.a, qd, kd, q, args[5], fresh);
  void *stream = stream_of(tensor(q));
  const int status = unlocked(tensor(q), [&] { return abi.attention(&qd, &kd, &vd, &call.a, &od, stream); });
  return answer("attention", status, out);
  SVODK_END
}

// (q, k, opts): the bytes of a split call's partial tensors (svodk_attention_workspace), 0 where the call would not split
PyObject *py_attention_workspace(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  SVODK_ARGS(3, "attention_workspace")
  SVODK_BEGIN
  AttnCall call(args[2]);
  svodk_tensor qd, kd;
  describe(args[0], qd), describe(args[1], kd);
  return PyLong_FromLongLong(abi.attention_workspace(&qd, &kd, &call.a));
  SVODK_END
}

// (q, k, v, opts, out)
PyObject *py_attention_noalloc(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  SVODK_ARGS(5, "attention_noalloc")
  SVODK_BEGIN
  AttnCall call(args[3]);
  svodk_tensor qd, kd, vd, od;
  describe(args[0], qd), describe(args[1], kd), describe(args[2], vd), describe(args[4], od);
  void *stream = stream_of(tensor(args[0]));
  const int status = unlocked(tensor(args[0]), [&] { return abi.attention_noalloc(&qd, &kd, &vd, &call.a, &od, stream); });
  Ref out(held(args[4]));
  return answer("attention", status, out);
  SVODK_END
}

// (qkv, heads, kv_heads, opts, out, workspace, fresh)
PyObject *py_attention_packed(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  SVODK_ARGS(7, "attention_packed")
  SVODK_BEGIN
  const at::Tensor &qkv = tensor(args[0]);
  const int64_t heads = as_int(args[1]), kv_heads = as_int(args[2]), slots = heads + 2 * kv_heads;
  PyObject *out_or_none = args[4], *fresh = args[6];
  const bool rows = qkv.dim() == 3;
  if (out_or_none != Py_None)
    out_or_none = held(out_or_none);
  else if (rows && slots > 0 && qkv.size(2) % slots == 0)
    out_or_none = allocate(fresh, {qkv.size(0), qkv.size(1), heads, qkv.size(2) / slots}, qkv.scalar_type(), args[0]);
  else
    out_or_none = allocate(Py_None, {1, 1, 1, 1}, qkv.scalar_type(), args[0]);  // the op rejects the shape itself
  Ref out(out_or_none);
  AttnCall call(args[3]);
  svodk_tensor xd, od;
  describe(args[0], xd), describe(out, od);
  Workspace ws;
  if (call.a.splits > 1 && rows) {
    // The keys' view of the fused rows: [B, T, kv_heads, D].
    const svodk_tensor kd = {xd.data, xd.dtype, 4, {xd.shape[0], xd.shape[1], kv_heads, od.shape[3]}};
    ws.lend(call.a, od, kd, args[0], args[5], fresh);
  }
  void *stream = stream_of(qkv);
  const int status =
      unlocked(qkv, [&] { return abi.attention_packed(&xd, (int32_t)heads, (int32_t)kv_heads, &call.a, &od, stream); });
  return answer("attention", status, out);
  SVODK_END
}

// (qkv, opts, out, fresh); out and the answer: (q, k, v)
PyObject *py_heads(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  SVODK_ARGS(4, "heads")
  SVODK_BEGIN
  const at::Tensor &qkv = tensor(args[0]);
  PyObject *opts = args[1];
  svodk_qkv o{};
  {
    Ref heads(get(opts, names.heads)), kv_heads(get(opts, names.kv_heads)), head_dim(get(opts, names.head_dim));
    o.heads = (int32_t)as_int(heads), o.kv_heads = (int32_t)as_int(kv_heads), o.head_dim = (int32_t)as_int(head_dim);
  }
  PyObject *made = args[2];
  if (made != Py_None) {
    made = held(made);
  } else {
    // With a shape the op will not take: let it word the error; the outputs are never touched.
    const bool rows = qkv.dim() == 3;
    const int64_t b = rows ? qkv.size(0) : 0, t = rows ? qkv.size(1) : 0, d = rows ? o.head_dim : 0;
    PyObject *f = rows ? args[3] : Py_None;
    Ref q(allocate(f, {b, t, rows ? o.heads : 0, d}, qkv.scalar_type(), args[0]));
    Ref k(allocate(f, {b, t, rows ? o.kv_heads : 0, d}, qkv.scalar_type(), args[0]));
    Ref v(allocate(f, {b, t, rows ? o.kv_heads : 0, d}, qkv.scalar_type(), args[0]));
    made = PyTuple_Pack(3, (PyObject *)q, (PyObject *)k, (PyObject *)v);
  }
  Ref out(made);
  svodk_tensor q_norm, k_norm, cos, sin, xd, qd, kd, vd;
  Kept kept;
  o.q_norm = maybe_attr(kept, opts, names.q_norm, q_norm), o.k_norm = maybe_attr(kept, opts, names.k_norm, k_norm);
  {
    Ref eps(get(opts, names.eps)), rope(get(opts, names.rope)), live(get(opts, names.batch_live));
    o.eps = as_double(eps);
    if (rope != Py_None) {
      o.cos = maybe(kept(PySequence_GetItem(rope, 0)), cos);
      o.sin = maybe(kept(PySequence_GetItem(rope, 1)), sin);
    }
    o.batch_live = int_or_zero(live);
  }
  describe(args[0], xd), describe(kept(PySequence_GetItem(out, 0)), qd);
  describe(kept(PySequence_GetItem(out, 1)), kd), describe(kept(PySequence_GetItem(out, 2)), vd);
  void *stream = stream_of(qkv);
  const int status = unlocked(qkv, [&] { return abi.heads(&xd, &o, &qd, &kd, &vd, stream); });
  return answer("heads", status, out);
  SVODK_END
}

// (x, w, opts, out, fresh)
PyObject *py_linear(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  SVODK_ARGS(5, "linear")
  SVODK_BEGIN
  const at::Tensor &x = tensor(args[0]), &w = tensor(args[1]);
  PyObject *opts = args[2];
  Ref out(held(args[3]));
  svodk_linear_opts o{};
  svodk_rotary r{};
  svodk_tensor bias, residual, cos, sin, xd, wd, od;
  Kept kept;
  if (opts != Py_None) {
    Ref gated(get(opts, names.gated));
    o.gated = truth(gated);
    Ref into(get(opts, names.into));
    if (into != Py_None) {
      out.take(PySequence_GetItem(into, 0));
      Ref at(PySequence_GetItem(into, 1));
      o.has_into = 1, o.into_at = as_int(at);
    }
  }
  if (out == Py_None) {
    c10::SmallVector<int64_t, 5> shape(x.sizes().begin(), x.sizes().end());
    if (shape.empty() || w.dim() < 1) {
      PyErr_SetString(PyExc_IndexError, "linear takes an x of rank at least 1 and a w of rank 2");
      throw Raised();
    }
    shape.back() = o.gated ? w.size(0) / 2 : w.size(0);
    out.take(allocate(args[4], shape, x.scalar_type(), args[0]));
  }
  if (opts != Py_None) {
    o.bias = maybe_attr(kept, opts, names.bias, bias), o.residual = maybe_attr(kept, opts, names.residual, residual);
    Ref act(get(opts, names.act)), scale(get(opts, names.scale)), rope(get(opts, names.rope)), live(get(opts, names.batch_live));
    o.act = (int32_t)as_int(act);
    if (scale != Py_None) o.has_scale = 1, o.scale = (float)as_double(scale);
    if (rope != Py_None) {
      r.cos = maybe_attr(kept, rope, names.cos, cos), r.sin = maybe_attr(kept, rope, names.sin, sin);
      Ref heads(get(rope, names.heads)), head_dim(get(rope, names.head_dim));
      r.heads = (int32_t)as_int(heads), r.head_dim = (int32_t)as_int(head_dim);
      o.rope = &r;
    }
    o.batch_live = int_or_zero(live);
  }
  describe(args[0], xd), describe(args[1], wd), describe(out, od);
  void *stream = stream_of(x);
  const int status = unlocked(x, [&] { return abi.linear(&xd, &wd, &o, &od, stream); });
  return answer("linear", status, out);
  SVODK_END
}

// (x, residual, w, b, eps, batch_live, out, fresh) of the norm LAYER and whether there is a residual name; out and
// the answer with a residual: (sum, y)
template <bool LAYER>
PyObject *py_norm(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  SVODK_ARGS(8, "norm")
  SVODK_BEGIN
  PyObject *x = args[0], *residual = args[1], *made = args[6];
  const bool fused = residual != Py_None;
  if (made != Py_None) {
    made = held(made);
  } else if (fused) {
    Ref sum(allocate_like(args[7], x));
    Ref y(allocate_like(args[7], x));
    made = PyTuple_Pack(2, (PyObject *)sum, (PyObject *)y);
  } else {
    made = allocate_like(args[7], x);
  }
  Ref out(made);
  svodk_tensor xd, rd, wd, bd, sd, yd;
  Kept kept;
  describe(x, xd);
  if (fused) describe(residual, rd);
  describe(args[2], wd);
  const svodk_tensor *b = LAYER ? maybe(args[3], bd) : nullptr;
  const double eps = as_double(args[4]);
  const int32_t live = int_or_zero(args[5]);
  if (fused) {
    describe(kept(PySequence_GetItem(out, 0)), sd), describe(kept(PySequence_GetItem(out, 1)), yd);
  } else {
    describe(out, yd);
  }
  void *stream = stream_of(tensor(x));
  const int status = unlocked(tensor(x), [&] {
    if (LAYER)
      return fused ? abi.add_layer_norm(&xd, &rd, &wd, b, eps, live, &sd, &yd, stream)
                   : abi.layer_norm(&xd, &wd, b, eps, live, &yd, stream);
    return fused ? abi.add_rms_norm(&xd, &rd, &wd, eps, live, &sd, &yd, stream) : abi.rms_norm(&xd, &wd, eps, live, &yd, stream);
  });
  return answer(LAYER ? "layer_norm" : "rms_norm", status, out);
  SVODK_END
}

// (keys, out, fresh)
PyObject *py_order_rows(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  SVODK_ARGS(3, "order_rows")
  SVODK_BEGIN
  const at::Tensor &keys = tensor(args[0]);
  Ref out(args[1] == Py_None ? allocate(args[2], keys.sizes().slice(0, keys.dim() > 0 ? 1 : 0), at::kInt, args[0]) : held(args[1]));
  svodk_tensor kd, od;
  describe(args[0], kd), describe(out, od);
  void *stream = stream_of(keys);
  const int status = unlocked(keys, [&] { return abi.order_rows(&kd, &od, stream); });
  return answer("order_rows", status, out);
  SVODK_END
}

// ({function name: address}, OpError, _finish, (dtype by svodk_dtype, ...))
PyObject *py_bind(PyObject *, PyObject *args) {
  PyObject *table, *error, *done, *types;
  if (!PyArg_ParseTuple(args, "O!OOO!", &PyDict_Type, &table, &error, &done, &PyTuple_Type, &types)) return nullptr;
  auto address = [&](const char *name) -> void * {
    PyObject *x = PyDict_GetItemString(table, name);
    void *p = x == nullptr ? nullptr : PyLong_AsVoidPtr(x);
    if (p == nullptr && !PyErr_Occurred()) PyErr_Format(PyExc_KeyError, "%s", name);
    return p;
  };
  Abi found;
#define SVODK_TAKE(f) \
  if ((found.f = (decltype(found.f))address("svodk_" #f)) == nullptr) return nullptr;
  SVODK_TAKE(attention) SVODK_TAKE(attention_noalloc) SVODK_TAKE(attention_packed) SVODK_TAKE(attention_workspace)
  SVODK_TAKE(heads) SVODK_TAKE(linear) SVODK_TAKE(layer_norm) SVODK_TAKE(add_layer_norm) SVODK_TAKE(rms_norm)
  SVODK_TAKE(add_rms_norm) SVODK_TAKE(order_rows)
#undef SVODK_TAKE
  if (PyTuple_GET_SIZE(types) != 6) {
    PyErr_SetString(PyExc_ValueError, "bind takes six dtypes");
    return nullptr;
  }
  abi = found;
  auto keep = [](PyObject *&slot, PyObject *x) {
    Py_INCREF(x);
    Py_XSETREF(slot, x);
  };
  keep(op_error, error), keep(finish, done);
  for (int i = 0; i < 6; i++) keep(dtypes[i], PyTuple_GET_ITEM(types, i));
  Py_RETURN_NONE;
}

#define SVODK_FAST(name, fn) {name, (PyCFunction)(void (*)(void))(fn), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    {"bind", py_bind, METH_VARARGS, nullptr},
    SVODK_FAST("attention", py_attention),
    SVODK_FAST("attention_noalloc", py_attention_noalloc),
    SVODK_FAST("attention_workspace", py_attention_workspace),
    SVODK_FAST("attention_packed", py_attention_packed),
    SVODK_FAST("heads", py_heads),
    SVODK_FAST("linear", py_linear),
    SVODK_FAST("layer_norm", py_norm<true>),
    SVODK_FAST("rms_norm", py_norm<false>),
    SVODK_FAST("order_rows", py_order_rows),
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) {
#define SVODK_INTERN(n) \
  if ((names.n = PyUnicode_InternFromString(#n)) == nullptr) return nullptr;
  SVODK_NAMES(SVODK_INTERN)
#undef SVODK_INTERN
  return PyModule_Create(&module);
}
