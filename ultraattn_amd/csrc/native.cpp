// Python binding of the entry points that are called once per tile, chunk pair or step: argument
// checks, result allocation, device and stream lookup and the C ABI call in one native function.
//
// What bounds a small call is the host: with the same work done in Python around ctypes a 256-token
// forward cost 19 us of host time against 7 us on the device, a chunk pair's forward and backward 57
// against 43.  One positional-only native call per operator leaves the kernel launches themselves
// (about 3 us each) and the allocator.
//
// Everything here works on tensors as torch hands them over; the exceptions are ValueError / TypeError
// for arguments and RuntimeError for a status of the C ABI.  The GIL is released around launches.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <ATen/ATen.h>
#include <ATen/core/CachingHostAllocator.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>
#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>
#include <string>
#include "../../include/ultraattn.h"

namespace {

constexpr int64_t kDim = UA_HEAD_DIM;
struct PyError {};                      // thrown with the Python error set

[[noreturn]] void fail(PyObject* type, const std::string& msg) {
  PyErr_SetString(type, msg.c_str());
  throw PyError();
}
std::string shape_str(at::IntArrayRef s) {
  std::string r = "(";
  for (size_t i = 0; i < s.size(); ++i) r += (i ? ", " : "") + std::to_string(s[i]);
  return r + (s.size() == 1 ? ",)" : ")");
}

const at::Tensor& tensor(PyObject* o, const char* name) {
  if (!THPVariable_Check(o)) fail(PyExc_TypeError, std::string(name) + " must be a tensor, got " + Py_TYPE(o)->tp_name);
  return THPVariable_Unpack(o);
}
double number(PyObject* o) {
  const double x = PyFloat_AsDouble(o);
  if (x == -1.0 && PyErr_Occurred()) throw PyError();
  return x;
}
int64_t integer(PyObject* o) {
  const int64_t x = PyLong_AsLongLong(o);
  if (x == -1 && PyErr_Occurred()) throw PyError();
  return x;
}
bool truth(PyObject* o) {
  const int x = PyObject_IsTrue(o);
  if (x < 0) throw PyError();
  return x != 0;
}
float scale_of(PyObject* o) { return o == Py_None ? (float)std::pow((double)kDim, -0.5) : (float)number(o); }

// A row tensor of the attention kernels: bf16 [B, S, Nh, 128] on the GPU, S a multiple of `multiple`.
void check_rows16(const char* name, const at::Tensor& t, int64_t multiple = UA_TILE) {
  if (!t.is_cuda()) fail(PyExc_ValueError, std::string(name) + " must be a CUDA (HIP) tensor");
  if (t.scalar_type() != at::kBFloat16) fail(PyExc_TypeError, std::string(name) + " must be bfloat16, got " + c10::toString(t.scalar_type()));
  if (t.dim() != 4 || t.size(3) != kDim)
    fail(PyExc_ValueError, std::string(name) + " must be [B, S, Nh, " + std::to_string(kDim) + "], got " + shape_str(t.sizes()));
  if (t.stride(3) != 1) fail(PyExc_ValueError, std::string(name) + ": head_dim axis must be contiguous");
  if (t.size(1) % multiple != 0)
    fail(PyExc_ValueError, std::string(name) + ": sequence length " + std::to_string(t.size(1)) + " is not a multiple of " + std::to_string(multiple));
}
// Row statistics: contiguous fp32 [B, Nh, S] of a row tensor.
void check_stat(const char* name, const at::Tensor& t, const at::Tensor& rows) {
  if (t.dim() != 3 || t.size(0) != rows.size(0) || t.size(1) != rows.size(2) || t.size(2) != rows.size(1) || t.scalar_type() != at::kFloat ||
      !t.is_contiguous()) fail(PyExc_ValueError, std::string(name) + " must be a contiguous fp32 [B, Nh, Sq] tensor");
}
void check_qkv(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v) {
  check_rows16("q", q);
  check_rows16("k", k);
  check_rows16("v", v);
  if (!k.sizes().equals(v.sizes()) || q.size(0) != k.size(0) || q.size(2) != k.size(2))
    fail(PyExc_ValueError, "shape mismatch: q " + shape_str(q.sizes()) + ", k " + shape_str(k.sizes()) + ", v " + shape_str(v.sizes()));
}
void check_like(const char* name, const at::Tensor& t, const at::Tensor& ref) {
  check_rows16(name, t);
  if (!t.sizes().equals(ref.sizes()))
    fail(PyExc_ValueError, std::string(name) + " has shape " + shape_str(t.sizes()) + ", expected " + shape_str(ref.sizes()));
}

struct Strides {
  int64_t s[3];
  explicit Strides(const at::Tensor& t) : s{t.stride(0), t.stride(1), t.stride(2)} {}
  Strides(int64_t b, int64_t t, int64_t h) : s{b, t, h} {}
  operator const int64_t*() const { return s; }
};
at::Tensor like(const at::Tensor& t) { return t.is_contiguous() ? at::empty(t.sizes(), t.options()) : at::empty_like(t); }
at::Tensor stat_of(const at::Tensor& rows) {
  return at::empty({rows.size(0), rows.size(2), rows.size(1)}, rows.options().dtype(at::kFloat));
}

// Result slot: the caller's tensor (returned as the same object) or a new one.
struct Slot {
  PyObject* given;
  at::Tensor t;
  explicit Slot(PyObject* o) : given(o == Py_None ? nullptr : o) {}
  PyObject* wrap() {
    if (given) { Py_INCREF(given); return given; }
    return THPVariable_Wrap(t);
  }
};
template <class... S> PyObject* tuple_of(S&... slots) {
  PyObject* items[] = {slots.wrap()...};
  PyObject* r = PyTuple_New(sizeof...(S));
  for (size_t i = 0; i < sizeof...(S); ++i) PyTuple_SET_ITEM(r, i, items[i]);
  return r;
}

// The tensor's device made current for the call, and its current stream.
struct On {
  int before, device;
  hipStream_t stream;
  explicit On(const at::Tensor& t) : before(c10::hip::current_device()), device(t.get_device()) {
    if (device != before) c10::hip::set_device(device);
    stream = c10::hip::getCurrentHIPStream(device).stream();
  }
  ~On() { if (device != before) c10::hip::set_device(before); }
};
void check_rc(int rc, const char* what) {
  if (rc != UA_OK) fail(PyExc_RuntimeError, std::string(what) + ": " + ua_strerror(rc) + " (code " + std::to_string(rc) + ")");
}
template <class F> void call(const char* what, F&& f) {
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = f();
  Py_END_ALLOW_THREADS
  check_rc(rc, what);
}

// ---- workspaces of cut dense calls ----------------------------------------------------------------
// `cache`: dict (device index, stream handle) -> uint8 tensor.  Calls on one stream run in order, so they can
// share it; it only ever grows.  At most kMaxWorkspaces are kept, the least recently used goes first (stream
// handles come and go).  `captured` (list) keeps those that a captured graph may replay into.
constexpr Py_ssize_t kMaxWorkspaces = 16;
// The launches of a cut call stay together when threads share its stream and so its workspace: each workspace has a mutex
// (one of 64 by its address; calls on different workspaces hardly ever meet).
std::mutex workspace_use[64];
std::unique_lock<std::mutex> hold(const at::Tensor& ws) {
  return ws.defined() ? std::unique_lock<std::mutex>(workspace_use[(reinterpret_cast<uintptr_t>(ws.data_ptr()) >> 9) % 64]) : std::unique_lock<std::mutex>();
}

at::Tensor workspace(PyObject* cache, PyObject* captured, const On& on, const at::Tensor& q, const at::Tensor& k, bool causal, bool backward) {
  const int64_t need = ua_dense_workspace_used((int)q.size(0), (int)q.size(2), (int)q.size(1), (int)k.size(1), causal, backward);
  if (need <= 0) return at::Tensor();
  PyObject* key = Py_BuildValue("(iK)", on.device, (unsigned long long)(uintptr_t)on.stream);
  if (!key) throw PyError();
  PyObject* kept = PyDict_GetItem(cache, key);              // borrowed
  at::Tensor ws;
  if (kept) ws = THPVariable_Unpack(kept);
  if (!kept || ws.numel() < need || PyDict_GET_SIZE(cache) > 1) {          // more than one: this one becomes the most recently used
    if (!kept || ws.numel() < need) ws = at::empty({need}, q.options().dtype(at::kByte));
    PyObject* obj = THPVariable_Wrap(ws);
    if (kept) PyDict_DelItem(cache, key);
    PyDict_SetItem(cache, key, obj);
    Py_DECREF(obj);
    while (PyDict_GET_SIZE(cache) > kMaxWorkspaces) {
      PyObject *k0, *v0;
      Py_ssize_t at = 0;
      PyDict_Next(cache, &at, &k0, &v0);
      Py_INCREF(k0);
      PyDict_DelItem(cache, k0);
      Py_DECREF(k0);
    }
  }
  Py_DECREF(key);
  if (c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None) {
    PyObject* obj = THPVariable_Wrap(ws);
    bool there = false;
    for (Py_ssize_t i = 0; i < PyList_GET_SIZE(captured) && !there; ++i) there = PyList_GET_ITEM(captured, i) == obj;
    if (!there) PyList_Append(captured, obj);               // outlives its cache entry: the graph keeps writing to it
    Py_DECREF(obj);
  }
  return ws;
}
// Per-device lookups of the library, done once and outside any capture.
void init_device(int device) {
  static bool done[64] = {};
  if (device >= 0 && device < 64 && done[device]) return;
  check_rc(ua_init(), "ua_init");
  if (device >= 0 && device < 64) done[device] = true;
}

at::Tensor delta_of(const at::Tensor& out, const at::Tensor& dout, at::Tensor delta) {
  check_rows16("out", out, 1);
  check_rows16("dout", dout, 1);
  if (!out.sizes().equals(dout.sizes())) fail(PyExc_ValueError, "out and dout must have the same shape");
  if (!delta.defined()) delta = stat_of(out);
  const On on(out);
  call("ua_bsa_bwd_delta", [&] {
    return ua_bsa_bwd_delta(out.data_ptr(), dout.data_ptr(), (float*)delta.data_ptr(), (int)out.size(0), (int)out.size(1), (int)out.size(2), (int)kDim,
                            Strides(out), Strides(dout), on.stream);
  });
  return delta;
}

// ---- operators ----------------------------------------------------------------------------------------
// dense_forward(q, k, v, softmax_scale, causal, out, cache, captured) -> (out, lse)
PyObject* dense_forward(PyObject* const* a) {
  const at::Tensor &q = tensor(a[0], "q"), &k = tensor(a[1], "k"), &v = tensor(a[2], "v");
  check_qkv(q, k, v);
  const float scale = scale_of(a[3]);
  const bool causal = truth(a[4]);
  Slot out(a[5]), lse(Py_None);
  if (out.given) {
    out.t = tensor(out.given, "out");
    check_rows16("out", out.t);
    if (!out.t.sizes().equals(q.sizes())) fail(PyExc_ValueError, "out must have q's shape");
  } else {
    out.t = like(q);
  }
  lse.t = stat_of(q);
  const On on(q);
  init_device(on.device);
  // (an output that is not contiguous is not cut)
  const at::Tensor ws = out.t.is_contiguous() ? workspace(a[6], a[7], on, q, k, causal, false) : at::Tensor();
  call("ua_dense_fwd", [&] {
    const auto held = hold(ws);
    return ua_dense_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.t.data_ptr(), (float*)lse.t.data_ptr(), (int)q.size(0), (int)q.size(2),
                        (int)q.size(1), (int)k.size(1), (int)kDim, Strides(q), Strides(k), Strides(v), Strides(out.t), scale, causal,
                        ws.defined() ? ws.data_ptr() : q.data_ptr(), ws.defined() ? ws.numel() : 0, on.stream);    // (NULL would rule out several groups)
  });
  return tuple_of(out, lse);
}

struct BwdArgs {
  const at::Tensor &dout, &q, &k, &v, &lse;
  Slot dq, dk, dv, delta;
  // a: dout, q, k, v, out, lse, dq, dk, dv, softmax_d
  explicit BwdArgs(PyObject* const* a, const char* lse_name)
      : dout(tensor(a[0], "dout")), q(tensor(a[1], "q")), k(tensor(a[2], "k")), v(tensor(a[3], "v")), lse(tensor(a[5], lse_name)),
        dq(a[6]), dk(a[7]), dv(a[8]), delta(a[9]) {
    check_qkv(q, k, v);
    check_rows16("dout", dout);
    if (!dout.sizes().equals(q.sizes())) fail(PyExc_ValueError, "dout must have q's shape");
    check_stat(lse_name, lse, q);
    if (delta.given) {
      delta.t = tensor(delta.given, "softmax_d");
      check_stat("softmax_d", delta.t, q);
    } else if (a[4] == Py_None) {
      fail(PyExc_ValueError, "either out or softmax_d is required");
    }
  }
  void allocate(PyObject* out) {
    fill(dq, "dq", q);
    fill(dk, "dk", k);
    fill(dv, "dv", v);
    if (!delta.given) delta.t = delta_of(tensor(out, "out"), dout, at::Tensor());
  }
  static void fill(Slot& s, const char* name, const at::Tensor& ref) {
    if (s.given) check_like(name, s.t = tensor(s.given, name), ref);
    else s.t = like(ref);
  }
};

// dense_backward(dout, q, k, v, out, lse, dq, dk, dv, softmax_d, softmax_scale, causal, cache, captured) -> (dq, dk, dv, softmax_d)
PyObject* dense_backward(PyObject* const* a) {
  BwdArgs x(a, "softmax_lse");
  const float scale = scale_of(a[10]);
  const bool causal = truth(a[11]);
  x.allocate(a[4]);
  const On on(x.q);
  init_device(on.device);
  const at::Tensor ws = workspace(a[12], a[13], on, x.q, x.k, causal, true);
  call("ua_dense_bwd", [&] {
    const auto held = hold(ws);
    return ua_dense_bwd(x.dout.data_ptr(), x.q.data_ptr(), x.k.data_ptr(), x.v.data_ptr(), (const float*)x.lse.data_ptr(),
                        (const float*)x.delta.t.data_ptr(), x.dq.t.data_ptr(), x.dk.t.data_ptr(), x.dv.t.data_ptr(), (int)x.q.size(0), (int)x.q.size(2),
                        (int)x.q.size(1), (int)x.k.size(1), (int)kDim, Strides(x.q), Strides(x.k), Strides(x.v), Strides(x.dout), Strides(x.dq.t),
                        Strides(x.dk.t), Strides(x.dv.t), scale, causal, ws.defined() ? ws.data_ptr() : x.q.data_ptr(), ws.defined() ? ws.numel() : 0, on.stream);
  });
  return tuple_of(x.dq, x.dk, x.dv, x.delta);
}

// Tile lists in one device buffer of 32-bit words: row_ptr, col_ptr, q_order, k_order, col_idx, row_idx, flag, cflag (the
// flags four to a word), so that a list travels in one copy.  Behind them may lie a second pair of launch orders, the
// longest lines first, for launches of up to kShortLaunch lines: their operands stay in the caches in any order, and how
// evenly the walks end decides.  Strided 8k, 16 heads: forward 135 -> 122 us; 32k, 8 heads: 452 -> 422; 64k: 1367 -> 1318
// (4096 lines); from 8192 lines on the shared tiles of the first order win (32k, 32 heads: 1772, 1847).
constexpr int64_t kShortLaunch = 4096;
struct Lists {
  int64_t at[11];            // first word of each array; at[8] = words without, at[10] with the second orders
  const int32_t *row_ptr, *col_ptr, *q_order, *k_order, *col_idx, *row_idx;
  const uint8_t *flag, *cflag;
  Lists(int64_t nqt, int64_t nkt, int64_t nnz) {
    const int64_t words[8] = {nqt + 1, nkt + 1, nqt, nkt, nnz, nnz, (nnz + 3) / 4, (nnz + 3) / 4};
    at[0] = 0;
    for (int i = 0; i < 8; ++i) at[i + 1] = at[i] + words[i];
    at[9] = at[8] + nqt;
    at[10] = at[9] + nkt;
  }
  void point_into(const void* base) {
    const int32_t* p = (const int32_t*)base;
    row_ptr = p + at[0]; col_ptr = p + at[1]; q_order = p + at[2]; k_order = p + at[3]; col_idx = p + at[4]; row_idx = p + at[5];
    flag = (const uint8_t*)(p + at[6]); cflag = (const uint8_t*)(p + at[7]);
  }
  Lists(PyObject* buf, int64_t nqt, int64_t nkt, int64_t nnz, int64_t heads) : Lists(nqt, nkt, nnz) {
    const at::Tensor& t = tensor(buf, "tile list");
    if (nqt <= 0 || nkt <= 0 || nnz < 0 || !t.is_cuda() || t.scalar_type() != at::kInt || !t.is_contiguous() || t.numel() < at[8])
      fail(PyExc_ValueError, "the tile list must be a contiguous int32 CUDA tensor that holds all of its arrays");
    point_into(t.data_ptr());
    if (t.numel() >= at[10]) {
      if (heads * nqt <= kShortLaunch) q_order = (const int32_t*)t.data_ptr() + at[8];
      if (heads * nkt <= kShortLaunch) k_order = (const int32_t*)t.data_ptr() + at[9];
    }
  }
};
void check_grid(const at::Tensor& q, const at::Tensor& k, int64_t nqt, int64_t nkt) {
  if (nqt * UA_TILE != q.size(1) || nkt * UA_TILE != k.size(1))
    fail(PyExc_ValueError, "tile list is " + std::to_string(nqt) + " x " + std::to_string(nkt) + " tiles (" + std::to_string(nqt * UA_TILE) + " x " +
                               std::to_string(nkt * UA_TILE) + " tokens) but q/k have " + std::to_string(q.size(1)) + " / " +
                               std::to_string(k.size(1)) + " tokens");
}

// bsa_forward(q, k, v, lists, n_qtiles, n_ktiles, nnz, softmax_scale, out, lse) -> (out, lse)
PyObject* bsa_forward(PyObject* const* a) {
  const at::Tensor &q = tensor(a[0], "q"), &k = tensor(a[1], "k"), &v = tensor(a[2], "v");
  check_qkv(q, k, v);
  const int64_t nqt = integer(a[4]), nkt = integer(a[5]), nnz = integer(a[6]);
  const Lists l(a[3], nqt, nkt, nnz, q.size(0) * q.size(2));
  check_grid(q, k, nqt, nkt);
  const float scale = scale_of(a[7]);
  Slot out(a[8]), lse(a[9]);
  if (out.given) {
    out.t = tensor(out.given, "out");
    check_rows16("out", out.t);
    if (!out.t.sizes().equals(q.sizes())) fail(PyExc_ValueError, "out must have q's shape");
  } else {
    out.t = like(q);
  }
  if (lse.given) check_stat("lse", lse.t = tensor(lse.given, "lse"), q);
  else lse.t = stat_of(q);
  const On on(q);
  call("ua_bsa_fwd", [&] {
    return ua_bsa_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.t.data_ptr(), (float*)lse.t.data_ptr(), l.row_ptr, l.col_idx, l.flag, l.q_order,
                      (int)q.size(0), (int)q.size(2), (int)nqt, (int)nkt, (int)nnz, (int)kDim, Strides(q), Strides(k), Strides(v), Strides(out.t),
                      scale, on.stream);
  });
  return tuple_of(out, lse);
}

// bsa_backward(dout, q, k, v, out, lse, dq, dk, dv, softmax_d, lists, n_qtiles, n_ktiles, nnz, softmax_scale) -> (dq, dk, dv)
PyObject* bsa_backward(PyObject* const* a) {
  const int64_t nqt = integer(a[11]), nkt = integer(a[12]), nnz = integer(a[13]);
  const float scale = scale_of(a[14]);
  BwdArgs x(a, "lse");
  const Lists l(a[10], nqt, nkt, nnz, x.q.size(0) * x.q.size(2));
  check_grid(x.q, x.k, nqt, nkt);
  x.allocate(a[4]);
  const On on(x.q);
  call("ua_bsa_bwd", [&] {
    return ua_bsa_bwd(x.q.data_ptr(), x.k.data_ptr(), x.v.data_ptr(), x.dout.data_ptr(), (const float*)x.lse.data_ptr(),
                      (const float*)x.delta.t.data_ptr(), x.dq.t.data_ptr(), x.dk.t.data_ptr(), x.dv.t.data_ptr(), l.row_ptr, l.col_idx, l.flag,
                      l.q_order, l.col_ptr, l.row_idx, l.cflag, l.k_order, (int)x.q.size(0), (int)x.q.size(2), (int)nqt, (int)nkt, (int)nnz,
                      (int)kDim, Strides(x.q), Strides(x.k), Strides(x.v), Strides(x.dout), Strides(x.dq.t), Strides(x.dk.t), Strides(x.dv.t),
                      scale, on.stream);
  });
  return tuple_of(x.dq, x.dk, x.dv);
}

// ---- tile lists ---------------------------------------------------------------------------------------
// `bytes` rounded up to whole 16-byte vectors.
at::Tensor pinned(int64_t bytes, at::ScalarType dt) {
  return at::empty({(bytes + 15) / 16 * 16 / (int64_t)c10::elementSize(dt)}, at::TensorOptions().dtype(dt).pinned_memory(true));
}
// A pinned tensor on the device, in stream order; torch keeps the pinned block until then.  What is small goes there by a kernel of
// this library, which the next kernel follows without a signal in between (mask per call, strided 8k, 8 heads: 73.6 -> 71.9 us).
constexpr int64_t kCopyInBytes = 1 << 20;
at::Tensor to_device(const at::Tensor& host, int device) {
  const int64_t bytes = host.numel() * host.element_size();
  if (bytes > kCopyInBytes) return host.to(at::Device(at::kCUDA, (c10::DeviceIndex)device), host.scalar_type(), /*non_blocking=*/true);
  const at::Tensor t = at::empty(host.sizes(), host.options().pinned_memory(false).device(at::Device(at::kCUDA, (c10::DeviceIndex)device)));
  const c10::hip::HIPStream st = c10::hip::getCurrentHIPStream((c10::DeviceIndex)device);
  call("ua_copy_in", [&] { return ua_copy_in(t.data_ptr(), host.data_ptr(), bytes, st.stream()); });
  at::getHostAllocator(at::kCUDA)->record_event(host.data_ptr(), host.storage().data_ptr().get_context(),
                                            c10::Stream(c10::Stream::UNSAFE, t.device(), st.id()));
  return t;
}

// lists_from_mask(mask, rows, columns, rate, device) -> (buffer, n_qtiles, n_ktiles, nnz): the lists of a mask that comes with the
// call (mask: host bytes, row major).
//
// A short list is built here and copied over: the device then does nothing but the copy (2 us), while
// the host still is far ahead of the kernel that will use it.  Host time grows with the list (44 us at 1000
// tiles, 110 at 8000, 820 at 74000); from kHostTiles on the mask is copied instead and the device builds the
// list in about 20 us.
constexpr int64_t kHostTiles = 4096;
PyObject* lists_from_mask(PyObject* const* a) {
  const int64_t nqb = integer(a[1]), nkb = integer(a[2]), rate = integer(a[3]), device = integer(a[4]);
  struct View {
    Py_buffer b;
    explicit View(PyObject* o) { if (PyObject_GetBuffer(o, &b, PyBUF_C_CONTIGUOUS)) throw PyError(); }
    ~View() { PyBuffer_Release(&b); }
  } mask(a[0]);
  if (nqb <= 0 || nkb <= 0 || mask.b.len != nqb * nkb) fail(PyExc_ValueError, "the block mask must hold rows * columns bytes");
  const uint8_t* bytes = (const uint8_t*)mask.b.buf;
  int64_t nqt, nkt, nnz;
  check_rc(ua_tilelist_size(bytes, (int)nqb, (int)nkb, (int)rate, &nqt, &nkt, &nnz), "ua_tilelist_size");
  const int before = c10::hip::current_device();
  struct Restore { int d; ~Restore() { if (c10::hip::current_device() != d) c10::hip::set_device(d); } } restore{before};
  if (device != before) c10::hip::set_device((int)device);
  if (c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None)
    fail(PyExc_RuntimeError, "a tile list must be built before the stream is captured into a graph");
  Lists l(nqt, nkt, nnz);
  at::Tensor buf;
  if (nnz <= kHostTiles) {
    const at::Tensor host = pinned(l.at[10] * 4, at::kInt);
    l.point_into(host.data_ptr());
    call("ua_tilelist_build", [&] {
      return ua_tilelist_build(bytes, (int)nqb, (int)nkb, (int)rate, (int32_t*)l.row_ptr, (int32_t*)l.col_idx, (uint8_t*)l.flag, (int32_t*)l.col_ptr,
                               (int32_t*)l.row_idx, (uint8_t*)l.cflag, (int32_t*)l.q_order, (int32_t*)l.k_order);
    });
    auto longest_first = [&](const int32_t* ptr, int64_t to, int64_t n) {
      int32_t* order = (int32_t*)host.data_ptr() + to;
      for (int64_t i = 0; i < n; ++i) order[i] = (int32_t)i;
      std::stable_sort(order, order + n, [ptr](int32_t i, int32_t j) { return ptr[i + 1] - ptr[i] > ptr[j + 1] - ptr[j]; });
    };
    longest_first(l.row_ptr, l.at[8], nqt);
    longest_first(l.col_ptr, l.at[9], nkt);
    buf = to_device(host, (int)device);
  } else {
    const at::Tensor host = pinned(nqb * nkb, at::kByte);
    memcpy(host.data_ptr(), bytes, (size_t)(nqb * nkb));
    const at::Tensor m = to_device(host, (int)device);
    buf = at::empty({l.at[8]}, m.options().dtype(at::kInt));
    const int64_t scratch = ua_tilelist_scratch_bytes((int)nqb, (int)nkb, (int)rate), work_words = (nqt + nkt + 7 + 3) / 4 * 4;      // (the scratch on a 16-byte boundary)
    const at::Tensor work = at::empty({work_words + scratch / 4}, buf.options());
    l.point_into(buf.data_ptr());
    const hipStream_t st = c10::hip::getCurrentHIPStream((c10::DeviceIndex)device).stream();
    call("ua_tilelist_build_device", [&] {
      return ua_tilelist_build_device_scratch((const uint8_t*)m.data_ptr(), (int)nqb, (int)nkb, (int)rate, (int32_t*)l.row_ptr, (int32_t*)l.col_idx,
                                              (uint8_t*)l.flag, (int32_t*)l.col_ptr, (int32_t*)l.row_idx, (uint8_t*)l.cflag, (int32_t*)l.q_order,
                                              (int32_t*)l.k_order, (int32_t*)work.data_ptr(), (int32_t*)work.data_ptr() + work_words, scratch, st);
    });
  }
  return Py_BuildValue("(NLLL)", THPVariable_Wrap(buf), (long long)nqt, (long long)nkt, (long long)nnz);
}

// build_lists_device(mask, rate, nnz) -> (row_ptr, col_idx, flag, col_ptr, row_idx, cflag, q_order, k_order, work) of a device mask; nnz < 0:
// sized for every tile active
PyObject* build_lists_device(PyObject* const* a) {
  const at::Tensor& m = tensor(a[0], "block_mask_dev");
  const int64_t rate = integer(a[1]), given = integer(a[2]);
  if (m.scalar_type() != at::kByte || m.dim() != 2 || !m.is_cuda() || !m.is_contiguous())
    fail(PyExc_ValueError, "block_mask_dev must be a contiguous 2-D uint8 CUDA tensor");
  const int64_t nqt = m.size(0) * rate, nkt = m.size(1) * rate, cap = given >= 0 ? given : nqt * nkt;
  const int64_t room = ((cap > 1 ? cap : 1) + 3) / 4 * 4;         // not empty, whole 32-bit words of flags
  // One allocation that the nine results and the scratch are parts of, each on a 64-byte boundary: nine of them took a third of the call.
  const int64_t scratch = ua_tilelist_scratch_bytes((int)m.size(0), (int)m.size(1), (int)rate);
  const int64_t bytes[10] = {4 * (nqt + 1), 4 * room, room, 4 * (nkt + 1), 4 * room, room, 4 * nqt, 4 * nkt, 4 * (nqt + nkt + 7), scratch};
  int64_t at_byte[11] = {0};
  for (int i = 0; i < 10; ++i) at_byte[i + 1] = at_byte[i] + (bytes[i] + 63) / 64 * 64;
  const at::Tensor all = at::empty({at_byte[10]}, m.options());
  at::Tensor t[9];
  for (int i = 0; i < 9; ++i) {
    const bool flags = i == 2 || i == 5, list = flags || i == 1 || i == 4;
    const int64_t size = flags ? 1 : 4;
    auto impl = c10::make_intrusive<at::TensorImpl>(c10::Storage(all.storage()), all.key_set(), c10::scalarTypeToTypeMeta(flags ? at::kByte : at::kInt));
    impl->set_storage_offset(at_byte[i] / size);
    impl->set_sizes_contiguous({list ? cap : bytes[i] / size});
    t[i] = at::Tensor(std::move(impl));
  }
  void* const base = all.data_ptr();
  auto part = [&](int i) { return (void*)((char*)base + at_byte[i]); };
  const On on(m);
  call("ua_tilelist_build_device", [&] {
    return ua_tilelist_build_device_scratch((const uint8_t*)m.data_ptr(), (int)m.size(0), (int)m.size(1), (int)rate, (int32_t*)part(0), (int32_t*)part(1),
                                            (uint8_t*)part(2), (int32_t*)part(3), (int32_t*)part(4), (uint8_t*)part(5), (int32_t*)part(6),
                                            (int32_t*)part(7), (int32_t*)part(8), part(9), scratch, on.stream);
  });
  PyObject* r = PyTuple_New(9);
  for (int i = 0; i < 9; ++i) PyTuple_SET_ITEM(r, i, THPVariable_Wrap(t[i]));
  return r;
}

// delta(out, dout, delta) -> delta
PyObject* delta(PyObject* const* a) {
  Slot d(a[2]);
  if (d.given) d.t = tensor(d.given, "delta");
  d.t = delta_of(tensor(a[0], "out"), tensor(a[1], "dout"), d.t);
  return d.wrap();
}

// grad_accumulate(partial, out, acc, init_from_out)
PyObject* grad_accumulate(PyObject* const* a) {
  const at::Tensor& partial = tensor(a[0], "partial");
  auto flat = [&](const char* name, PyObject* o, at::ScalarType dt, const char* dt_name) -> void* {
    if (o == Py_None) return nullptr;
    const at::Tensor& t = tensor(o, name);
    if (!t.is_cuda() || t.scalar_type() != dt || !t.is_contiguous() || t.numel() != partial.numel())
      fail(PyExc_ValueError, std::string(name) + " must be a contiguous " + dt_name + " CUDA tensor of " + std::to_string(partial.numel()) + " elements");
    return t.data_ptr();
  };
  const void* p = flat("partial", a[0], at::kBFloat16, "torch.bfloat16");
  void* out = flat("out", a[1], at::kBFloat16, "torch.bfloat16");
  float* acc = (float*)flat("acc", a[2], at::kFloat, "torch.float32");
  const bool init = truth(a[3]);
  const On on(partial);
  call("ua_grad_accumulate", [&] { return ua_grad_accumulate(acc, p, out, partial.numel(), init, on.stream); });
  Py_RETURN_NONE;
}

// Partial tensors given as a Python list or tuple.
struct Items {
  PyObject* seq;
  explicit Items(PyObject* o) : seq(PySequence_Fast(o, "expected a sequence of tensors")) { if (!seq) throw PyError(); }
  ~Items() { Py_DECREF(seq); }
  int64_t size() const { return PySequence_Fast_GET_SIZE(seq); }
  const at::Tensor& at(int64_t i, const char* name) const { return tensor(PySequence_Fast_GET_ITEM(seq, i), name); }
};

// merge(outs, lses, out, lse) -> (out, lse)
PyObject* merge(PyObject* const* a) {
  const Items outs(a[0]), lses(a[1]);
  const int64_t n = outs.size();
  if (n == 0 || n != lses.size()) fail(PyExc_ValueError, "need as many lses as outs, at least one");
  const at::Tensor& first = outs.at(0, "partial out");
  if (n > UA_MAX_PARTS) check_rc(UA_ERR_UNSUPPORTED, "ua_merge");
  const void* op[UA_MAX_PARTS];
  const float* lp[UA_MAX_PARTS];
  auto is_stat = [&](const at::Tensor& l) {
    return l.dim() == 3 && l.size(0) == first.size(0) && l.size(1) == first.size(2) && l.size(2) == first.size(1) && l.scalar_type() == at::kFloat &&
           l.is_contiguous();
  };
  for (int64_t i = 0; i < n; ++i) {
    const at::Tensor &o = outs.at(i, "partial out"), &l = lses.at(i, "partial lse");
    check_rows16("partial out", o, 1);
    if (!o.sizes().equals(first.sizes()) || !o.is_contiguous()) fail(PyExc_ValueError, "partial outs must be contiguous and of equal shape");
    if (!is_stat(l)) fail(PyExc_ValueError, "partial lses must be contiguous fp32 [B, Nh, S]");
    op[i] = o.data_ptr();
    lp[i] = (const float*)l.data_ptr();
  }
  Slot out(a[2]), lse(a[3]);
  out.t = out.given ? tensor(out.given, "out") : like(first);
  lse.t = lse.given ? tensor(lse.given, "lse") : stat_of(first);
  if (!out.t.sizes().equals(first.sizes()) || !out.t.is_contiguous() || out.t.scalar_type() != at::kBFloat16)
    fail(PyExc_ValueError, "out must be a contiguous bf16 tensor of the partials' shape");
  if (!is_stat(lse.t)) fail(PyExc_ValueError, "lse must be a contiguous fp32 [B, Nh, S] tensor");
  const On on(out.t);
  call("ua_merge", [&] {
    return ua_merge(op, lp, (int)n, out.t.data_ptr(), (float*)lse.t.data_ptr(), (int)first.size(0), (int)first.size(1), (int)first.size(2), (int)kDim,
                    on.stream);
  });
  return tuple_of(out, lse);
}

// grad_sum(parts, out, scale) -> out
PyObject* grad_sum(PyObject* const* a) {
  const Items parts(a[0]);
  const int64_t n = parts.size();
  if (n == 0) fail(PyExc_ValueError, "need at least one partial gradient");
  const at::Tensor& first = parts.at(0, "partial gradient");
  const at::ScalarType dt = first.scalar_type();
  if (dt != at::kBFloat16 && dt != at::kFloat) fail(PyExc_TypeError, "partial gradients must be bfloat16 or float32");
  const void* pp[UA_MAX_PARTS];
  for (int64_t i = 0; i < n; ++i) {
    const at::Tensor& t = parts.at(i, "partial gradient");
    if (!t.is_cuda() || t.scalar_type() != dt || !t.sizes().equals(first.sizes()) || !t.is_contiguous() || t.dim() != 4 || t.size(3) != kDim)
      fail(PyExc_ValueError, "partial gradients must be contiguous [B, S, Nh, 128] CUDA tensors of one dtype and shape");
    if (i < UA_MAX_PARTS) pp[i] = t.data_ptr();
  }
  if (n > UA_MAX_PARTS) check_rc(UA_ERR_UNSUPPORTED, "ua_grad_sum");
  Slot out(a[1]);
  out.t = out.given ? tensor(out.given, "out") : at::empty(first.sizes(), first.options().dtype(at::kBFloat16));
  check_rows16("out", out.t, 1);
  if (!out.t.sizes().equals(first.sizes())) fail(PyExc_ValueError, "out must have the partials' shape");
  const float scale = (float)number(a[2]);
  const On on(out.t);
  call("ua_grad_sum", [&] {
    return ua_grad_sum(pp, (int)n, dt == at::kFloat, out.t.data_ptr(), (int)first.size(0), (int)first.size(1), (int)first.size(2), (int)kDim,
                       Strides(out.t), scale, on.stream);
  });
  return out.wrap();
}

void check_rows_any(const char* name, const at::Tensor& t) {
  if (!t.is_cuda() || (t.scalar_type() != at::kBFloat16 && t.scalar_type() != at::kFloat))
    fail(PyExc_TypeError, std::string(name) + " must be a bfloat16 or float32 CUDA tensor");
  if (t.dim() != 4 || t.size(3) != kDim || t.stride(3) != 1)
    fail(PyExc_ValueError, std::string(name) + " must be [B, S, Nh, " + std::to_string(kDim) + "] with a contiguous last axis, got " + shape_str(t.sizes()));
}
// (batch, token, head) strides of the statistics of `rows`, given as [B, S, Nh, 1] or [B, Nh, S].
Strides stat_strides(const char* name, const at::Tensor& t, const at::Tensor& rows) {
  const int64_t B = rows.size(0), S = rows.size(1), Nh = rows.size(2);
  if (t.scalar_type() != at::kFloat || !t.is_cuda()) fail(PyExc_TypeError, std::string(name) + " must be a float32 CUDA tensor");
  if (t.dim() == 4 && t.size(0) == B && t.size(1) == S && t.size(2) == Nh && t.size(3) == 1) return Strides(t);
  if (t.dim() == 3 && t.size(0) == B && t.size(1) == Nh && t.size(2) == S) return Strides(t.stride(0), t.stride(2), t.stride(1));
  fail(PyExc_ValueError, std::string(name) + " must be [B, S, Nh, 1] or [B, Nh, S] = (" + std::to_string(B) + ", " + std::to_string(S) + ", " +
                             std::to_string(Nh) + "), got " + shape_str(t.sizes()));
}

// merge_update(out, lse, block_out, block_lse, in_place) -> (new_out, new_lse): fp32 rows in new tensors, or out and lse themselves
PyObject* merge_update(PyObject* const* a) {
  const at::Tensor &out = tensor(a[0], "out"), &lse = tensor(a[1], "lse"), &blk = tensor(a[2], "block_out"), &blk_lse = tensor(a[3], "block_lse");
  check_rows_any("out", out);
  check_rows_any("block_out", blk);
  if (!blk.sizes().equals(out.sizes()))
    fail(PyExc_ValueError, "block_out is " + shape_str(blk.sizes()) + ", the rows to update are " + shape_str(out.sizes()));
  const Strides ls = stat_strides("lse", lse, out), bls = stat_strides("block_lse", blk_lse, out);
  const bool in_place = truth(a[4]);
  Slot new_out(in_place ? a[0] : Py_None), new_lse(in_place ? a[1] : Py_None);
  new_out.t = in_place ? out : at::empty(out.sizes(), out.options().dtype(at::kFloat));
  new_lse.t = in_place ? lse : at::empty(lse.sizes(), lse.options());
  const Strides nls = stat_strides("lse", new_lse.t, out);
  const On on(out);
  call("ua_merge_update", [&] {
    return ua_merge_update(out.data_ptr(), (const float*)lse.data_ptr(), blk.data_ptr(), (const float*)blk_lse.data_ptr(), new_out.t.data_ptr(),
                           (float*)new_lse.t.data_ptr(), (int)out.size(0), (int)out.size(1), (int)out.size(2), (int)kDim, out.scalar_type() == at::kFloat,
                           blk.scalar_type() == at::kFloat, new_out.t.scalar_type() == at::kFloat, Strides(out), ls, Strides(blk), bls,
                           Strides(new_out.t), nls, on.stream);
  });
  return tuple_of(new_out, new_lse);
}

// permute_cols(src, out, n_chunks, batch, inner, gather) -> out
PyObject* permute_cols(PyObject* const* a) {
  const at::Tensor& src = tensor(a[0], "the column buffer");
  const int64_t y = integer(a[2]), b = integer(a[3]), inner = integer(a[4]), n = 2 * y * b * inner;
  const bool gather = truth(a[5]);
  if (src.dim() != 1 || src.scalar_type() != at::kBFloat16 || !src.is_cuda() || src.numel() < n)
    fail(PyExc_ValueError, "the column buffer must be a flat bfloat16 CUDA tensor of at least " + std::to_string(n) + " elements");
  Slot out(a[1]);
  out.t = out.given ? tensor(out.given, "out") : at::empty({n}, src.options());
  if (out.t.dim() != 1 || out.t.scalar_type() != at::kBFloat16 || out.t.device() != src.device() || out.t.numel() < n)
    fail(PyExc_ValueError, "out must be a flat bfloat16 tensor of at least " + std::to_string(n) + " elements on the source's device");
  const On on(src);
  call(gather ? "ua_cols_gather" : "ua_cols_scatter", [&] {
    return gather ? ua_cols_gather(src.data_ptr(), out.t.data_ptr(), (int)y, (int)b, inner, on.stream)
                  : ua_cols_scatter(src.data_ptr(), out.t.data_ptr(), (int)y, (int)b, inner, on.stream);
  });
  return out.wrap();
}

// ---- module ---------------------------------------------------------------------------------------------
template <PyObject* (*F)(PyObject* const*), int N>
PyObject* entry(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != N) return PyErr_Format(PyExc_TypeError, "expected %d arguments, got %zd", N, n);
  try {
    return F(args);
  } catch (const PyError&) {
    return nullptr;
  } catch (const c10::OutOfMemoryError& e) {
    PyObject* torch = PyImport_ImportModule("torch");
    PyObject* type = torch ? PyObject_GetAttrString(torch, "OutOfMemoryError") : nullptr;
    PyErr_SetString(type ? type : PyExc_MemoryError, e.what_without_backtrace());
    Py_XDECREF(type);
    Py_XDECREF(torch);
    return nullptr;
  } catch (const std::exception& e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
    return nullptr;
  }
}
#define UA_METHOD(NAME, N) {#NAME, (PyCFunction)(void (*)(void))entry<NAME, N>, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    UA_METHOD(dense_forward, 8), UA_METHOD(dense_backward, 14), UA_METHOD(bsa_forward, 10), UA_METHOD(bsa_backward, 15),
    UA_METHOD(delta, 3), UA_METHOD(grad_accumulate, 4), UA_METHOD(merge, 4), UA_METHOD(grad_sum, 3),
    UA_METHOD(merge_update, 5), UA_METHOD(permute_cols, 6), UA_METHOD(lists_from_mask, 5),
    UA_METHOD(build_lists_device, 3), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_native", "Native host side of the attention operators.", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native() { return PyModule_Create(&module_def); }
