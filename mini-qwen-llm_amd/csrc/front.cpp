// CPython extension `mqk._front`: the Python entry points' checks, output
// allocations and native call in C++, for ordinary calls.
//
// A decode-size kernel takes 5-16 us, and the Python of one call (a dozen tensors
// checked attribute by attribute, three torch.empty, two ctypes calls) took 11-30 us,
// so those calls ran at the host's pace.  Measured per call, host only: mqk.fused_qkv_rope
// 13.7 -> 7.7 us, fused_qkv_rope_ex with the input norm and the paged write 19.1 -> 10.0 us,
// its W4A16 twin 29.9 -> 8.9 us, a LinearW4A16 11.3 -> 6.0 us (what is left is mostly the
// launches themselves).
//
// Every function returns a result only if the call is an ordinary one: plain dense
// tensors on the current device with the expected types and shapes, contiguous and
// 16-byte aligned, no tensor subclass, functorch wrapper or torch mode, and a
// workspace that is there and large enough.  Anything else -- an error to raise, a
// tensor to copy or convert, another device, a workspace to make -- returns None, and
// the Python code beside it, which remains the definition of the entry point, takes
// the call.  A native failure returns the status for Python to raise.
//
// The GIL is released where a call can wait for the driver: the output allocations and
// the launches (a full queue, or one whose host function needs the GIL).  Every pointer
// is read from its tensor before; 0.1 us of a call.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/ops/empty.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/core/impl/VirtualGuardImpl.h>

#include <dlfcn.h>

#include "../../include/mqk.h"

namespace {

// Entry points of the loaded libmqk.so (bind()).
struct Lib {
  decltype(&mqk_fused_qkv_rope_bf16) bf16 = nullptr;
  decltype(&mqk_fused_qkv_rope_f32) f32 = nullptr;
  decltype(&mqk_fused_qkv_rope_f16_ws) f16 = nullptr;
  decltype(&mqk_fused_qkv_rope_f16_workspace_size) f16_size = nullptr;
  decltype(&mqk_fused_qkv_rope_workspace_size) size = nullptr;
  decltype(&mqk_fused_qkv_rope_ex_workspace_size) ex_size = nullptr;
  decltype(&mqk_fused_qkv_rope_w4a16_workspace_size) w4_size = nullptr;
  decltype(&mqk_fused_qkv_rope_ex_bf16) ex = nullptr;
  decltype(&mqk_fused_qkv_rope_ex_w4a16) ex_w4 = nullptr;
  decltype(&mqk_w4a16_gemm_workspace_size) gemm_size = nullptr;
  decltype(&mqk_w4a16_gemm_ex) gemm = nullptr;
} g_lib;

PyObject* g_workspaces = nullptr;  // mqk._native._workspaces: {(device index, stream): uint8 tensor}
PyObject* g_raw_stream = nullptr;  // torch's raw current-stream accessor
PyObject* g_parameter = nullptr;   // torch.nn.Parameter
PyObject* g_capturing = nullptr;   // mqk._native.capturing: is the current stream being captured?
bool g_bound = false;

constexpr float kEps = 1e-6f;  // the op's fixed QK-Norm epsilon

// A tensor argument of an ordinary call: exactly torch.Tensor or Parameter, dense
// strided on the GPU, and no key but the ones a plain (or autograd) tensor carries.
const at::Tensor* plain(PyObject* o) {
  PyTypeObject* t = Py_TYPE(o);
  if (reinterpret_cast<PyObject*>(t) != THPVariableClass && reinterpret_cast<PyObject*>(t) != g_parameter) return nullptr;
  const at::Tensor& v = THPVariable_Unpack(o);
  static const c10::DispatchKeySet allowed =
      c10::DispatchKeySet({c10::DispatchKey::CUDA, c10::DispatchKey::AutogradCUDA, c10::DispatchKey::ADInplaceOrView,
                            c10::DispatchKey::AutocastCUDA});
  if (!v.defined() || v.layout() != c10::kStrided || !v.is_cuda() || !allowed.has_all(v.key_set()))
    return nullptr;
  return &v;
}

struct Call {
  c10::DeviceIndex dev = -1;
  bool ok = true;

  // An operand read through 16-byte loads: on the call's device, of type `type`,
  // contiguous and aligned.
  const at::Tensor* operand(PyObject* o, at::ScalarType type) {
    const at::Tensor* t = ok ? plain(o) : nullptr;
    if (!t || t->scalar_type() != type || !t->is_contiguous() || (reinterpret_cast<uintptr_t>(t->data_ptr()) & 15u) != 0 ||
        (dev >= 0 && t->get_device() != dev)) {
      ok = false;
      return nullptr;
    }
    dev = t->get_device();
    return t;
  }
  // ... or None (null); int32 tensors of n entries
  const int32_t* ints(PyObject* o, int64_t n) {
    if (o == Py_None) return nullptr;
    const at::Tensor* t = operand(o, at::kInt);
    if (ok && t->numel() != n) ok = false;
    return ok ? t->data_ptr<int32_t>() : nullptr;
  }
};

// Without the GIL while it lives.  Nothing in its scope touches a Python object.
class Unlocked {
 public:
  Unlocked() : state_(PyEval_SaveThread()) {}
  ~Unlocked() { PyEval_RestoreThread(state_); }
  Unlocked(const Unlocked&) = delete;
  Unlocked& operator=(const Unlocked&) = delete;

 private:
  PyThreadState* state_;
};

template <class T>
const T* ptr(const at::Tensor* t) {
  return static_cast<const T*>(t->data_ptr());
}

bool current_device_is(c10::DeviceIndex dev) {
  static const c10::impl::VirtualGuardImpl guard(c10::DeviceType::CUDA);
  return guard.getDevice().index() == dev;
}

bool modes_off() {
  return !at::impl::torch_function_mode_enabled() && !c10::impl::TorchDispatchModeTLS::any_modes_set();
}

// The raw current stream of device dev, as a Python int (new reference).
PyObject* stream_of(c10::DeviceIndex dev) {
  PyObject* index = PyLong_FromLong(dev);
  if (!index) return nullptr;
  PyObject* s = PyObject_CallOneArg(g_raw_stream, index);
  Py_DECREF(index);
  return s;
}

// The workspace of (dev, stream) if it holds n bytes; none needed for n == 0.  False:
// absent or too small (Python makes or grows it).
struct Workspace {
  at::Tensor buf;  // (held: another thread may replace it while the GIL is released)
  void* ptr = nullptr;
  size_t bytes = 0;
};
bool workspace(c10::DeviceIndex dev, PyObject* stream, size_t n, Workspace* ws) {
  if (n == 0) return true;
  PyObject* key = Py_BuildValue("(iO)", int(dev), stream);
  if (!key) {
    PyErr_Clear();
    return false;
  }
  PyObject* buf = PyDict_GetItem(g_workspaces, key);  // (borrowed)
  Py_DECREF(key);
  if (!buf || !THPVariable_Check(buf)) return false;
  const at::Tensor& t = THPVariable_Unpack(buf);
  if (size_t(t.numel()) < n) return false;
  ws->buf = t;
  ws->ptr = t.data_ptr();
  ws->bytes = size_t(t.numel());
  return true;
}

// Whether the current stream is being captured (also when that cannot be told).
bool capturing() {
  PyObject* r = PyObject_CallNoArgs(g_capturing);
  if (!r) {
    PyErr_Clear();
    return true;
  }
  const bool yes = r != Py_False;
  Py_DECREF(r);
  return yes;
}

// head_dim 64 and 128 (128-column blocks of whole heads) are taken here; other sizes in Python.
bool blocks_of(int64_t D, int64_t hq, int64_t hkv, int* bq, int* bkv) {
  if (D != 128 && D != 64) return false;
  if (hq < 1 || hkv < 1 || hq > 1 << 20 || hkv > 1 << 20) return false;
  *bq = int(hq * D / 128);
  *bkv = int(hkv * D / 128);
  return true;
}

PyObject* none() { Py_RETURN_NONE; }

at::Tensor fresh(at::IntArrayRef shape, at::ScalarType type, c10::DeviceIndex dev) {
  return at::empty(shape, at::TensorOptions().dtype(type).device(c10::Device(c10::DeviceType::CUDA, dev)));
}

PyObject* wrap3(at::Tensor q, at::Tensor k, at::Tensor v) {
  PyObject* out = PyTuple_New(3);
  if (!out) return nullptr;
  at::Tensor* t[3] = {&q, &k, &v};
  for (int i = 0; i < 3; ++i) {
    PyObject* o;
    if (t[i]->defined()) {
      o = THPVariable_Wrap(*t[i]);
    } else {
      o = Py_None;
      Py_INCREF(o);
    }
    if (!o) {
      Py_DECREF(out);
      return nullptr;
    }
    PyTuple_SET_ITEM(out, i, o);
  }
  return out;
}

// Norm weights and RoPE tables shared by the fronts: gamma [D], cos / sin [rows, D].
struct Rope {
  const at::Tensor *gq, *gk, *cos, *sin;
  int64_t D = 0, rows = 0;
  bool read(Call& c, PyObject* const* a, at::ScalarType type) {
    gq = c.operand(a[0], type);
    gk = c.operand(a[1], type);
    cos = c.operand(a[2], type);
    sin = c.operand(a[3], type);
    if (!c.ok || gq->dim() != 1 || gk->dim() != 1 || cos->dim() != 2 || sin->dim() != 2) return false;
    D = gq->size(0);
    rows = cos->size(0);
    return gk->size(0) == D && cos->size(1) == D && sin->size(1) == D && sin->size(0) == rows && rows >= 1;
  }
};

// fused(x, w_q, w_k, w_v, q_norm_w, k_norm_w, cos, sin, positions)
PyObject* fused(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 9 || !g_bound || !modes_off()) return none();
  const at::Tensor* x0 = plain(a[0]);
  if (!x0) return none();
  const at::ScalarType type = x0->scalar_type();
  if (type != at::kBFloat16 && type != at::kHalf && type != at::kFloat) return none();
  Call c;
  const at::Tensor* x = c.operand(a[0], type);
  const at::Tensor* w[3];
  for (int i = 0; i < 3; ++i) w[i] = c.operand(a[1 + i], type);
  Rope r;
  if (!c.ok || !r.read(c, a + 4, type) || x->dim() != 3) return none();
  const int64_t B = x->size(0), S = x->size(1), H = x->size(2), T = B * S, D = r.D;
  for (int i = 0; i < 3; ++i)
    if (w[i]->dim() != 2 || w[i]->size(1) != H) return none();
  const int64_t hq = w[0]->size(0) / D, hkv = w[1]->size(0) / D;
  int bq, bkv;
  if (T == 0 || !blocks_of(D, hq, hkv, &bq, &bkv) || w[0]->size(0) != hq * D || w[1]->size(0) != hkv * D ||
      w[2]->size(0) != hkv * D)
    return none();
  const int32_t* pos = c.ints(a[8], T);
  if (!c.ok || !current_device_is(c.dev)) return none();
  PyObject* stream = stream_of(c.dev);
  if (!stream) return nullptr;
  size_t need = 0;
  if (type == at::kBFloat16) need = g_lib.size(T, bq, bkv, H);
  else if (type == at::kHalf) need = g_lib.f16_size(T, int(hq), int(hkv), H, int(D));
  if (type == at::kHalf && need > 0 && capturing()) {  // (a workspace of the graph's own: Python)
    Py_DECREF(stream);
    return none();
  }
  Workspace ws;
  const bool have = workspace(c.dev, stream, need, &ws);
  void* hs = PyLong_AsVoidPtr(stream);
  Py_DECREF(stream);
  if (!have) return none();
  const void* in[8] = {x->data_ptr(),    w[0]->data_ptr(), w[1]->data_ptr(),  w[2]->data_ptr(),
                       r.gq->data_ptr(), r.gk->data_ptr(), r.cos->data_ptr(), r.sin->data_ptr()};
  at::Tensor q, k, v;
  int st;
  {
    Unlocked unlocked;
    q = fresh({B, S, hq, D}, type, c.dev);
    k = fresh({B, S, hkv, D}, type, c.dev);
    v = fresh({B, S, hkv, D}, type, c.dev);
    if (type == at::kFloat) {
      auto p = [&](int i) { return static_cast<const float*>(in[i]); };
      st = g_lib.f32(p(0), p(1), p(2), p(3), p(4), p(5), p(6), p(7), pos, T, S, H, int(hq), int(hkv), int(D), r.rows, kEps,
                     static_cast<float*>(q.data_ptr()), static_cast<float*>(k.data_ptr()),
                     static_cast<float*>(v.data_ptr()), hs);
    } else {
      auto p = [&](int i) { return static_cast<const uint16_t*>(in[i]); };
      auto o = [](at::Tensor& t) { return static_cast<uint16_t*>(t.data_ptr()); };
      const auto fn = type == at::kHalf ? g_lib.f16 : g_lib.bf16;
      st = fn(p(0), p(1), p(2), p(3), p(4), p(5), p(6), p(7), pos, T, S, H, int(hq), int(hkv), int(D), r.rows, kEps, o(q),
              o(k), o(v), ws.ptr, ws.bytes, hs);
    }
  }
  if (st != 0) return PyLong_FromLong(st);
  return wrap3(std::move(q), std::move(k), std::move(v));
  END_HANDLE_TH_ERRORS
}

// The optional features: a = (positions, cu_seqlens, seq_pos0, input_norm_w, input_eps,
// k_cache, v_cache, block_table, kv_seq, kv_pos, return_kv).
struct Ext {
  mqk_fused_ext ext{};
  mqk_paged_kv kv{};
  const int32_t* pos = nullptr;
  bool return_kv = true;
  bool read(Call& c, PyObject* const* a, int64_t T, int64_t H, int64_t hkv, int64_t D) {
    pos = c.ints(a[0], T);
    if (a[1] != Py_None) {
      if (a[0] != Py_None) return false;
      const at::Tensor* cu = c.operand(a[1], at::kInt);
      if (!c.ok || cu->dim() != 1 || cu->numel() < 2) return false;
      ext.cu_seqlens = cu->data_ptr<int32_t>();
      ext.n_seqs = cu->numel() - 1;
      ext.seq_pos0 = c.ints(a[2], ext.n_seqs);
    } else if (a[2] != Py_None) {
      return false;
    }
    if (a[3] != Py_None) {
      const at::Tensor* g = c.operand(a[3], at::kBFloat16);
      if (!c.ok || g->dim() != 1 || g->size(0) != H || !PyFloat_CheckExact(a[4])) return false;
      ext.in_gamma = static_cast<const uint16_t*>(g->data_ptr());
      ext.in_eps = float(PyFloat_AS_DOUBLE(a[4]));
    }
    const bool cache = a[5] != Py_None;
    if (cache != (a[6] != Py_None) || cache != (a[7] != Py_None)) return false;
    if (!cache && (a[8] != Py_None || a[9] != Py_None)) return false;
    if (cache) {
      const at::Tensor* kc = c.operand(a[5], at::kBFloat16);
      const at::Tensor* vc = c.operand(a[6], at::kBFloat16);
      const at::Tensor* bt = c.operand(a[7], at::kInt);
      if (!c.ok || kc->dim() != 4 || kc->size(2) != hkv || kc->size(3) != D || vc->sizes() != kc->sizes() || bt->dim() != 2)
        return false;
      if (a[0] != Py_None && (a[8] == Py_None || a[9] == Py_None)) return false;
      kv.kv_seq = c.ints(a[8], T);
      kv.kv_pos = c.ints(a[9], T);
      kv.k_cache = static_cast<uint16_t*>(kc->data_ptr());
      kv.v_cache = static_cast<uint16_t*>(vc->data_ptr());
      kv.block_table = bt->data_ptr<int32_t>();
      kv.bt_rows = bt->size(0);
      kv.bt_cols = bt->size(1);
      kv.num_blocks = kc->size(0);
      kv.block_size = int32_t(kc->size(1));
      ext.kv = &kv;
    }
    if (!PyBool_Check(a[10])) return false;
    return_kv = a[10] == Py_True;
    return c.ok && (return_kv || cache);
  }
};

// x [B, S, hidden], or [T, hidden] with cu_seqlens: leading output dims and S.
bool lead_shape(const at::Tensor& x, bool varlen, int64_t* lead, int* n_lead, int64_t* S) {
  if (x.dim() == 3) {
    lead[0] = x.size(0);
    lead[1] = x.size(1);
    *n_lead = 2;
    *S = x.size(1);
    return true;
  }
  if (x.dim() == 2 && varlen) {
    lead[0] = x.size(0);
    *n_lead = 1;
    *S = x.size(0);
    return true;
  }
  return false;
}

// Outputs [*lead, heads, D] in bf16 (k and v undefined without return_kv).
struct Outputs {
  at::Tensor q, k, v;
  void make(const int64_t* lead, int n_lead, int64_t hq, int64_t hkv, int64_t D, bool kv, c10::DeviceIndex dev) {
    int64_t s[4] = {lead[0], lead[1], 0, 0};
    auto one = [&](int64_t h) {
      s[n_lead] = h;
      s[n_lead + 1] = D;
      return fresh(at::IntArrayRef(s, size_t(n_lead) + 2), at::kBFloat16, dev);
    };
    q = one(hq);
    if (kv) {
      k = one(hkv);
      v = one(hkv);
    }
  }
  static uint16_t* ptr(const at::Tensor& t) { return t.defined() ? static_cast<uint16_t*>(t.data_ptr()) : nullptr; }
};

// ex(x, w_q, w_k, w_v, q_norm_w, k_norm_w, cos, sin, <Ext's eleven>)
PyObject* fused_ex(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 19 || !g_bound || !modes_off()) return none();
  Call c;
  const at::Tensor* x = c.operand(a[0], at::kBFloat16);
  const at::Tensor* w[3];
  for (int i = 0; i < 3; ++i) w[i] = c.operand(a[1 + i], at::kBFloat16);
  Rope r;
  int64_t lead[2] = {0, 0}, S = 0;
  int n_lead = 0;
  if (!c.ok || !r.read(c, a + 4, at::kBFloat16) || !lead_shape(*x, a[9] != Py_None, lead, &n_lead, &S)) return none();
  const int64_t H = x->size(-1), D = r.D;
  for (int i = 0; i < 3; ++i)
    if (w[i]->dim() != 2 || w[i]->size(1) != H) return none();
  const int64_t hq = w[0]->size(0) / D, hkv = w[1]->size(0) / D, T = H > 0 ? x->numel() / H : 0;
  int bq, bkv;
  if (T == 0 || !blocks_of(D, hq, hkv, &bq, &bkv) || w[0]->size(0) != hq * D || w[1]->size(0) != hkv * D ||
      w[2]->size(0) != hkv * D)
    return none();
  Ext e;
  if (!e.read(c, a + 8, T, H, hkv, D) || !current_device_is(c.dev)) return none();
  PyObject* stream = stream_of(c.dev);
  if (!stream) return nullptr;
  Workspace ws;
  const bool have = workspace(c.dev, stream, g_lib.ex_size(T, bq, bkv, H, &e.ext), &ws);
  void* hs = PyLong_AsVoidPtr(stream);
  Py_DECREF(stream);
  if (!have) return none();
  const uint16_t* in[8] = {ptr<uint16_t>(x),    ptr<uint16_t>(w[0]), ptr<uint16_t>(w[1]),  ptr<uint16_t>(w[2]),
                           ptr<uint16_t>(r.gq), ptr<uint16_t>(r.gk), ptr<uint16_t>(r.cos), ptr<uint16_t>(r.sin)};
  Outputs o;
  int st;
  {
    Unlocked unlocked;
    o.make(lead, n_lead, hq, hkv, D, e.return_kv, c.dev);
    st = g_lib.ex(in[0], in[1], in[2], in[3], in[4], in[5], in[6], in[7], e.pos, T, S, H, int(hq), int(hkv), int(D), r.rows,
                  kEps, o.ptr(o.q), o.ptr(o.k), o.ptr(o.v), &e.ext, ws.ptr, ws.bytes, hs);
  }
  if (st != 0) return PyLong_FromLong(st);
  return wrap3(std::move(o.q), std::move(o.k), std::move(o.v));
  END_HANDLE_TH_ERRORS
}

// One projection's (qweight, scales, qzeros) for K inputs and group size g.
struct Int4 {
  const at::Tensor *qw, *sc, *qz;
  int64_t N = 0;
  int scale_type = 0;
  bool read(Call& c, PyObject* const* a, int64_t K, int64_t g) {
    qw = c.operand(a[0], at::kInt);
    qz = c.operand(a[2], at::kInt);
    if (!c.ok) return false;
    const at::Tensor* s0 = plain(a[1]);
    if (!s0 || (s0->scalar_type() != at::kBFloat16 && s0->scalar_type() != at::kHalf)) return false;
    scale_type = s0->scalar_type() == at::kHalf ? MQK_SCALE_FP16 : MQK_SCALE_BF16;
    sc = c.operand(a[1], s0->scalar_type());
    if (!c.ok || qw->dim() != 2 || sc->dim() != 2 || qz->dim() != 2) return false;
    N = qw->size(1);
    return N > 0 && N % 8 == 0 && qw->size(0) == K / 8 && sc->size(0) == K / g && sc->size(1) == N && qz->size(0) == K / g &&
           qz->size(1) == N / 8;
  }
};

bool group_of(PyObject* o, int64_t K, int64_t* g) {
  if (!PyLong_CheckExact(o)) return false;
  int overflow = 0;
  *g = PyLong_AsLongLongAndOverflow(o, &overflow);
  return !overflow && *g > 0 && *g <= 1 << 24 && K % *g == 0 && K % 8 == 0;
}

// ex_w4(x, 9 int4 tensors, q_norm_w, k_norm_w, cos, sin, <Ext's eleven>, group_size)
PyObject* fused_ex_w4(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 26 || !g_bound || !modes_off()) return none();
  Call c;
  const at::Tensor* x = c.operand(a[0], at::kBFloat16);
  int64_t lead[2] = {0, 0}, S = 0, g = 0;
  int n_lead = 0;
  if (!c.ok || !lead_shape(*x, a[15] != Py_None, lead, &n_lead, &S)) return none();
  const int64_t H = x->size(-1), T = H > 0 ? x->numel() / H : 0;
  if (T == 0 || !group_of(a[25], H, &g)) return none();
  Int4 w[3];
  for (int i = 0; i < 3; ++i)
    if (!w[i].read(c, a + 1 + 3 * i, H, g)) return none();
  if (w[1].scale_type != w[0].scale_type || w[2].scale_type != w[0].scale_type) return none();
  Rope r;
  if (!r.read(c, a + 10, at::kBFloat16)) return none();
  const int64_t D = r.D, hq = w[0].N / D, hkv = w[1].N / D;
  int bq, bkv;
  if (!blocks_of(D, hq, hkv, &bq, &bkv) || w[0].N != hq * D || w[1].N != hkv * D || w[2].N != hkv * D) return none();
  Ext e;
  if (!e.read(c, a + 14, T, H, hkv, D) || !current_device_is(c.dev)) return none();
  PyObject* stream = stream_of(c.dev);
  if (!stream) return nullptr;
  Workspace ws;
  const size_t need = g_lib.w4_size(T, bq, bkv, H, &e.ext);
  // (a captured call that unpacks its weights has a workspace of the graph's own: Python)
  const bool own = need > g_lib.ex_size(T, bq, bkv, H, &e.ext) && capturing();
  const bool have = !own && workspace(c.dev, stream, need, &ws);
  void* hs = PyLong_AsVoidPtr(stream);
  Py_DECREF(stream);
  if (!have) return none();
  const uint16_t* in[5] = {ptr<uint16_t>(x), ptr<uint16_t>(r.gq), ptr<uint16_t>(r.gk), ptr<uint16_t>(r.cos),
                           ptr<uint16_t>(r.sin)};
  const int32_t *qw[3], *qz[3];
  const void* sc[3];
  for (int i = 0; i < 3; ++i) {
    qw[i] = ptr<int32_t>(w[i].qw);
    sc[i] = w[i].sc->data_ptr();
    qz[i] = ptr<int32_t>(w[i].qz);
  }
  Outputs o;
  int st;
  {
    Unlocked unlocked;
    o.make(lead, n_lead, hq, hkv, D, e.return_kv, c.dev);
    st = g_lib.ex_w4(in[0], qw[0], sc[0], qz[0], qw[1], sc[1], qz[1], qw[2], sc[2], qz[2], int(g), w[0].scale_type, in[1],
                     in[2], in[3], in[4], e.pos, T, S, H, int(hq), int(hkv), int(D), r.rows, kEps, o.ptr(o.q), o.ptr(o.k),
                     o.ptr(o.v), &e.ext, ws.ptr, ws.bytes, hs);
  }
  if (st != 0) return PyLong_FromLong(st);
  return wrap3(std::move(o.q), std::move(o.k), std::move(o.v));
  END_HANDLE_TH_ERRORS
}

// gemm(x [M, K], qweight, scales, qzeros, group_size)
PyObject* gemm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 5 || !g_bound || !modes_off()) return none();
  Call c;
  const at::Tensor* x = c.operand(a[0], at::kBFloat16);
  int64_t g = 0;
  if (!c.ok || x->dim() != 2) return none();
  const int64_t M = x->size(0), K = x->size(1);
  Int4 w;
  if (M == 0 || !group_of(a[4], K, &g) || !w.read(c, a + 1, K, g) || !current_device_is(c.dev)) return none();
  PyObject* stream = stream_of(c.dev);
  if (!stream) return nullptr;
  Workspace ws;
  const bool have = workspace(c.dev, stream, g_lib.gemm_size(M, K, w.N), &ws);
  void* hs = PyLong_AsVoidPtr(stream);
  Py_DECREF(stream);
  if (!have) return none();
  const uint16_t* xp = ptr<uint16_t>(x);
  const int32_t *qw = ptr<int32_t>(w.qw), *qz = ptr<int32_t>(w.qz);
  const void* sc = w.sc->data_ptr();
  at::Tensor out;
  int st;
  {
    Unlocked unlocked;
    out = fresh({M, w.N}, at::kBFloat16, c.dev);
    st = g_lib.gemm(xp, qw, sc, qz, M, K, w.N, int(g), w.scale_type, static_cast<uint16_t*>(out.data_ptr()), ws.ptr,
                    ws.bytes, hs);
  }
  if (st != 0) return PyLong_FromLong(st);
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// bind(dlopen handle of libmqk.so, workspaces dict, raw-stream accessor, Parameter class,
// capture check)
PyObject* bind(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 5 || !PyDict_Check(a[1]) || !PyCallable_Check(a[2]) || !PyType_Check(a[3]) || !PyCallable_Check(a[4])) {
    PyErr_SetString(PyExc_TypeError, "bind(handle, workspaces, raw_stream, parameter_class, capturing)");
    return nullptr;
  }
  void* h = PyLong_AsVoidPtr(a[0]);
  if (!h && PyErr_Occurred()) return nullptr;
  bool all = true;
  auto get = [&](auto& fn, const char* name) {
    fn = reinterpret_cast<std::decay_t<decltype(fn)>>(dlsym(h, name));
    all = all && fn;
  };
  get(g_lib.bf16, "mqk_fused_qkv_rope_bf16");
  get(g_lib.f32, "mqk_fused_qkv_rope_f32");
  get(g_lib.f16, "mqk_fused_qkv_rope_f16_ws");
  get(g_lib.f16_size, "mqk_fused_qkv_rope_f16_workspace_size");
  get(g_lib.size, "mqk_fused_qkv_rope_workspace_size");
  get(g_lib.ex_size, "mqk_fused_qkv_rope_ex_workspace_size");
  get(g_lib.w4_size, "mqk_fused_qkv_rope_w4a16_workspace_size");
  get(g_lib.ex, "mqk_fused_qkv_rope_ex_bf16");
  get(g_lib.ex_w4, "mqk_fused_qkv_rope_ex_w4a16");
  get(g_lib.gemm_size, "mqk_w4a16_gemm_workspace_size");
  get(g_lib.gemm, "mqk_w4a16_gemm_ex");
  if (!all) {
    PyErr_SetString(PyExc_RuntimeError, "libmqk.so lacks an entry point mqk._front calls");
    return nullptr;
  }
  for (int i = 1; i < 5; ++i) Py_INCREF(a[i]);
  g_workspaces = a[1];
  g_raw_stream = a[2];
  g_parameter = a[3];
  g_capturing = a[4];
  g_bound = true;
  Py_RETURN_NONE;
}

template <class F>
PyCFunction fast(F f) {
  return reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(f));
}

PyMethodDef g_methods[] = {
    {"bind", fast(bind), METH_FASTCALL, "bind(libmqk handle, workspaces, raw stream accessor, Parameter class, capture check)"},
    {"fused", fast(fused), METH_FASTCALL, "fused_qkv_rope of an ordinary call: (q, k, v), a status, or None"},
    {"fused_ex", fast(fused_ex), METH_FASTCALL, "fused_qkv_rope_ex of an ordinary call"},
    {"fused_ex_w4", fast(fused_ex_w4), METH_FASTCALL, "fused_qkv_rope_w4a16_ex of an ordinary call"},
    {"gemm", fast(gemm), METH_FASTCALL, "w4a16_gemm of an ordinary call: the output, a status, or None"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_front", nullptr, -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__front() { return PyModule_Create(&g_module); }
