// The package's launch calls for Python: reads tensors' pointers, shapes and
// strides in C++ and calls the C ABI (include/cev_hip.h) with them.
//
// A packed pass through two decoder layers makes 28 ABI calls, one small
// attention layer two.  Through ctypes each cost 9-16 us of host time
// (tensor.stride() and data_ptr() from Python, a c_void_p per pointer, the
// argument conversion), which was most of a small pass: one question through
// two layers took 500 us with 200 us of kernels, one attention layer 22.5 us
// with 15 us of kernels.  Here the same call costs 1-2 us plus the launch.
//
// The library itself is not linked: cev_hip._abi loads it (its path can be
// chosen) and hands the entry points' addresses to bind().
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPCachingAllocator.h>
#include <c10/hip/HIPStream.h>

#include <string>

#include "../../include/cev_hip.h"

namespace {

struct Api {
  decltype(&cev_qknorm_desc_init) qknorm_desc_init;
  decltype(&cev_qknorm_rope) qknorm_rope;
  decltype(&cev_qknorm_rope_kv) qknorm_rope_kv;
  decltype(&cev_packed_attention) packed_attention;
  decltype(&cev_rms_norm) rms_norm;
  decltype(&cev_rms_norm_seq) rms_norm_seq;
  decltype(&cev_swiglu) swiglu;
  decltype(&cev_linear) linear;
  decltype(&cev_gather_rows) gather_rows;
  decltype(&cev_gdn_forward) gdn_forward;
  decltype(&cev_last_error) last_error;
} api;
PyObject* cev_error = nullptr;  // cev_hip.CevError

// A Python exception that has been set.
struct Raised {};

[[noreturn]] void raise_cev(int code, const std::string& msg) {
  PyObject* e = PyObject_CallFunction(cev_error, "is", code, msg.c_str());
  if (e) {
    PyErr_SetObject(cev_error, e);
    Py_DECREF(e);
  }
  throw Raised{};
}
[[noreturn]] void raise_py(PyObject* type, const std::string& msg) {
  PyErr_SetString(type, msg.c_str());
  throw Raised{};
}
void check(int32_t rc) {
  if (rc != CEV_OK) raise_cev(rc, api.last_error());
}

const at::Tensor& tensor(PyObject* o, const char* name) {
  if (!THPVariable_Check(o)) raise_py(PyExc_TypeError, std::string(name) + " must be a tensor");
  return THPVariable_Unpack(o);
}
const at::Tensor* tensor_or_none(PyObject* o, const char* name) { return o == Py_None ? nullptr : &tensor(o, name); }
void* ptr(const at::Tensor& t) { return t.data_ptr(); }
void* ptr(const at::Tensor* t) { return t ? t->data_ptr() : nullptr; }

int64_t as_int(PyObject* o) {
  const int64_t v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) throw Raised{};
  return v;
}
double as_double(PyObject* o) {
  const double v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) throw Raised{};
  return v;
}
bool as_bool(PyObject* o) {
  const int v = PyObject_IsTrue(o);
  if (v < 0) throw Raised{};
  return v != 0;
}

int dtype_code(const at::Tensor& t) {
  if (t.scalar_type() == at::kFloat) return CEV_F32;
  if (t.scalar_type() == at::kBFloat16) return CEV_BF16;
  raise_cev(CEV_ERR_UNSUPPORTED, std::string("dtype torch.") + c10::toString(t.scalar_type()) + " not supported (float32, bfloat16)");
}

// The stream object's handle (None there is the default stream), or the current stream's.
void* stream_of(PyObject* o) {
  if (o == Py_None) return (void*)c10::hip::getCurrentHIPStream().stream();
  PyObject* v = PyObject_GetAttrString(o, "cuda_stream");
  if (!v) throw Raised{};
  const unsigned long long h = v == Py_None ? 0 : PyLong_AsUnsignedLongLong(v);
  Py_DECREF(v);
  if (h == (unsigned long long)-1 && PyErr_Occurred()) throw Raised{};
  return (void*)(uintptr_t)h;
}

// The bytes of a ctypes structure or numpy array.
struct Bytes {
  Py_buffer b;
  Bytes(PyObject* o, bool writable) {
    if (PyObject_GetBuffer(o, &b, writable ? PyBUF_WRITABLE : PyBUF_SIMPLE) != 0) throw Raised{};
  }
  ~Bytes() { PyBuffer_Release(&b); }
  Bytes(const Bytes&) = delete;
  Bytes& operator=(const Bytes&) = delete;
};

void need_args(Py_ssize_t n, Py_ssize_t want) {
  if (n != want) raise_py(PyExc_TypeError, "expected " + std::to_string(want) + " arguments, got " + std::to_string(n));
}

// The interpreter lock let go of for its lifetime.
struct Unlocked {
  PyThreadState* state = PyEval_SaveThread();
  ~Unlocked() { PyEval_RestoreThread(state); }
};

// Runs an ABI call without the interpreter lock.  The lock is held again
// before an exception of fn's tensor accessors leaves.
template <typename Fn>
void call(Fn&& fn) {
  int32_t rc;
  {
    Unlocked unlocked;
    rc = fn();
  }
  check(rc);
}

template <typename Fn>
PyObject* guarded(Fn&& fn) {
  HANDLE_TH_ERRORS
  try {
    fn();
  } catch (const Raised&) {
    return nullptr;
  }
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

void rows_contiguous(const at::Tensor& t, const char* msg = "last dimension must be contiguous") {
  if (t.stride(-1) != 1) raise_cev(CEV_ERR_UNSUPPORTED, msg);
}

// qknorm_rope(q_in, k_in, w_q, w_k, pos, cos, sin, rotary_dim, n_pos, eps, plus_one, q_out, k_out, v_in, v_out, slots, n_slots, stream):
// cev_qknorm_rope, or cev_qknorm_rope_kv when v_in is given
PyObject* py_qknorm_rope(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&] {
    need_args(n, 18);
    const at::Tensor &q_in = tensor(a[0], "q_in"), &k_in = tensor(a[1], "k_in"), &pos = tensor(a[4], "pos"),
                     &q_out = tensor(a[11], "q_out"), &k_out = tensor(a[12], "k_out");
    // (the ABI says which of these a call may go without)
    const at::Tensor *w_q = tensor_or_none(a[2], "w_q"), *w_k = tensor_or_none(a[3], "w_k"), *cos = tensor_or_none(a[5], "cos"),
                     *sin = tensor_or_none(a[6], "sin");
    const at::Tensor *v_in = tensor_or_none(a[13], "v_in"), *v_out = tensor_or_none(a[14], "v_out"), *slots = tensor_or_none(a[15], "slots");
    if (q_in.dim() != 3) raise_py(PyExc_ValueError, "q_in must be (t, heads, head_dim)");
    cev_qknorm_desc d;
    check(api.qknorm_desc_init(&d, dtype_code(q_in), (int32_t)q_in.size(1), (int32_t)k_in.size(1), (int32_t)q_in.size(2),
                               (int32_t)q_in.size(0), (int32_t)as_int(a[7]), (int32_t)as_int(a[8]), as_bool(a[10]) ? 1 : 0,
                               (float)as_double(a[9]), 0));
    for (const at::Tensor* t : {&q_in, &k_in, &q_out, &k_out}) rows_contiguous(*t);
    if (v_in) {
      if (!v_out) raise_py(PyExc_TypeError, "v_out must be a tensor");
      rows_contiguous(*v_in);
      rows_contiguous(*v_out);
    }
    d.qi_stride_t = q_in.stride(0), d.qi_stride_h = q_in.stride(1);
    d.ki_stride_t = k_in.stride(0), d.ki_stride_h = k_in.stride(1);
    d.qo_stride_t = q_out.stride(0), d.qo_stride_h = q_out.stride(1);
    d.ko_stride_t = k_out.stride(0), d.ko_stride_h = k_out.stride(1);
    if (pos.scalar_type() != at::kInt || (slots && slots->scalar_type() != at::kInt))
      raise_cev(CEV_ERR_INVALID, v_in ? "positions and slots must be int32" : "positions must be int32");
    void* const s = stream_of(a[17]);
    if (!v_in) {
      call([&] { return api.qknorm_rope(&d, ptr(q_in), ptr(k_in), ptr(w_q), ptr(w_k), (const int32_t*)ptr(pos), ptr(cos), ptr(sin), ptr(q_out), ptr(k_out), s); });
      return;
    }
    const int32_t n_slots = (int32_t)as_int(a[16]);
    call([&] {
      return api.qknorm_rope_kv(&d, ptr(q_in), ptr(k_in), ptr(v_in), v_in->stride(0), v_in->stride(1), ptr(w_q), ptr(w_k),
                                (const int32_t*)ptr(pos), ptr(cos), ptr(sin), (const int32_t*)ptr(slots), n_slots, ptr(q_out), ptr(k_out),
                                ptr(v_out), v_out->stride(0), v_out->stride(1), s);
    });
  });
}

// attention(desc, plan_host, plan_dev, q, k_new, v_new, k_cache, v_cache, gate, out, workspace, workspace_bytes, stream): takes the
// tensors' strides into desc, then cev_packed_attention
PyObject* py_attention(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&] {
    need_args(n, 13);
    const at::Tensor &q = tensor(a[3], "q"), &kn = tensor(a[4], "k_new"), &vn = tensor(a[5], "v_new"), &out = tensor(a[9], "out");
    const at::Tensor *dev = tensor_or_none(a[2], "plan"), *kc = tensor_or_none(a[6], "k_cache"), *vc = tensor_or_none(a[7], "v_cache"),
                     *gate = tensor_or_none(a[8], "gate"), *ws = tensor_or_none(a[10], "workspace");
    for (const at::Tensor* t : {&q, &kn, &vn, kc, vc, &out, gate})
      if (t) rows_contiguous(*t);
    Bytes desc(a[0], true), host(a[1], false);
    if (desc.b.len != (Py_ssize_t)sizeof(cev_attn_desc)) raise_py(PyExc_TypeError, "desc must be an AttnDesc");
    cev_attn_desc* d = (cev_attn_desc*)desc.b.buf;
    d->q_stride_t = q.stride(0), d->q_stride_h = q.stride(1);
    d->kn_stride_t = kn.stride(0), d->kn_stride_h = kn.stride(1);
    d->vn_stride_t = vn.stride(0), d->vn_stride_h = vn.stride(1);
    if (kc) {
      if (!vc) raise_py(PyExc_TypeError, "v_cache must be a tensor");
      d->kc_stride_h = kc->stride(0), d->kc_stride_s = kc->stride(1);
      d->vc_stride_h = vc->stride(0), d->vc_stride_s = vc->stride(1);
    }
    d->o_stride_t = out.stride(0), d->o_stride_h = out.stride(1);
    if (gate) d->g_stride_t = gate->stride(0), d->g_stride_h = gate->stride(1);
    const size_t ws_bytes = (size_t)as_int(a[11]);
    void* const s = stream_of(a[12]);
    const cev_attn_desc mine = *d;  // another thread may set the shared one's strides while this call runs
    call([&] {
      return api.packed_attention(&mine, host.b.buf, ptr(dev), ptr(q), ptr(kc), ptr(vc), ptr(kn), ptr(vn), ptr(gate), ptr(out), ptr(ws),
                                  ws_bytes, s);
    });
  });
}

// rms_norm(x, w, eps, h, x_out, y, plus_one, stream, sequential)
PyObject* py_rms_norm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&] {
    need_args(n, 9);
    const at::Tensor &x = tensor(a[0], "x"), &w = tensor(a[1], "w"), &y = tensor(a[5], "y");
    const at::Tensor *h = tensor_or_none(a[3], "h"), *x_out = tensor_or_none(a[4], "x_out");
    if (x.dim() != 2) raise_py(PyExc_ValueError, "x must be (rows, hidden)");
    for (const at::Tensor* t : {&x, &y, &w, h, h ? x_out : nullptr})
      if (t && (t->stride(-1) != 1 || t->scalar_type() != x.scalar_type()))
        raise_cev(CEV_ERR_UNSUPPORTED, "rms_norm: tensors must share the dtype and have a contiguous last dim");
    const auto fn = as_bool(a[8]) ? api.rms_norm_seq : api.rms_norm;
    const int dt = dtype_code(x);
    const float eps = (float)as_double(a[2]);
    const int32_t plus = as_bool(a[6]) ? 1 : 0;
    void* const s = stream_of(a[7]);
    call([&] {
      return fn(dt, x.size(0), (int32_t)x.size(1), ptr(x), x.stride(0), ptr(h), h ? h->stride(0) : 0, ptr(x_out),
                x_out ? x_out->stride(0) : 0, ptr(w), eps, plus, ptr(y), y.stride(0), s);
    });
  });
}

// swiglu(gate, up, out, stream)
PyObject* py_swiglu(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&] {
    need_args(n, 4);
    const at::Tensor &g = tensor(a[0], "gate"), &u = tensor(a[1], "up"), &out = tensor(a[2], "out");
    if (g.dim() != 2) raise_py(PyExc_ValueError, "gate must be (rows, inter)");
    if (!u.sizes().equals(g.sizes()) || u.stride(0) != g.stride(0))
      raise_cev(CEV_ERR_INVALID, "swiglu: gate and up must have the same shape and row stride");
    const int dt = dtype_code(g);
    void* const s = stream_of(a[3]);
    call([&] { return api.swiglu(dt, g.size(0), (int32_t)g.size(1), ptr(g), ptr(u), g.stride(0), ptr(out), out.stride(0), s); });
  });
}

// A device buffer of one call, from torch's allocator for the call's stream:
// given back once the call is queued, so only later work of that stream gets
// the memory, and a captured call's belongs to its graph.
struct CallBuffer {
  void* p = nullptr;
  CallBuffer(const at::Tensor& on, size_t bytes, void* stream) {
    if (bytes == 0 || !on.is_cuda()) return;
    const c10::DeviceGuard guard(on.device());
    p = c10::hip::HIPCachingAllocator::raw_alloc_with_stream(bytes, (hipStream_t)stream);
  }
  ~CallBuffer() {
    if (p) c10::hip::HIPCachingAllocator::raw_delete(p);
  }
  CallBuffer(const CallBuffer&) = delete;
  CallBuffer& operator=(const CallBuffer&) = delete;
};

// linear(x, w, out, alpha, handle, workspace, workspace_bytes, stream): without a workspace one of workspace_bytes is taken for the call
PyObject* py_linear(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&] {
    need_args(n, 8);
    const at::Tensor &x = tensor(a[0], "x"), &w = tensor(a[1], "w"), &out = tensor(a[2], "out");
    const at::Tensor* ws = tensor_or_none(a[5], "workspace");
    if (x.dim() != 2) raise_py(PyExc_ValueError, "x must be (m, k)");
    const int dt = dtype_code(x);
    if (w.scalar_type() != x.scalar_type() || w.size(1) != x.size(1)) raise_cev(CEV_ERR_INVALID, "linear: w must be (n, k) in x's dtype");
    for (const at::Tensor* t : {&x, &w, &out}) rows_contiguous(*t, "linear: last dimension must be contiguous");
    const int odt = dtype_code(out);
    const float alpha = (float)as_double(a[3]);
    const cev_blas handle = a[4] == Py_None ? nullptr : (cev_blas)(uintptr_t)as_int(a[4]);
    void* const s = stream_of(a[7]);
    size_t bytes = ws ? (size_t)ws->numel() : (size_t)as_int(a[6]);
    const CallBuffer own(x, ws ? 0 : bytes, s);
    void* const buffer = ws ? ptr(ws) : own.p;
    if (!buffer) bytes = 0;
    call([&] {
      return api.linear(handle, dt, odt, x.size(0), w.size(0), x.size(1), ptr(x), x.stride(0), ptr(w), w.stride(0), alpha, ptr(out),
                        out.stride(0), buffer, bytes, s);
    });
  });
}

// gather_rows(table, ids, out, stream)
PyObject* py_gather_rows(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&] {
    need_args(n, 4);
    const at::Tensor &table = tensor(a[0], "table"), &out = tensor(a[2], "out");
    const at::Tensor* ids = tensor_or_none(a[1], "ids");
    if (table.dim() != 2) raise_py(PyExc_ValueError, "table must be (rows, width)");
    if (ids && (ids->scalar_type() != at::kInt || !ids->is_contiguous()))
      raise_cev(CEV_ERR_INVALID, "gather_rows: ids must be contiguous int32");
    const int dt = dtype_code(table), odt = dtype_code(out);
    void* const s = stream_of(a[3]);
    call([&] {
      return api.gather_rows(dt, odt, ids ? ids->size(0) : table.size(0), table.size(1), ptr(table), table.stride(0), table.size(0),
                             (const int32_t*)ptr(ids), ptr(out), out.stride(0), s);
    });
  });
}

// gdn(desc, mixed, z, b, a, conv_w, neg_a, dt_bias, norm_w, conv_in, s_in, y, conv_out, s_out, workspace, stream)
PyObject* py_gdn(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&] {
    need_args(n, 16);
    Bytes desc(a[0], true);
    if (desc.b.len != (Py_ssize_t)sizeof(cev_gdn_desc)) raise_py(PyExc_TypeError, "desc must be a GdnDesc");
    cev_gdn_desc* d = (cev_gdn_desc*)desc.b.buf;
    const at::Tensor &mixed = tensor(a[1], "mixed"), &z = tensor(a[2], "z"), &b = tensor(a[3], "b"), &av = tensor(a[4], "a"),
                     &y = tensor(a[11], "y"), &conv_out = tensor(a[12], "conv_out"), &s_out = tensor(a[13], "s_out"),
                     &ws = tensor(a[14], "workspace");
    const at::Tensor *conv_w = tensor_or_none(a[5], "conv_w"), *neg_a = tensor_or_none(a[6], "neg_a"), *dt_bias = tensor_or_none(a[7], "dt_bias"),
                     *norm_w = tensor_or_none(a[8], "norm_w"), *conv_in = tensor_or_none(a[9], "conv_in"), *s_in = tensor_or_none(a[10], "s_in");
    const auto want = d->dtype == CEV_BF16 ? at::kBFloat16 : at::kFloat;
    const char* const names[] = {"mixed", "z", "b", "a"};
    const at::Tensor* const in[] = {&mixed, &z, &b, &av};
    for (int i = 0; i < 4; ++i)
      if (in[i]->stride(-1) != 1 || in[i]->scalar_type() != want)
        raise_py(PyExc_ValueError, std::string(names[i]) + " must be torch." + (want == at::kFloat ? "float32" : "bfloat16") + " with unit channel stride");
    d->mixed_stride_b = mixed.stride(0), d->mixed_stride_t = mixed.stride(1);
    d->z_stride_b = z.stride(0), d->z_stride_t = z.stride(1);
    if (!av.strides().equals(b.strides())) raise_py(PyExc_ValueError, "a and b must share strides");
    d->ab_stride_b = av.stride(0), d->ab_stride_t = av.stride(1);
    if (conv_in) {
      if (conv_in->stride(1) != d->conv_kernel - 1 || conv_in->stride(2) != 1)
        raise_py(PyExc_ValueError, "conv_in must be (B, conv_dim, K-1) with contiguous rows");
      d->conv_in_stride_b = conv_in->stride(0);
    }
    if (s_in) {
      const int64_t dk = d->head_k_dim, dv = d->head_v_dim;
      if (s_in->scalar_type() != at::kFloat || s_in->dim() != 4 || s_in->stride(1) != dk * dv || s_in->stride(2) != dv || s_in->stride(3) != 1)
        raise_py(PyExc_ValueError, "s_in must be f32 (B, nv, dk, dv) with contiguous heads");
      d->s_in_stride_b = s_in->stride(0);
    }
    d->y_stride_b = y.stride(0), d->y_stride_t = y.stride(1);
    void* const s = stream_of(a[15]);
    const cev_gdn_desc mine = *d;
    call([&] {
      return api.gdn_forward(&mine, ptr(mixed), ptr(z), ptr(b), ptr(av), ptr(conv_w), (const float*)ptr(neg_a), (const float*)ptr(dt_bias),
                             (const float*)ptr(norm_w), ptr(conv_in), (const float*)ptr(s_in), ptr(y), ptr(conv_out), (float*)ptr(s_out),
                             ptr(ws), (size_t)ws.numel(), s);
    });
  });
}

// bind(error_class, {symbol: address})
PyObject* py_bind(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&] {
    need_args(n, 2);
    auto get = [&](const char* name, auto& fn) {
      PyObject* v = PyDict_GetItemString(a[1], name);
      if (!v) raise_py(PyExc_KeyError, name);
      const unsigned long long p = PyLong_AsUnsignedLongLong(v);
      if (p == (unsigned long long)-1 && PyErr_Occurred()) throw Raised{};
      fn = (std::remove_reference_t<decltype(fn)>)(uintptr_t)p;
    };
    get("cev_qknorm_desc_init", api.qknorm_desc_init);
    get("cev_qknorm_rope", api.qknorm_rope);
    get("cev_qknorm_rope_kv", api.qknorm_rope_kv);
    get("cev_packed_attention", api.packed_attention);
    get("cev_rms_norm", api.rms_norm);
    get("cev_rms_norm_seq", api.rms_norm_seq);
    get("cev_swiglu", api.swiglu);
    get("cev_linear", api.linear);
    get("cev_gather_rows", api.gather_rows);
    get("cev_gdn_forward", api.gdn_forward);
    get("cev_last_error", api.last_error);
    Py_INCREF(a[0]);
    cev_error = a[0];
  });
}

#define CEV_METHOD(name) {#name, (PyCFunction)(void (*)(void))py_##name, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {CEV_METHOD(bind),   CEV_METHOD(qknorm_rope), CEV_METHOD(attention),   CEV_METHOD(rms_norm), CEV_METHOD(swiglu),
                         CEV_METHOD(linear), CEV_METHOD(gather_rows), CEV_METHOD(gdn), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_cev_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__cev_calls() { return PyModule_Create(&module); }
