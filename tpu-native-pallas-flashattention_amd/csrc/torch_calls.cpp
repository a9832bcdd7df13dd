// Host side of the public calls for the plain case, in C++.
//
// A decode of one conversation keeps the GPU busy for about 10 us; checking
// its arguments, allocating and filling the C-ABI blocks through ctypes took
// the Python path 23 us, and a small training step 110-150 us of Python around
// 30-100 us of kernels. The functions here do the same from C++.
//
// Every function takes the plain case only -- exact torch.Tensor arguments on
// one GPU, one supported dtype, a kernel head_dim, whole shapes, plain numbers,
// no tracing, transform or dispatch mode -- and returns None for anything
// else, without side effects: the Python function then runs its general path,
// which validates, converts or raises. So nothing is accepted or refused here
// that is not there.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/version.h>

#include <array>
#include <climits>
#include <cmath>
#include <cstring>
#include <exception>
#include <initializer_list>

#include "../../include/pallas_flash_amd.h"

namespace {

using at::Tensor;

// A tensor subclass, functorch or FakeTensor wrapper, lazy conjugate or
// negative, ... : anything whose memory is not simply its values.
constexpr c10::DispatchKeySet kNotPlain({
    c10::DispatchKey::Python,
    c10::DispatchKey::PythonTLSSnapshot,
    c10::DispatchKey::FuncTorchGradWrapper,
    c10::DispatchKey::FuncTorchBatched,
    c10::DispatchKey::BatchedNestedTensor,
    c10::DispatchKey::Batched,
    c10::DispatchKey::Functionalize,
    c10::DispatchKey::Conjugate,
    c10::DispatchKey::Negative,
    c10::DispatchKey::ZeroTensor,
});

// Whether this thread runs plain eager code: no tracer, function or dispatch
// mode, functorch transform or Python dispatcher would see the calls the
// general path makes.
bool plain_thread() {
  const auto inc = c10::impl::tls_local_dispatch_key_set().included_;
  return !torch::jit::tracer::isTracing() && !at::impl::torch_function_mode_enabled() &&
         !c10::impl::TorchDispatchModeTLS::any_modes_set() &&
         !inc.has_any(c10::DispatchKeySet({c10::DispatchKey::FuncTorchDynamicLayerFrontMode,
                                           c10::DispatchKey::FuncTorchDynamicLayerBackMode,
                                           c10::DispatchKey::FuncTorchVmapMode, c10::DispatchKey::VmapMode,
                                           c10::DispatchKey::Functionalize, c10::DispatchKey::PythonDispatcher}));
}

// The tensor of a plain CUDA (HIP) tensor object, or null.
const Tensor* plain_tensor(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || t.key_set().has_any(kNotPlain)) return nullptr;
  return &t;
}

// dtype tag of the C ABI, or -1.
int dtype_tag(const Tensor& t) {
  switch (t.scalar_type()) {
    case at::kFloat: return PF_DTYPE_F32;
    case at::kBFloat16: return PF_DTYPE_BF16;
    case at::kHalf: return PF_DTYPE_F16;
    default: return -1;
  }
}

bool same_kind(const Tensor& a, std::initializer_list<const Tensor*> rest) {
  for (const Tensor* t : rest)
    if (t->scalar_type() != a.scalar_type() || t->device() != a.device()) return false;
  return true;
}

bool fits_i32(const Tensor& t) {
  for (const int64_t s : t.sizes())
    if (s > INT_MAX || s < 1) return false;  // empty tensors take the general path
  return true;
}

// Forward-mode AD: the general path's autograd function refuses dual tensors.
bool has_tangent(std::initializer_list<const Tensor*> ts) {
  for (const Tensor* t : ts)
    if (t->_fw_grad(/*level=*/0).defined()) return true;
  return false;
}

bool wants_grad(std::initializer_list<const Tensor*> ts) {
  if (!at::GradMode::is_enabled()) return false;
  for (const Tensor* t : ts)
    if (t->requires_grad()) return true;
  return false;
}

// None, a float or an int -> *scale (default: 1 / sqrt(head_dim)).
bool get_scale(PyObject* o, int64_t head_dim, float* scale) {
  double s;
  if (o == Py_None) {
    s = 1.0 / std::sqrt((double)head_dim);
  } else if (PyFloat_CheckExact(o)) {
    s = PyFloat_AS_DOUBLE(o);
  } else {
    return false;
  }
  *scale = (float)s;
  return std::isfinite(*scale);
}

bool get_bool(PyObject* o, bool* v) {
  if (o != Py_True && o != Py_False) return false;
  *v = o == Py_True;
  return true;
}

// An int in [1, most].
bool get_len(PyObject* o, int64_t most, int32_t* v) {
  if (!PyLong_CheckExact(o)) return false;
  int overflow = 0;
  const long long x = PyLong_AsLongLongAndOverflow(o, &overflow);
  if (overflow != 0 || x < 1 || x > most) return false;
  *v = (int32_t)x;
  return true;
}

bool kernel_head_dim(int64_t d, int tag) { return d == 64 || d == 128 || (d == 256 && tag != PF_DTYPE_F32); }
bool decode_head_dim(int64_t d, int tag) {
  return d >= 1 && d <= (tag == PF_DTYPE_F32 ? 128 : 256) && d * (tag == PF_DTYPE_F32 ? 4 : 2) % 16 == 0;
}

void* stream_of(const Tensor& t) {
  return at::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream();
}

Tensor bytes(size_t n, const Tensor& like) {
  return at::empty({(int64_t)n}, at::TensorOptions().dtype(at::kByte).device(like.device()));
}

// Thrown where the library refuses a call that passed the checks here (sizes
// past its 32-bit ranges): the general path reports it.
struct Declined {};

// Runs f without the GIL and wraps its tensor; None where it declines.
template <typename F>
PyObject* guarded(F&& f) {
  HANDLE_TH_ERRORS
  Tensor out;
  bool declined = false;
  {
    pybind11::gil_scoped_release no_gil;
    try {
      out = f();
    } catch (const Declined&) {
      declined = true;
    }
  }
  if (declined) Py_RETURN_NONE;
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

void accept(int status) {
  if (status != PF_OK) throw Declined();
}

struct Attn {
  float scale;
  int32_t kv_len;
  bool causal;
};

// q, k, v plain, contiguous and checked. The output, and the LSE where wanted.
Tensor attn_forward(const Tensor& q, const Tensor& k, const Tensor& v, const Attn& a, Tensor* lse) {
  const c10::DeviceGuard guard(q.device());
  Tensor o = at::empty(q.sizes(), q.options());
  if (lse != nullptr) *lse = at::empty({q.size(0), q.size(1), q.size(2)}, q.options().dtype(at::kFloat));
  const pf_attn_fwd_args args{q.data_ptr(),
                              k.data_ptr(),
                              v.data_ptr(),
                              o.data_ptr(),
                              lse != nullptr ? lse->data_ptr<float>() : nullptr,
                              (int32_t)q.size(0),
                              (int32_t)q.size(1),
                              (int32_t)k.size(1),
                              (int32_t)q.size(2),
                              (int32_t)k.size(2),
                              (int32_t)q.size(3),
                              a.kv_len,
                              a.causal ? 1 : 0,
                              a.scale,
                              dtype_tag(q)};
  const size_t n = pf_attn_fwd_workspace_size(&args);
  const Tensor ws = n > 0 ? bytes(n, q) : Tensor();
  accept(pf_attn_fwd_ws(&args, n > 0 ? ws.data_ptr() : nullptr, n, stream_of(q)));
  return o;
}

// Counterpart of `_flash_attention_vjp` (flash_attention.py:448-476): saves
// (q, k, v, out, lse); the backward recomputes P from the LSE.
struct FlashAttentionFn : torch::autograd::Function<FlashAttentionFn> {
  static Tensor forward(torch::autograd::AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v,
                        double scale, int64_t kv_len, bool causal) {
    Tensor lse;
    Tensor o = attn_forward(q, k, v, Attn{(float)scale, (int32_t)kv_len, causal}, &lse);
    ctx->save_for_backward({q, k, v, o, lse});
    ctx->saved_data["scale"] = scale;
    ctx->saved_data["kv_len"] = kv_len;
    ctx->saved_data["causal"] = causal;
    return o;
  }

  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                 torch::autograd::variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &q = saved[0], &k = saved[1], &v = saved[2], &o = saved[3], &lse = saved[4];
    const c10::DeviceGuard guard(q.device());
    const Tensor dout = grads[0].to(q.scalar_type()).contiguous();
    Tensor dq = at::empty(q.sizes(), q.options()), dk = at::empty(k.sizes(), k.options()),
           dv = at::empty(v.sizes(), v.options());
    const Tensor delta = at::empty(lse.sizes(), lse.options());
    const pf_attn_bwd_args args{q.data_ptr(),
                                k.data_ptr(),
                                v.data_ptr(),
                                o.data_ptr(),
                                dout.data_ptr(),
                                lse.data_ptr<float>(),
                                delta.data_ptr<float>(),
                                dq.data_ptr(),
                                dk.data_ptr(),
                                dv.data_ptr(),
                                (int32_t)q.size(0),
                                (int32_t)q.size(1),
                                (int32_t)k.size(1),
                                (int32_t)q.size(2),
                                (int32_t)k.size(2),
                                (int32_t)q.size(3),
                                (int32_t)ctx->saved_data["kv_len"].toInt(),
                                ctx->saved_data["causal"].toBool() ? 1 : 0,
                                (float)ctx->saved_data["scale"].toDouble(),
                                dtype_tag(q)};
    const size_t n = pf_attn_bwd_workspace_size(&args);
    const Tensor ws = n > 0 ? bytes(n, q) : Tensor();
    const int st = pf_attn_bwd_ws(&args, n > 0 ? ws.data_ptr() : nullptr, n, stream_of(q));
    TORCH_CHECK_VALUE(st != PF_ERR_INVALID, "flash_attention backward: invalid arguments (rejected by the C ABI)");
    TORCH_CHECK_NOT_IMPLEMENTED(st != PF_ERR_UNSUPPORTED, "flash_attention backward: unsupported configuration");
    TORCH_CHECK(st == PF_OK, "flash_attention backward: HIP launch failed (status ", st, ")");
    return {dq, dk, dv, Tensor(), Tensor(), Tensor()};
  }
};

// The shared checks of the prefill calls. False: general path.
bool prefill_ok(const Tensor& q, const Tensor& k, const Tensor& v, PyObject* causal, PyObject* scale, PyObject* kv_len,
                Attn* a) {
  const int tag = dtype_tag(q);
  if (tag < 0 || !same_kind(q, {&k, &v}) || q.dim() != 4 || k.dim() != 4 || !fits_i32(q) || !fits_i32(k)) return false;
  if (k.sizes() != v.sizes() || k.size(0) != q.size(0) || k.size(3) != q.size(3)) return false;
  if (!kernel_head_dim(q.size(3), tag) || q.size(1) % k.size(1) != 0) return false;
  if (!get_bool(causal, &a->causal) || !get_scale(scale, q.size(3), &a->scale)) return false;
  if (kv_len == Py_None) a->kv_len = (int32_t)k.size(2);
  else if (!get_len(kv_len, k.size(2), &a->kv_len)) return false;
  return !has_tangent({&q, &k, &v});
}

// attention(q, k, v, causal, sm_scale, kv_len) -> o | None
PyObject* attention(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 6 || !plain_thread()) Py_RETURN_NONE;
  const Tensor *q = plain_tensor(args[0]), *k = plain_tensor(args[1]), *v = plain_tensor(args[2]);
  Attn a;
  if (!q || !k || !v || !prefill_ok(*q, *k, *v, args[3], args[4], args[5], &a)) Py_RETURN_NONE;
  return guarded([&]() -> Tensor {
    const Tensor qc = q->contiguous(), kc = k->contiguous(), vc = v->contiguous();
    if (wants_grad({q, k, v})) return FlashAttentionFn::apply(qc, kc, vc, (double)a.scale, (int64_t)a.kv_len, a.causal);
    return attn_forward(qc, kc, vc, a, nullptr);
  });
}

// A [rows, head_dim] float32 table in device memory, not differentiated.
bool table_ok(const Tensor* t, const Tensor& q, int64_t rows) {
  return t && t->scalar_type() == at::kFloat && t->device() == q.device() && t->dim() == 2 && t->size(0) == rows &&
         t->size(1) == q.size(3) && t->is_contiguous() && !wants_grad({t}) && !has_tangent({t});
}

// rope(q, k, v, q_cos, q_sin, k_cos, k_sin, causal, sm_scale, kv_len) -> o |
// None; the forward without gradients.
PyObject* rope(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 10 || !plain_thread()) Py_RETURN_NONE;
  const Tensor *q = plain_tensor(args[0]), *k = plain_tensor(args[1]), *v = plain_tensor(args[2]);
  Attn a;
  if (!q || !k || !v || !prefill_ok(*q, *k, *v, args[7], args[8], args[9], &a)) Py_RETURN_NONE;
  if (wants_grad({q, k, v})) Py_RETURN_NONE;
  const bool own_k = args[5] != Py_None && args[6] != Py_None;
  if (!own_k && k->size(2) != q->size(2)) Py_RETURN_NONE;
  const Tensor *qc = plain_tensor(args[3]), *qs = plain_tensor(args[4]);
  const Tensor *kc = own_k ? plain_tensor(args[5]) : qc, *ks = own_k ? plain_tensor(args[6]) : qs;
  if (!table_ok(qc, *q, q->size(2)) || !table_ok(qs, *q, q->size(2)) || !table_ok(kc, *q, k->size(2)) ||
      !table_ok(ks, *q, k->size(2)))
    Py_RETURN_NONE;
  return guarded([&]() -> Tensor {
    const c10::DeviceGuard guard(q->device());
    const Tensor q1 = q->contiguous(), k1 = k->contiguous(), v1 = v->contiguous();
    Tensor o = at::empty(q1.sizes(), q1.options());
    pf_attn_fwd_rope_args r{{q1.data_ptr(), k1.data_ptr(), v1.data_ptr(), o.data_ptr(), nullptr, (int32_t)q1.size(0),
                             (int32_t)q1.size(1), (int32_t)k1.size(1), (int32_t)q1.size(2), (int32_t)k1.size(2),
                             (int32_t)q1.size(3), a.kv_len, a.causal ? 1 : 0, a.scale, dtype_tag(q1)},
                            qc->data_ptr<float>(),
                            qs->data_ptr<float>(),
                            kc->data_ptr<float>(),
                            ks->data_ptr<float>(),
                            nullptr,
                            0};
    r.workspace_bytes = pf_attn_fwd_rope_workspace_size(&r);
    if (r.workspace_bytes == 0) throw Declined();
    const Tensor ws = bytes(r.workspace_bytes, q1);
    r.workspace = ws.data_ptr();
    accept(pf_attn_fwd_rope(&r, stream_of(q1)));
    return o;
  });
}

// The checks of a one-row query [B, Hq, 1, D] against `kv` with Hkv heads in
// dimension 1 and the same head_dim.
bool query_ok(const Tensor& q, const Tensor& k, const Tensor& v) {
  const int tag = dtype_tag(q);
  return tag >= 0 && same_kind(q, {&k, &v}) && q.dim() == 4 && k.dim() == 4 && fits_i32(q) && fits_i32(k) &&
         q.size(2) == 1 && k.sizes() == v.sizes() && k.size(3) == q.size(3) && q.size(1) % k.size(1) == 0 &&
         decode_head_dim(q.size(3), tag) && !has_tangent({&q, &k, &v});
}

// decode(q, k_cache, v_cache, cache_len, sm_scale) -> o | None
PyObject* decode(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 5 || !plain_thread()) Py_RETURN_NONE;
  const Tensor *q = plain_tensor(args[0]), *k = plain_tensor(args[1]), *v = plain_tensor(args[2]);
  int32_t len;
  float scale;
  if (!q || !k || !v || wants_grad({q, k, v}) || !query_ok(*q, *k, *v) || k->size(0) != q->size(0) ||
      !get_len(args[3], k->size(2), &len) || !get_scale(args[4], q->size(3), &scale))
    Py_RETURN_NONE;
  return guarded([&]() -> Tensor {
    const c10::DeviceGuard guard(q->device());
    const Tensor q1 = q->contiguous(), k1 = k->contiguous(), v1 = v->contiguous();
    Tensor o = at::empty(q1.sizes(), q1.options());
    pf_attn_decode_args a{q1.data_ptr(), k1.data_ptr(), v1.data_ptr(), o.data_ptr(), (int32_t)q1.size(0),
                          (int32_t)q1.size(1), (int32_t)k1.size(1), (int32_t)k1.size(2), (int32_t)q1.size(3), len,
                          scale, dtype_tag(q1), nullptr, 0};
    a.workspace_bytes = pf_attn_decode_workspace_min(&a);
    if (a.workspace_bytes == 0) throw Declined();
    const Tensor ws = bytes(a.workspace_bytes, q1);
    a.workspace = ws.data_ptr();
    accept(pf_attn_decode(&a, stream_of(q1)));
    return o;
  });
}

// An int32 tensor in q's device memory, contiguous.
bool ints_ok(const Tensor* t, const Tensor& q) {
  return t && t->scalar_type() == at::kInt && t->device() == q.device() && t->is_contiguous();
}

// paged(q, k_pages, v_pages, block_tables, context_lens, sm_scale) -> o | None
PyObject* paged(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 6 || !plain_thread()) Py_RETURN_NONE;
  const Tensor *q = plain_tensor(args[0]), *k = plain_tensor(args[1]), *v = plain_tensor(args[2]);
  const Tensor *tab = plain_tensor(args[3]), *lens = plain_tensor(args[4]);
  float scale;
  if (!q || !k || !v || !query_ok(*q, *k, *v) || !k->is_contiguous() || !v->is_contiguous() || !ints_ok(tab, *q) ||
      !ints_ok(lens, *q) || tab->dim() != 2 || tab->size(0) != q->size(0) || !fits_i32(*tab) || lens->dim() != 1 ||
      lens->size(0) != q->size(0) || !get_scale(args[5], q->size(3), &scale))
    Py_RETURN_NONE;
  return guarded([&]() -> Tensor {
    const c10::DeviceGuard guard(q->device());
    const Tensor q1 = q->detach().contiguous();
    Tensor o = at::empty(q1.sizes(), q1.options());
    pf_paged_attn_args a{q1.data_ptr(), k->data_ptr(), v->data_ptr(), tab->data_ptr<int32_t>(),
                         lens->data_ptr<int32_t>(), o.data_ptr(), (int32_t)q1.size(0), (int32_t)q1.size(1),
                         (int32_t)k->size(1), (int32_t)k->size(0), (int32_t)k->size(2), (int32_t)q1.size(3),
                         (int32_t)tab->size(1), scale, dtype_tag(q1), nullptr, 0};
    a.workspace_bytes = pf_paged_attn_workspace_min(&a);
    if (a.workspace_bytes == 0) throw Declined();
    const Tensor ws = bytes(a.workspace_bytes, q1);
    a.workspace = ws.data_ptr();
    accept(pf_paged_attn(&a, stream_of(q1)));
    return o;
  });
}

bool aligned16(const Tensor& t) { return ((uintptr_t)t.data_ptr() & 15) == 0; }

// step(q, k_new, v_new, k_cache, v_cache, positions, cos, sin, ring, sm_scale)
// -> o | None (the caches are written in place)
PyObject* step(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 10 || !plain_thread()) Py_RETURN_NONE;
  const Tensor *q = plain_tensor(args[0]), *kn = plain_tensor(args[1]), *vn = plain_tensor(args[2]);
  const Tensor *kc = plain_tensor(args[3]), *vc = plain_tensor(args[4]), *pos = plain_tensor(args[5]);
  const bool rot = args[6] != Py_None || args[7] != Py_None;
  const Tensor *cos = rot ? plain_tensor(args[6]) : nullptr, *sin = rot ? plain_tensor(args[7]) : nullptr;
  float scale;
  bool ring;
  if (!q || !kn || !vn || !kc || !vc || !query_ok(*q, *kc, *vc) || !same_kind(*q, {kn, vn}) || kn->dim() != 4 ||
      kn->sizes() != vn->sizes() || kc->size(0) != q->size(0) || kn->size(0) != q->size(0) ||
      kn->size(1) != kc->size(1) || kn->size(2) != 1 || kn->size(3) != q->size(3) || !kc->is_contiguous() ||
      !vc->is_contiguous() || !ints_ok(pos, *q) || pos->dim() > 1 ||
      (pos->numel() != 1 && pos->numel() != q->size(0)) || has_tangent({kn, vn}) || !aligned16(*kc) ||
      !aligned16(*vc) || !aligned16(*q) || !get_bool(args[8], &ring) ||
      !get_scale(args[9], q->size(3), &scale))
    Py_RETURN_NONE;
  if (rot && (!cos || !sin || cos->dim() != 2 || !fits_i32(*cos) || !table_ok(cos, *q, cos->size(0)) ||
              !table_ok(sin, *q, cos->size(0))))
    Py_RETURN_NONE;
  return guarded([&]() -> Tensor {
    const c10::DeviceGuard guard(q->device());
    const Tensor q1 = q->detach().contiguous(), k1 = kn->detach().contiguous(), v1 = vn->detach().contiguous();
    Tensor o = at::empty(q1.sizes(), q1.options());
    pf_attn_decode_step_args a{q1.data_ptr(), k1.data_ptr(), v1.data_ptr(), kc->data_ptr(), vc->data_ptr(),
                               o.data_ptr(), pos->data_ptr<int32_t>(), pos->numel() == 1 ? 0 : 1,
                               rot ? cos->data_ptr<float>() : nullptr, rot ? sin->data_ptr<float>() : nullptr,
                               rot ? (int32_t)cos->size(0) : 0, (int32_t)q1.size(0), (int32_t)q1.size(1),
                               (int32_t)kc->size(1), (int32_t)kc->size(2), (int32_t)q1.size(3), ring ? 1 : 0, scale,
                               dtype_tag(q1), nullptr, 0};
    a.workspace_bytes = pf_attn_decode_step_workspace_size(&a);
    if (a.workspace_bytes == 0) throw Declined();
    const Tensor ws = bytes(a.workspace_bytes, q1);
    a.workspace = ws.data_ptr();
    accept(pf_attn_decode_step(&a, stream_of(q1)));
    return o;
  });
}

#define PF_CALL(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {PF_CALL(attention), PF_CALL(rope), PF_CALL(decode), PF_CALL(paged), PF_CALL(step),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_torch_calls", nullptr, -1, methods};

}  // namespace

// Built against one torch release's C++ interfaces: refuses to be imported under
// another one, whose layouts may differ even where every symbol is found.
PyMODINIT_FUNC PyInit__torch_calls() {
  PyObject* torch = PyImport_ImportModule("torch");
  if (torch == nullptr) return nullptr;
  PyObject* version = PyObject_GetAttrString(torch, "__version__");
  Py_DECREF(torch);
  const char* v = version != nullptr ? PyUnicode_AsUTF8(version) : nullptr;
  const size_t n = sizeof(TORCH_VERSION) - 1;
  const bool same = v != nullptr && std::strncmp(v, TORCH_VERSION, n) == 0 && (v[n] == 0 || v[n] == '+');
  if (!same && !PyErr_Occurred()) PyErr_Format(PyExc_ImportError, "built for torch %s, not %s", TORCH_VERSION, v);
  Py_XDECREF(version);
  return same ? PyModule_Create(&module) : nullptr;
}
