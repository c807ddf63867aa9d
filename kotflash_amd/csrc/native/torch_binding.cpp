// The torch side of the launch path, in C++ (module kotflash_amd._native).
//
// A call of the public attention API on small tensors is bound by its host
// work: argument checks, output and workspace allocation, the C-ABI call's
// argument marshalling and, for training, autograd's Python Function. This
// module does that work for the ordinary case and leaves every other one to
// the Python path above it: each entry returns NotImplemented, before it has
// allocated or launched anything, unless all of its conditions hold, and the
// Python path then checks, raises or runs exactly as it would alone.
//
// Measured on MI355X, us per call through the public API among other calls,
// Python path -> this one:
//   one-token append_and_attend over 2000 keys (B=2 Hq=8 Hkv=2 D=64)  28.2 -> 9.7
//   decode over 16384 keys, same heads                                17.7 -> 9.2
//   ragged append of 4 tokens to 8 sequences, then set_lengths       105.3 -> 38.0
//   causal forward, S=512, same heads                                 15.5 -> 5.8
//   training step, B=4 H=12 S=1000 D=64 causal                       139.3 -> 79.6
//   training step, B=4 H=8 Sq=300 Sk=1500 D=80                       129.1 -> 75.1
// (the two training steps with the backward kernels of that measurement; 65.9
// and 59.5 with the present forms and dK/dV plans).
// The calls are then bound by their kernels and launches (about 2.7 us of host
// time per launch in this HIP runtime).
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstring>
#include <vector>

#include "../../../include/kotflash_amd.h"

namespace {

using at::Tensor;

// ---------------------------------------------------------------------------
// Conditions of the fast path.

// gfx950 by device index: 0 unknown, 1 yes, 2 no.
std::atomic<int8_t> g_gfx950[64];

bool is_gfx950(int64_t index) {
  if (index < 0 || index >= 64) return false;
  int8_t known = g_gfx950[index].load(std::memory_order_relaxed);
  if (known == 0) {
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, (int)index) != hipSuccess) {
      (void)hipGetLastError();
      return false;
    }
    known = strncmp(prop.gcnArchName, "gfx950", 6) == 0 && (prop.gcnArchName[6] == '\0' || prop.gcnArchName[6] == ':') ? 1 : 2;
    g_gfx950[index].store(known, std::memory_order_relaxed);
  }
  return known == 1;
}

// Modes under which a call must go through torch's own Python machinery:
// function and dispatch modes, functorch transforms (vmap, grad, jvp) and
// TorchScript tracing.
bool plain_mode() {
  using c10::DispatchKey;
  return !at::impl::torch_function_mode_enabled() && !c10::impl::dispatch_mode_enabled() &&
         !c10::impl::tls_is_dispatch_key_included(DispatchKey::FuncTorchDynamicLayerFrontMode) &&
         !torch::jit::tracer::isTracing();
}

// An argument that is exactly a torch.Tensor (or Parameter) backed by plain
// GPU memory; null otherwise.
const Tensor* plain_tensor(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || !t.has_storage() || t.layout() != at::kStrided || t.is_neg() ||
      t._is_zerotensor() || t._fw_grad(0).defined())
    return nullptr;
  return &t;
}

bool half_type(const Tensor& t) {
  return t.scalar_type() == at::kHalf || t.scalar_type() == at::kBFloat16;
}

// The kernels read a tensor in place with a unit head_dim stride, other
// strides in multiples of 8 elements and a 16-byte aligned base.
bool layout_ok(const Tensor& t) {
  const auto s = t.strides();
  return s[3] == 1 && s[0] % 8 == 0 && s[1] % 8 == 0 && s[2] % 8 == 0 &&
         reinterpret_cast<uintptr_t>(t.const_data_ptr()) % 16 == 0;
}

Tensor readable(const Tensor& t) { return layout_ok(t) ? t : t.contiguous(); }

// q [B, Hq, Sq, D] with k and v [B, Hkv, Sk, D]: one 16-bit dtype, one gfx950
// device, sizes the kernels take without padding.
bool attention_args(const Tensor& q, const Tensor& k, const Tensor& v) {
  if (q.dim() != 4 || k.dim() != 4 || v.dim() != 4) return false;
  const auto qs = q.sizes(), ks = k.sizes();
  if (ks != v.sizes() || qs[0] != ks[0] || qs[3] != ks[3]) return false;
  for (int i = 0; i < 4; ++i)
    if (qs[i] <= 0 || ks[i] <= 0) return false;
  if (qs[1] % ks[1] || qs[3] % 8 || qs[3] < 8 || qs[3] > 128) return false;
  if (!half_type(q) || k.scalar_type() != q.scalar_type() || v.scalar_type() != q.scalar_type()) return false;
  const auto dev = q.device();
  return k.device() == dev && v.device() == dev && is_gfx950(dev.index());
}

bool wants_grad(std::initializer_list<const Tensor*> ts) {
  if (!at::GradMode::is_enabled()) return false;
  for (const Tensor* t : ts)
    if (t->requires_grad()) return true;
  return false;
}

// ---------------------------------------------------------------------------
// Launches. `check` turns a library error into the RuntimeError that the
// ctypes path raises.

void check(int rc, const char* what) {
  TORCH_CHECK(rc == 0, what, " failed (code ", rc, "): ", kf_last_error());
}

int dtype_code(const Tensor& t) { return t.scalar_type() == at::kHalf ? KF_F16 : KF_BF16; }

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

Tensor bytes_like(const Tensor& t, size_t n) {
  return at::empty({(int64_t)(n < 256 ? 256 : n)}, t.options().dtype(at::kByte));
}

bool decode_envelope(int64_t sq, int64_t sk, bool causal) { return !causal && sq <= 16 && sk >= 1024; }

// The split-KV decode over K/V views read in place; `seqlens` may be null.
Tensor launch_decode(const Tensor& q, const Tensor& k, const Tensor& v, double scale, int splits,
                     const int32_t* seqlens, int64_t sk, Tensor* lse) {
  const int64_t b = q.size(0), hq = q.size(1), sq = q.size(2), d = q.size(3), hkv = k.size(1);
  Tensor out = at::empty({b, hq, sq, d}, q.options());
  const size_t need = kf_decode_workspace_bytes(b, hq, hkv, sq, d, splits);
  Tensor ws;
  if (need) ws = bytes_like(q, need);
  check(kf_attn_decode(q.const_data_ptr(), k.const_data_ptr(), v.const_data_ptr(), out.data_ptr(),
                       lse ? lse->data_ptr<float>() : nullptr, seqlens, b, hq, hkv, sq, sk, d,
                       q.strides().data(), k.strides().data(), v.strides().data(),
                       out.strides().data(), (float)scale, splits, dtype_code(q),
                       need ? ws.data_ptr() : nullptr, need ? (size_t)ws.numel() : 0, stream_of(q)),
        "kf_attn_decode");
  return out;
}

// O and LSE for readable q, k, v (the launcher's own choice between the
// forward kernel and the split-KV decode).
Tensor launch_forward(const Tensor& q, const Tensor& k, const Tensor& v, bool causal, double scale,
                      Tensor& lse) {
  const int64_t b = q.size(0), hq = q.size(1), sq = q.size(2), d = q.size(3);
  const int64_t hkv = k.size(1), sk = k.size(2);
  lse = at::empty({b, hq, sq}, q.options().dtype(at::kFloat));
  if (decode_envelope(sq, sk, causal))
    return launch_decode(q, k, v, scale, kf_decode_num_splits(b, hq, hkv, sq, sk, d), nullptr, sk, &lse);
  Tensor out = at::empty({b, hq, sq, d}, q.options());
  check(kf_attn_fwd(q.const_data_ptr(), k.const_data_ptr(), v.const_data_ptr(), out.data_ptr(),
                    lse.data_ptr<float>(), b, hq, hkv, sq, sk, d, q.strides().data(),
                    k.strides().data(), v.strides().data(), out.strides().data(), (float)scale,
                    causal, dtype_code(q), stream_of(q)),
        "kf_attn_fwd");
  return out;
}

// Autograd over the forward and backward; saves (q, k, v, out, lse) as the
// Python Function of attention.py does. The node runs without the GIL.
struct HipAttention : torch::autograd::Function<HipAttention> {
  static Tensor forward(torch::autograd::AutogradContext* ctx, const Tensor& q, const Tensor& k,
                        const Tensor& v, bool causal, double scale) {
    Tensor lse;
    Tensor out = launch_forward(readable(q), readable(k), readable(v), causal, scale, lse);
    ctx->save_for_backward({q, k, v, out, lse});
    ctx->saved_data["causal"] = causal;
    ctx->saved_data["scale"] = scale;
    return out;
  }

  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                 torch::autograd::variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &out = saved[3], &lse = saved[4], &dout = grads[0];
    const bool causal = ctx->saved_data["causal"].toBool();
    const double scale = ctx->saved_data["scale"].toDouble();
    TORCH_CHECK(dout.sizes() == out.sizes(), "out and grad_out must have q's shape");
    TORCH_CHECK(dout.scalar_type() == out.scalar_type(),
                "HIP attention backward: all tensors must share one dtype");
    TORCH_CHECK(dout.device() == out.device(),
                "HIP attention backward: all tensors must be on the same device");
    const c10::OptionalDeviceGuard guard(out.device());
    const at::AutoGradMode no_grad(false);
    const Tensor q = readable(saved[0]), k = readable(saved[1]), v = readable(saved[2]);
    const Tensor o = readable(out), g = readable(dout), l = lse.contiguous();
    const int64_t b = q.size(0), hq = q.size(1), sq = q.size(2), d = q.size(3);
    const int64_t hkv = k.size(1), sk = k.size(2);
    Tensor dq = at::empty({b, hq, sq, d}, q.options());
    Tensor dk = at::empty({b, hkv, sk, d}, k.options());
    Tensor dv = at::empty({b, hkv, sk, d}, v.options());
    Tensor ws = bytes_like(q, kf_attn_bwd_workspace_bytes(b, hq, hkv, sq, sk, d, causal));
    check(kf_attn_bwd(q.const_data_ptr(), k.const_data_ptr(), v.const_data_ptr(),
                      o.const_data_ptr(), l.const_data_ptr<float>(), g.const_data_ptr(),
                      dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), b, hq, hkv, sq, sk, d,
                      q.strides().data(), k.strides().data(), v.strides().data(),
                      o.strides().data(), g.strides().data(), dq.strides().data(),
                      dk.strides().data(), dv.strides().data(), (float)scale, causal,
                      dtype_code(q), ws.data_ptr(), (size_t)ws.numel(), stream_of(q)),
          "kf_attn_bwd");
    return {dq, dk, dv, Tensor(), Tensor()};
  }
};

// Visible (query, key) pairs times 4 D B Hq, upper-left causal
// (_planning.attention_fwd_flops).
double forward_flops(const Tensor& q, const Tensor& k, bool causal) {
  const double b = q.size(0), hq = q.size(1), sq = q.size(2), d = q.size(3), sk = k.size(2);
  const double n = std::min(sq, sk);
  const double pairs = causal ? n * (n + 1) / 2 + std::max(0.0, sq - sk) * sk : sq * sk;
  return 4 * d * b * hq * pairs;
}

// ---------------------------------------------------------------------------
// Python entries (METH_FASTCALL).

PyObject* not_handled() { Py_RETURN_NOTIMPLEMENTED; }

bool exact_bool(PyObject* o, bool& v) {
  v = o == Py_True;
  return o == Py_True || o == Py_False;
}

// attention(q, k, v, causal, scale or None, backend, min_train_flops): the
// whole of the public attention() for calls that run on the HIP kernels. auto
// leaves training calls below min_train_flops to the Python path (SDPA).
PyObject* py_attention(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  bool causal;
  if (n != 7 || !exact_bool(args[3], causal) || !PyUnicode_CheckExact(args[5])) return not_handled();
  const bool automatic = PyUnicode_CompareWithASCIIString(args[5], "auto") == 0;
  if (!automatic && PyUnicode_CompareWithASCIIString(args[5], "hip") != 0 &&
      PyUnicode_CompareWithASCIIString(args[5], "triton") != 0)
    return not_handled();
  const Tensor *q = plain_tensor(args[0]), *k = plain_tensor(args[1]), *v = plain_tensor(args[2]);
  if (!q || !k || !v || !plain_mode() || !attention_args(*q, *k, *v)) return not_handled();
  double scale;
  if (args[4] == Py_None) scale = 1.0 / std::sqrt((double)q->size(3));
  else if (PyFloat_CheckExact(args[4])) scale = PyFloat_AS_DOUBLE(args[4]);
  else return not_handled();
  if (!std::isfinite(scale)) return not_handled();
  const bool grad = wants_grad({q, k, v});
  const bool decode = decode_envelope(q->size(2), k->size(2), causal);
  if (automatic && grad && !decode && forward_flops(*q, *k, causal) < PyFloat_AsDouble(args[6]))
    return not_handled();
  Tensor out;
  {
    pybind11::gil_scoped_release nogil;
    const c10::OptionalDeviceGuard guard(q->device());
    if (grad) {
      out = HipAttention::apply(*q, *k, *v, causal, scale);
    } else if (decode && layout_ok(*q) && layout_ok(*k) && layout_ok(*v)) {
      out = launch_decode(*q, *k, *v, scale,
                          kf_decode_num_splits(q->size(0), q->size(1), k->size(1), q->size(2),
                                               k->size(2), q->size(3)),
                          nullptr, k->size(2), nullptr);
    } else {
      Tensor lse;
      out = launch_forward(readable(*q), readable(*k), readable(*v), causal, scale, lse);
    }
  }
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// Caches [B, Hkv, capacity, D] with new tokens [B, Hkv, n, D] and queries
// [B, Hq, Sq, D] that the fused append + decode takes as they are.
bool append_args(const Tensor& q, const Tensor& kc, const Tensor& vc, const Tensor& nk, const Tensor& nv) {
  if (!attention_args(q, kc, vc) || nk.dim() != 4 || nk.sizes() != nv.sizes()) return false;
  const auto ns = nk.sizes(), cs = kc.sizes();
  if (ns[0] != cs[0] || ns[1] != cs[1] || ns[2] <= 0 || ns[3] != cs[3]) return false;
  if (nk.scalar_type() != q.scalar_type() || nv.scalar_type() != q.scalar_type() ||
      nk.device() != q.device() || nv.device() != q.device())
    return false;
  // The fused store may land anywhere below the capacity, through 32-bit
  // buffer offsets.
  if (((cs[2] - 1) * kc.stride(2) + cs[3]) * 2 >= (1ll << 31) ||
      ((cs[2] - 1) * vc.stride(2) + cs[3]) * 2 >= (1ll << 31))
    return false;
  return layout_ok(q) && layout_ok(kc) && layout_ok(vc);
}

struct AppendTensors {
  const Tensor *q, *kc, *vc, *nk, *nv;
  explicit AppendTensors(PyObject* const* a)
      : q(plain_tensor(a[0])), kc(plain_tensor(a[1])), vc(plain_tensor(a[2])),
        nk(plain_tensor(a[3])), nv(plain_tensor(a[4])) {}
  bool ok() const { return q && kc && vc && nk && nv && plain_mode() && append_args(*q, *kc, *vc, *nk, *nv); }
};

Tensor launch_append_decode(const AppendTensors& t, const int32_t* seqlens, int64_t past, int64_t max_length,
                            int splits, double scale) {
  const Tensor &q = *t.q, &kc = *t.kc, &vc = *t.vc;
  const Tensor nk = readable(*t.nk), nv = readable(*t.nv);
  const int64_t b = q.size(0), hq = q.size(1), sq = q.size(2), d = q.size(3), hkv = kc.size(1);
  Tensor out = at::empty({b, hq, sq, d}, q.options());
  Tensor ws = bytes_like(q, kf_decode_workspace_bytes(b, hq, hkv, sq, d, splits + 1));
  check(kf_attn_append_decode(q.const_data_ptr(), kc.data_ptr(), vc.data_ptr(), nk.const_data_ptr(),
                              nv.const_data_ptr(), out.data_ptr(), nullptr, seqlens, past, b, hq, hkv,
                              sq, nk.size(2), max_length, kc.size(2), d, q.strides().data(),
                              kc.strides().data(), vc.strides().data(), nk.strides().data(),
                              nv.strides().data(), out.strides().data(), (float)scale, splits,
                              dtype_code(q), ws.data_ptr(), (size_t)ws.numel(), stream_of(q)),
        "kf_attn_append_decode");
  return out;
}

// append_step(q, k_cache, v_cache, new_k, new_v, past_length, scale): one
// token at a scalar position (attention_forward_strided_append).
PyObject* py_append_step(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 7 || !PyLong_CheckExact(args[5]) || !PyFloat_CheckExact(args[6])) return not_handled();
  const AppendTensors t(args);
  if (!t.ok() || t.q->size(2) != 1 || t.nk->size(2) != 1) return not_handled();
  int over = 0;
  const long long past = PyLong_AsLongLongAndOverflow(args[5], &over);
  const double scale = PyFloat_AS_DOUBLE(args[6]);
  if (over || past < 0 || past + 1 > t.kc->size(2) || !std::isfinite(scale)) return not_handled();
  Tensor out;
  {
    pybind11::gil_scoped_release nogil;
    const c10::OptionalDeviceGuard guard(t.q->device());
    const int splits = kf_decode_num_splits(t.q->size(0), t.q->size(1), t.kc->size(1), 1, past, t.q->size(3));
    out = launch_append_decode(t, nullptr, past, past, splits, scale);
  }
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// Host lengths from a list of exact ints in [0, 2^30]; false otherwise.
bool read_lengths(PyObject* o, std::vector<int32_t>& out) {
  if (!PyList_CheckExact(o)) return false;
  const Py_ssize_t n = PyList_GET_SIZE(o);
  out.resize(n);
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject* x = PyList_GET_ITEM(o, i);
    if (!PyLong_CheckExact(x)) return false;
    int over = 0;
    const long v = PyLong_AsLongAndOverflow(x, &over);
    if (over || v < 0 || v > (1 << 30)) return false;
    out[i] = (int32_t)v;
  }
  return n > 0;
}

const int32_t* device_lengths(PyObject* o, const Tensor& q) {
  const Tensor* s = plain_tensor(o);
  if (!s || s->scalar_type() != at::kInt || s->device() != q.device() || s->dim() != 1 ||
      s->size(0) != q.size(0) || !s->is_contiguous())
    return nullptr;
  return s->const_data_ptr<int32_t>();
}

// append_ragged(q, k_cache, v_cache, new_k, new_v, seqlens, host_lengths,
// scale): n tokens at each sequence's own position
// (attention_append_decode_ragged without LSE).
PyObject* py_append_ragged(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  std::vector<int32_t> lens;
  if (n != 8 || !PyFloat_CheckExact(args[7]) || !read_lengths(args[6], lens)) return not_handled();
  const AppendTensors t(args);
  if (!t.ok() || (int64_t)lens.size() != t.q->size(0)) return not_handled();
  const int32_t* seqlens = device_lengths(args[5], *t.q);
  const int32_t top = *std::max_element(lens.begin(), lens.end());
  const double scale = PyFloat_AS_DOUBLE(args[7]);
  if (!seqlens || top + t.nk->size(2) > t.kc->size(2) || !std::isfinite(scale)) return not_handled();
  Tensor out;
  {
    pybind11::gil_scoped_release nogil;
    const c10::OptionalDeviceGuard guard(t.q->device());
    const int64_t b = t.q->size(0), hq = t.q->size(1), sq = t.q->size(2), d = t.q->size(3), hkv = t.kc->size(1);
    const int splits = top > 0 ? kf_decode_num_splits_ragged(b, hq, hkv, sq, lens.data(), d)
                               : kf_decode_num_splits(b, hq, hkv, sq, 0, d);
    out = launch_append_decode(t, seqlens, 0, top, splits, scale);
  }
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// decode_ragged(q, k_cache, v_cache, seqlens, host_lengths, scale): every
// sequence's own prefix (attention_decode_ragged without LSE, max_seqlen the
// longest host length).
PyObject* py_decode_ragged(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  std::vector<int32_t> lens;
  if (n != 6 || !PyFloat_CheckExact(args[5]) || !read_lengths(args[4], lens)) return not_handled();
  const Tensor *q = plain_tensor(args[0]), *k = plain_tensor(args[1]), *v = plain_tensor(args[2]);
  if (!q || !k || !v || !plain_mode() || !attention_args(*q, *k, *v) || !layout_ok(*q) ||
      !layout_ok(*k) || !layout_ok(*v) || (int64_t)lens.size() != q->size(0))
    return not_handled();
  const int32_t* seqlens = device_lengths(args[3], *q);
  const int32_t top = *std::max_element(lens.begin(), lens.end());
  const double scale = PyFloat_AS_DOUBLE(args[5]);
  if (!seqlens || top <= 0 || top > k->size(2) || !std::isfinite(scale)) return not_handled();
  Tensor out;
  {
    pybind11::gil_scoped_release nogil;
    const c10::OptionalDeviceGuard guard(q->device());
    const int splits = kf_decode_num_splits_ragged(q->size(0), q->size(1), k->size(1), q->size(2),
                                                   lens.data(), q->size(3));
    out = launch_decode(*q, *k, *v, scale, splits, seqlens, top, nullptr);
  }
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// step_args(q, k_cache, v_cache, new_k, new_v): True when a cache's
// append_and_attend would find nothing wrong with these tensors and the fused
// append + decode takes them (inference, gfx950, 16-bit, plain layouts).
PyObject* py_step_args(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 5) Py_RETURN_FALSE;
  const AppendTensors t(args);
  if (!t.ok() || wants_grad({t.q, t.nk, t.nv})) Py_RETURN_FALSE;
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

// store_lengths(starts, seqlens, lengths): the host lengths into a ragged
// cache's int64 and int32 device arrays, one launch that carries them by value
// instead of two copies. Like a copy from pageable memory it returns when the
// stream has done it: the cache's tensors may then be read on any stream. Not
// under graph capture, where a replay would repeat these values.
PyObject* py_store_lengths(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  std::vector<int32_t> lens;
  if (n != 3 || !read_lengths(args[2], lens)) return not_handled();
  const Tensor *starts = plain_tensor(args[0]), *seqlens = plain_tensor(args[1]);
  const int64_t count = (int64_t)lens.size();
  if (!starts || !seqlens || !plain_mode() || starts->scalar_type() != at::kLong ||
      seqlens->scalar_type() != at::kInt || starts->device() != seqlens->device() ||
      starts->dim() != 1 || seqlens->dim() != 1 || starts->size(0) != count ||
      seqlens->size(0) != count || !starts->is_contiguous() || !seqlens->is_contiguous() ||
      starts->is_inference() || seqlens->is_inference() || !is_gfx950(starts->device().index()))
    return not_handled();
  const c10::OptionalDeviceGuard guard(starts->device());
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  const auto stream = (hipStream_t)stream_of(*starts);
  if (hipStreamIsCapturing(stream, &capture) != hipSuccess || capture != hipStreamCaptureStatusNone) {
    (void)hipGetLastError();
    return not_handled();
  }
  {
    pybind11::gil_scoped_release nogil;
    check(kf_store_lengths(starts->data_ptr<int64_t>(), seqlens->data_ptr<int32_t>(), lens.data(), count, stream),
          "kf_store_lengths");
    c10::hip::getCurrentHIPStream(starts->device().index()).synchronize();
  }
  starts->unsafeGetTensorImpl()->bump_version();
  seqlens->unsafeGetTensorImpl()->bump_version();
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

PyMethodDef kMethods[] = {
    {"store_lengths", (PyCFunction)(void (*)(void))py_store_lengths, METH_FASTCALL, nullptr},
    {"attention", (PyCFunction)(void (*)(void))py_attention, METH_FASTCALL, nullptr},
    {"append_step", (PyCFunction)(void (*)(void))py_append_step, METH_FASTCALL, nullptr},
    {"append_ragged", (PyCFunction)(void (*)(void))py_append_ragged, METH_FASTCALL, nullptr},
    {"decode_ragged", (PyCFunction)(void (*)(void))py_decode_ragged, METH_FASTCALL, nullptr},
    {"step_args", (PyCFunction)(void (*)(void))py_step_args, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_native",
                       "C++ launch path of the kotflash_amd kernels.", -1, kMethods,
                       nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) { return PyModule_Create(&kModule); }
