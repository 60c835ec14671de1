// Native side of taomate_amd/kernels.py: checks torch tensors and calls the C
// ABI entry points with their pointers and strides.
//
// What bounds the small layers is the host: a 75-query audio layer is 50 us of
// GPU work behind 160 us of Python, of which the norm and attention wrappers'
// shape and stride checks and their 35-argument ctypes calls took 23 us each.
// The same checks here take about 2 us.  The functions take Python objects
// (METH_FASTCALL, no argument parsing), raise what the Python wrappers raised
// (ValueError, TypeError, NativeCallError) and let no C++ exception out.  The
// entry points' addresses come from the loaded library (bind), so this module
// links against torch only.

#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/autocast_mode.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <map>
#include <mutex>
#include <optional>
#include <string>
#include <utility>
#include <vector>

#include "../../include/taomate_ltx.h"

namespace {

struct Api {
  decltype(&ltx_last_error) last_error;
  decltype(&ltx_qk_rmsnorm_rope) qk_rmsnorm_rope;
  decltype(&ltx_qk_rmsnorm_rope_v) qk_rmsnorm_rope_v;
  decltype(&ltx_kv_append) kv_append;
  decltype(&ltx_kv_append_fp8_pair) kv_append_fp8_pair;
  decltype(&ltx_flash_attn_fwd) flash_attn_fwd;
  decltype(&ltx_flash_attn_fwd_noalloc) flash_attn_fwd_noalloc;
  decltype(&ltx_flash_attn_fwd_plain) flash_attn_fwd_plain;
  decltype(&ltx_flash_attn_workspace_size) flash_attn_workspace_size;
  decltype(&ltx_adaln) adaln;
  decltype(&ltx_skinny_linear) skinny_linear;
} api;
PyObject* native_call_error = nullptr;  // taomate_amd._native.NativeCallError

// An error to raise in Python; type nullptr: the Python error is already set.
struct Refused {
  PyObject* type;
  std::string msg;
};
[[noreturn]] void value_error(std::string msg) { throw Refused{PyExc_ValueError, std::move(msg)}; }
[[noreturn]] void type_error(std::string msg) { throw Refused{PyExc_TypeError, std::move(msg)}; }

using Opt = const at::Tensor*;  // nullptr: None

std::string shape(const at::Tensor& t) {
  std::string s = "(";
  for (int64_t i = 0; i < t.dim(); ++i) s += (i ? ", " : "") + std::to_string(t.size(i));
  return s + (t.dim() == 1 ? ",)" : ")");
}

const at::Tensor& tensor(PyObject* o) {
  if (!THPVariable_Check(o)) type_error(std::string("expected a tensor, got ") + Py_TYPE(o)->tp_name);
  return THPVariable_Unpack(o);
}
Opt optional(PyObject* o) { return o == Py_None ? nullptr : &tensor(o); }

int64_t integer(PyObject* o) {
  PyObject* n = PyNumber_Long(o);
  if (n == nullptr) throw Refused{nullptr, ""};
  const int64_t v = PyLong_AsLongLong(n);
  Py_DECREF(n);
  if (v == -1 && PyErr_Occurred()) throw Refused{nullptr, ""};
  return v;
}
double real(PyObject* o) {
  const double v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) throw Refused{nullptr, ""};
  return v;
}
bool truth(PyObject* o) {
  const int v = PyObject_IsTrue(o);
  if (v < 0) throw Refused{nullptr, ""};
  return v != 0;
}

// An owned reference.
struct Ref {
  PyObject* o;
  explicit Ref(PyObject* p) : o(p) {
    if (p == nullptr) throw Refused{nullptr, ""};
  }
  Ref(Ref&& r) noexcept : o(std::exchange(r.o, nullptr)) {}
  Ref& operator=(Ref&& r) noexcept {
    std::swap(o, r.o);
    return *this;
  }
  ~Ref() { Py_XDECREF(o); }
};

void need_gpu(Opt t) {
  if (t != nullptr && !t->is_cuda()) value_error("taomate_amd kernels take device tensors (got a CPU tensor)");
}
int code(const at::Tensor& t) {
  switch (t.scalar_type()) {
    case at::kFloat: return LTX_F32;
    case at::kBFloat16: return LTX_BF16;
    case at::kByte:
    case at::kFloat8_e4m3fn: return LTX_F8E4M3;
    default: type_error("unsupported dtype torch." + std::string(at::toString(t.scalar_type())));
  }
}
void* ptr(Opt t) { return t == nullptr ? nullptr : t->data_ptr(); }
template <typename T = float>
T* ptr_as(Opt t) { return static_cast<T*>(ptr(t)); }
void* stream_of(const at::Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

struct GilReleased {
  PyThreadState* state = PyEval_SaveThread();
  ~GilReleased() { PyEval_RestoreThread(state); }
};
// Runs enqueue(), which calls the entry point `name`, with the GIL released, as ctypes does.
template <typename Enqueue>
void released(const char* name, Enqueue enqueue) {
  if (api.last_error == nullptr) throw Refused{PyExc_RuntimeError, "the native library is not bound"};
  int rc;
  {
    GilReleased r;
    rc = enqueue();
  }
  if (rc != 0)
    throw Refused{native_call_error, std::string(name) + " failed (" + std::to_string(rc) + "): " + api.last_error()};
}
template <typename Fn, typename... Args>
void call(const char* name, Fn fn, Args... args) {
  released(name, [&] { return fn(args...); });
}

// ---------------------------------------------------------------- norm + RoPE
struct Rows {
  int64_t len, bs, ls;
};
// (len, batch stride, row stride) of a [B, L, H*D] (or [B, L, H, D]) row tensor.
Rows rows(const at::Tensor& t, int64_t hd) {
  if (t.dim() == 4) {
    if (t.stride(3) != 1 || t.stride(2) != t.size(3)) value_error("rows must be contiguous over (H, D)");
  } else if (t.dim() != 3 || t.size(-1) != hd || t.stride(2) != 1) {
    value_error("expected [B, L, " + std::to_string(hd) + "] rows with a contiguous last dim, got " + shape(t));
  }
  return {t.size(1), t.stride(0), t.stride(1)};
}

// cos and sin point into `pair`, which may be the only holder of its items (a
// table given as one stacked tensor or an iterator): it lives as long as they do.
struct Table {
  std::optional<Ref> pair;
  Opt cos = nullptr, sin = nullptr;
  int64_t tb = 0, th = 0, tt = 0;
};
Table table(PyObject* o, int64_t H, int64_t D, int64_t L, int64_t B) {
  Table r;
  if (o == Py_None) return r;
  PyObject* seq = r.pair.emplace(PySequence_Fast(o, "a RoPE table is a (cos, sin) pair")).o;
  if (PySequence_Fast_GET_SIZE(seq) != 2) value_error("a RoPE table is a (cos, sin) pair");
  r.cos = &tensor(PySequence_Fast_GET_ITEM(seq, 0));
  r.sin = &tensor(PySequence_Fast_GET_ITEM(seq, 1));
  const at::Tensor &c = *r.cos, &s = *r.sin;
  if (c.sizes() != s.sizes() || c.strides() != s.strides() || c.scalar_type() != s.scalar_type())
    value_error("cos/sin tables must share shape, strides and dtype");
  if (c.dim() != 4 || c.size(1) != H || c.size(3) != D / 2 || c.size(2) < L)
    value_error("RoPE table " + shape(c) + " does not match H=" + std::to_string(H) + " D/2=" + std::to_string(D / 2) +
                " T>=" + std::to_string(L));
  if (c.stride(3) != 1) value_error("RoPE table last dim must be contiguous");
  if (c.size(0) != 1 && c.size(0) != B)
    value_error("RoPE table batch " + std::to_string(c.size(0)) + " vs input batch " + std::to_string(B));
  r.tb = c.size(0) == 1 ? 0 : c.stride(0);
  r.th = c.stride(1);
  r.tt = c.stride(2);
  return r;
}

// (q_in, q_out, gamma_q, eps_q, q_tab, H, D, k_in, k_out, gamma_k, eps_k, k_tab, v_in, v_out)
void qk_rmsnorm_rope(PyObject* const* a) {
  const at::Tensor &q_in = tensor(a[0]), &q_out = tensor(a[1]);
  const Opt gq = optional(a[2]), k_in = optional(a[7]), k_out = optional(a[8]), gk = optional(a[9]);
  const Opt v_in = optional(a[12]), v_out = optional(a[13]);
  const int64_t H = integer(a[5]), D = integer(a[6]), HD = H * D;
  for (Opt t : {Opt(&q_in), Opt(&q_out), k_in, k_out, gq, gk, v_in, v_out}) need_gpu(t);
  for (Opt t : {Opt(&q_out), k_in, k_out, gq, gk})
    if (t != nullptr && t->scalar_type() != q_in.scalar_type())
      type_error("q/k inputs, outputs and gammas must share one dtype");
  const Rows q = rows(q_in, HD), qo = rows(q_out, HD);
  const int64_t B = q_in.size(0);
  if (qo.len != q.len || q_out.size(0) != B) value_error("q_out shape mismatch");
  const Table qt = table(a[4], H, D, q.len, B);
  Rows k{0, 0, 0}, ko{0, 0, 0};
  Table kt;
  if (k_in != nullptr) {
    if (k_out == nullptr) value_error("k_out shape mismatch");
    k = rows(*k_in, HD);
    ko = rows(*k_out, HD);
    if (ko.len != k.len || k_in->size(0) != B || k_out->size(0) != B) value_error("k_out shape mismatch");
    kt = table(a[11], H, D, k.len, B);
  }
  if (qt.cos != nullptr && kt.cos != nullptr && qt.cos->scalar_type() != kt.cos->scalar_type())
    type_error("q and k RoPE tables must share a dtype");
  const Opt tab = qt.cos != nullptr ? qt.cos : kt.cos;
  const int tab_code = tab != nullptr ? code(*tab) : LTX_BF16;
  for (Opt g : {gq, gk})
    if (g != nullptr && (g->numel() != HD || !g->is_contiguous()))
      value_error("gamma must be a contiguous [H*D] vector");
  const float eq = a[3] == Py_None ? -1.0f : (float)real(a[3]), ek = a[10] == Py_None ? -1.0f : (float)real(a[10]);
  const int c = code(q_in);
  if (v_in == nullptr && v_out == nullptr) {
    call("ltx_qk_rmsnorm_rope", api.qk_rmsnorm_rope, c, B, H, D, ptr(&q_in), q.len, q.bs, q.ls, ptr(&q_out), qo.bs,
         qo.ls, ptr(gq), eq, ptr(qt.cos), ptr(qt.sin), qt.tb, qt.th, qt.tt, ptr(k_in), k.len, k.bs, k.ls,
         ptr(k_out), ko.bs, ko.ls, ptr(gk), ek, ptr(kt.cos), ptr(kt.sin), kt.tb, kt.th,
         kt.tt, tab_code, stream_of(q_in));
    return;
  }
  if (v_in == nullptr || v_out == nullptr) value_error("v_in and v_out go together");
  if (v_in->dim() != 4 || v_out->sizes() != v_in->sizes() || v_in->size(0) != B || v_in->size(2) != H ||
      v_in->size(3) != D)
    value_error("V " + shape(*v_in) + " -> " + shape(*v_out) + " does not match B=" + std::to_string(B) +
                " H=" + std::to_string(H) + " D=" + std::to_string(D));
  if (v_in->scalar_type() != at::kBFloat16 || v_out->scalar_type() != at::kBFloat16 || v_in->stride(3) != 1)
    value_error("V must be bf16 with a contiguous head dim");
  if (v_out->stride(1) != 1) value_error("v_out must be key-major (token stride 1)");
  call("ltx_qk_rmsnorm_rope_v", api.qk_rmsnorm_rope_v, c, B, H, D, ptr(&q_in), q.len, q.bs, q.ls, ptr(&q_out), qo.bs,
       qo.ls, ptr(gq), eq, ptr(qt.cos), ptr(qt.sin), qt.tb, qt.th, qt.tt, ptr(k_in), k.len, k.bs, k.ls, ptr(k_out),
       ko.bs, ko.ls, ptr(gk), ek, ptr(kt.cos), ptr(kt.sin), kt.tb, kt.th, kt.tt, tab_code, ptr(v_in), v_in->size(1),
       v_in->stride(0), v_in->stride(1), v_in->stride(2), ptr(v_out), v_out->stride(0), v_out->stride(2),
       v_out->stride(3), stream_of(q_in));
}

// --------------------------------------------------------------------- append
// (src, dst, scales, frame_tokens)
void kv_append(PyObject* const* a) {
  const at::Tensor &src = tensor(a[0]), &dst = tensor(a[1]);
  const Opt scales = optional(a[2]);
  const int64_t frame = integer(a[3]);
  need_gpu(&src), need_gpu(&dst), need_gpu(scales);
  if (src.dim() != 4 || dst.sizes() != src.sizes())
    value_error("kv_append: shapes " + shape(src) + " vs " + shape(dst));
  if (src.stride(3) != 1) value_error("kv_append: src head dim must be contiguous");
  const int64_t B = src.size(0), L = src.size(1), H = src.size(2), D = src.size(3);
  if (dst.stride(3) != 1 && (dst.stride(1) != 1 || code(dst) != LTX_BF16))
    value_error("kv_append: dst must be token-major or bf16 key-major");
  int64_t sc_bs = 0, sc_hs = 0;
  if (code(dst) == LTX_F8E4M3) {
    if (scales == nullptr || scales->scalar_type() != at::kFloat)
      value_error("kv_append: fp8 destination needs float32 scales");
    if (frame <= 0 || L % frame != 0 || scales->dim() != 3 || scales->size(0) != B || scales->size(1) != H ||
        scales->size(2) != L / frame || (L != 0 && scales->stride(2) != 1))
      value_error("kv_append: scales " + shape(*scales) + " for L=" + std::to_string(L) +
                  ", frame=" + std::to_string(frame));
    sc_bs = scales->stride(0), sc_hs = scales->stride(1);
  }
  call("ltx_kv_append", api.kv_append, code(src), code(dst), B, L, H, D, ptr(&src), src.stride(0), src.stride(1),
       src.stride(2), ptr(&dst), dst.stride(0), dst.stride(1), dst.stride(2), dst.stride(3), ptr_as(scales), sc_bs,
       sc_hs, frame, stream_of(src));
}

// (k, k_dst, k_scales, v, v_dst, v_scales, frame_tokens)
void kv_append_fp8_pair(PyObject* const* a) {
  const at::Tensor &k = tensor(a[0]), &kd = tensor(a[1]), &ks = tensor(a[2]);
  const at::Tensor &v = tensor(a[3]), &vd = tensor(a[4]), &vs = tensor(a[5]);
  const int64_t frame = integer(a[6]);
  for (Opt t : {&k, &kd, &ks, &v, &vd, &vs}) need_gpu(t);
  if (k.dim() != 4 || v.sizes() != k.sizes() || kd.sizes() != k.sizes() || vd.sizes() != k.sizes())
    value_error("kv_append_fp8_pair: shapes " + shape(k) + ", " + shape(v) + ", " + shape(kd) + ", " + shape(vd));
  if (k.scalar_type() != at::kBFloat16 || v.scalar_type() != at::kBFloat16)
    type_error("kv_append_fp8_pair: K and V must be bf16");
  if (code(kd) != LTX_F8E4M3 || code(vd) != LTX_F8E4M3)
    type_error("kv_append_fp8_pair: destinations must be fp8 (uint8 codes)");
  if (k.stride(3) != 1 || v.stride(3) != 1 || kd.stride(3) != 1 || vd.stride(3) != 1)
    value_error("kv_append_fp8_pair: head dim must be contiguous");
  if (kd.strides() != vd.strides()) value_error("kv_append_fp8_pair: K and V destinations must share strides");
  const int64_t B = k.size(0), L = k.size(1), H = k.size(2), D = k.size(3);
  if (frame <= 0 || L % frame != 0)
    value_error("kv_append_fp8_pair: L=" + std::to_string(L) + " is not a whole number of " + std::to_string(frame) +
                "-token frames");
  for (Opt s : {&ks, &vs})
    if (s->scalar_type() != at::kFloat || s->dim() != 3 || s->size(0) != B || s->size(1) != H ||
        s->size(2) != L / frame || (L != 0 && s->stride(2) != 1))
      value_error("kv_append_fp8_pair: scales " + shape(*s) + " for L=" + std::to_string(L) +
                  ", frame=" + std::to_string(frame));
  if (ks.strides() != vs.strides()) value_error("kv_append_fp8_pair: K and V scales must share strides");
  call("ltx_kv_append_fp8_pair", api.kv_append_fp8_pair, B, L, H, D, frame, ptr(&k), k.stride(0), k.stride(1),
       k.stride(2), ptr(&kd), ptr_as(&ks), ptr(&v), v.stride(0), v.stride(1), v.stride(2), ptr(&vd), ptr_as(&vs),
       kd.stride(0), kd.stride(1), kd.stride(2), ks.stride(0), ks.stride(1), stream_of(k));
}

// ------------------------------------------------------------------ attention
// The split's workspace: one tensor per (device, stream), grown on demand and
// at most the library's largest plan.  A call enqueues the attention and the
// merge of its partials as separate launches, so it holds the workspace's lock
// until both are in the stream: threads that share a stream (PyTorch's all start
// on one) take turns.  The lock is taken with the GIL released and given back
// before the GIL is taken again, so neither waits for the other.  The map is
// kept for the life of the process (never destroyed: the allocator may be gone
// by then), and its entries never move.
//
// A call that is captured into a graph takes a tensor of its own instead, from
// the graph's memory pool: replays keep its address, which must neither be freed
// when a later call grows the stream's workspace nor be shared with other graphs
// or eager calls that run beside them.
struct Workspace {
  std::mutex mu;
  at::Tensor buf;
};
Workspace& workspace(const at::Tensor& q, void* stream) {
  static std::mutex mu;
  static auto* kept = new std::map<std::pair<int, void*>, Workspace>;
  std::lock_guard<std::mutex> lock(mu);
  return (*kept)[{q.device().index(), stream}];
}

bool capturing(void* stream) {
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  return stream != nullptr && hipStreamIsCapturing(static_cast<hipStream_t>(stream), &st) == hipSuccess &&
         st != hipStreamCaptureStatusNone;
}

PyObject *str_k, *str_v, *str_ks, *str_vs;

// (q, segments, out, key_mask, lse, scale, frame_tokens, noalloc, key_lens, segment_batch_strides)
void flash_attn(PyObject* const* a) {
  const at::Tensor &q = tensor(a[0]), &out = tensor(a[2]);
  const Opt mask = optional(a[3]), lse = optional(a[4]);
  const float scale = a[5] == Py_None ? 0.0f : (float)real(a[5]);
  const int64_t frame = integer(a[6]);
  const bool noalloc = truth(a[7]), own_bs = truth(a[9]);
  need_gpu(&q), need_gpu(&out), need_gpu(mask), need_gpu(lse);
  if (q.scalar_type() != at::kBFloat16 || out.scalar_type() != at::kBFloat16)
    type_error("flash_attn: q and out must be bf16");
  if (q.dim() != 4 || out.sizes() != q.sizes() || q.stride(3) != 1 || out.stride(3) != 1)
    value_error("flash_attn: q/out must be [B, Lq, H, D] with contiguous D");
  const int64_t B = q.size(0), Lq = q.size(1), H = q.size(2), D = q.size(3);

  Ref list(PySequence_Fast(a[1], "flash_attn: segments must be a sequence"));
  const Py_ssize_t n_all = PySequence_Fast_GET_SIZE(list.o);
  std::vector<Ref> held;  // the segments' attributes, alive for the call
  held.reserve(4 * n_all);
  const at::Tensor* k[LTX_MAX_SEGMENTS];
  const at::Tensor* v[LTX_MAX_SEGMENTS];
  PyObject* seg[LTX_MAX_SEGMENTS];
  int n = 0, total = 0;
  for (Py_ssize_t i = 0; i < n_all; ++i) {
    PyObject* s = PySequence_Fast_GET_ITEM(list.o, i);
    held.emplace_back(PyObject_GetAttr(s, str_k));
    const at::Tensor& kk = tensor(held.back().o);
    if (kk.size(1) <= 0) continue;
    ++total;
    if (n == LTX_MAX_SEGMENTS) continue;
    held.emplace_back(PyObject_GetAttr(s, str_v));
    k[n] = &kk;
    v[n] = &tensor(held.back().o);
    seg[n++] = s;
  }
  if (total == 0) value_error("flash_attn: no keys");
  if (total > LTX_MAX_SEGMENTS)
    value_error("flash_attn: " + std::to_string(total) + " segments > " + std::to_string(LTX_MAX_SEGMENTS));
  const int kv_code = code(*k[0]);
  int64_t lk = 0;
  const void *kp[LTX_MAX_SEGMENTS], *vp[LTX_MAX_SEGMENTS];
  int64_t lens[LTX_MAX_SEGMENTS], seg_bs[LTX_MAX_SEGMENTS];
  for (int i = 0; i < n; ++i) {
    for (const at::Tensor* t : {k[i], v[i]}) {
      need_gpu(t);
      if (t->dim() != 4 || t->size(0) != B || t->size(2) != H || t->size(3) != D)
        value_error("flash_attn: segment " + shape(*t) + " vs q " + shape(q));
      if (code(*t) != kv_code) value_error("flash_attn: segments must share one dtype");
    }
    const at::Tensor &ki = *k[i], &vi = *v[i], &k0 = *k[0], &v0 = *v[0];
    if (ki.stride(3) != 1) value_error("flash_attn: K head dim must be contiguous");
    if (vi.stride(3) != 1 && vi.stride(1) != 1) value_error("flash_attn: V must be token-major or key-major");
    for (int d = own_bs ? 1 : 0; d < 4; ++d)
      if ((d < 3 && ki.stride(d) != k0.stride(d)) || vi.stride(d) != v0.stride(d))
        value_error("flash_attn: all K/V segments must share strides");
    if (own_bs && (ki.stride(0) != vi.stride(0) || ki.stride(1) != vi.stride(1) || ki.stride(2) != vi.stride(2) ||
                   vi.stride(3) != 1 || kv_code != LTX_BF16))
      value_error("flash_attn: segment_batch_strides takes token-major bf16 K and V of equal strides");
    if (vi.size(1) != ki.size(1)) value_error("flash_attn: k/v segment lengths differ");
    lk += ki.size(1);
    kp[i] = ki.data_ptr();
    vp[i] = vi.data_ptr();
    lens[i] = ki.size(1);
    seg_bs[i] = ki.stride(0);
  }
  const at::Tensor &k0 = *k[0], &v0 = *v[0];
  const bool fp8 = kv_code == LTX_F8E4M3;
  const float *ksp[LTX_MAX_SEGMENTS], *vsp[LTX_MAX_SEGMENTS];
  int64_t sc_bs = 0, sc_hs = 0;
  if (fp8)
    for (int i = 0; i < n; ++i)
      for (int w = 0; w < 2; ++w) {
        held.emplace_back(PyObject_GetAttr(seg[i], w ? str_vs : str_ks));
        const Opt sc = optional(held.back().o);
        if (sc == nullptr || sc->scalar_type() != at::kFloat || sc->dim() != 3 || sc->size(0) != B ||
            sc->size(1) != H)
          value_error("flash_attn: fp8 segments need float32 [B, H, nF] scales");
        if (sc->size(2) * frame < lens[i] || (sc->size(2) > 1 && sc->stride(2) != 1))
          value_error("flash_attn: fp8 scales do not cover the segment");
        if (i == 0 && w == 0)
          sc_bs = sc->stride(0), sc_hs = sc->stride(1);
        else if (sc->stride(0) != sc_bs || sc->stride(1) != sc_hs)
          value_error("flash_attn: fp8 scale tensors must share strides");
        (w ? vsp : ksp)[i] = static_cast<const float*>(sc->data_ptr());
      }
  int64_t mask_bs = 0;
  if (mask != nullptr) {
    if (mask->scalar_type() != at::kFloat || mask->dim() != 2 || mask->size(1) != lk ||
        (mask->size(0) != 1 && mask->size(0) != B) || mask->stride(1) != 1)
      value_error("flash_attn: key_mask must be float32 [B, " + std::to_string(lk) + "] with contiguous keys");
    mask_bs = mask->size(0) == 1 ? 0 : mask->stride(0);
  }
  if (lse != nullptr && (lse->scalar_type() != at::kFloat || lse->dim() != 3 || lse->size(0) != B ||
                         lse->size(1) != H || lse->size(2) != Lq || !lse->is_contiguous()))
    value_error("flash_attn: lse must be contiguous float32 [B, H, Lq]");
  if (own_bs && (mask != nullptr || a[8] != Py_None || noalloc))
    value_error("flash_attn: segment_batch_strides takes no mask, key counts or noalloc");
  std::vector<int64_t> kl;
  if (a[8] != Py_None) {
    Ref seq(PySequence_Fast(a[8], "flash_attn: key_lens must be a sequence"));
    bool ok = PySequence_Fast_GET_SIZE(seq.o) == B;
    for (Py_ssize_t i = 0; ok && i < PySequence_Fast_GET_SIZE(seq.o); ++i) {
      kl.push_back(integer(PySequence_Fast_GET_ITEM(seq.o, i)));
      ok = kl.back() >= 0 && kl.back() <= lk;
    }
    if (!ok)
      value_error("flash_attn: key_lens must hold " + std::to_string(B) + " counts in [0, " + std::to_string(lk) + "]");
  }
  void* st = stream_of(q);
  const int64_t* kl_data = a[8] != Py_None ? kl.data() : nullptr;
  auto general = [&](auto fn, auto... tail) {
    return fn(ptr(&q), B, Lq, H, D, q.stride(0), q.stride(1), q.stride(2), (int64_t)n, kp, vp, lens, k0.stride(0),
              k0.stride(1), k0.stride(2), v0.stride(0), v0.stride(1), v0.stride(2), v0.stride(3), kv_code,
              fp8 ? ksp : nullptr, fp8 ? vsp : nullptr, sc_bs, sc_hs, frame, ptr_as(mask), mask_bs, kl_data, ptr(&out),
              out.stride(0), out.stride(1), out.stride(2), ptr_as(lse), scale, tail...);
  };
  if (noalloc) {
    released("ltx_flash_attn_fwd_noalloc", [&] { return general(api.flash_attn_fwd_noalloc, st); });
    return;
  }
  int64_t need = 0;
  call("ltx_flash_attn_workspace_size", api.flash_attn_workspace_size, B, Lq, H, D, &need);
  released(own_bs ? "ltx_flash_attn_fwd_plain" : "ltx_flash_attn_fwd", [&] {
    std::unique_lock<std::mutex> lock;
    at::Tensor buf;
    const auto bytes = [&] { return at::empty({need}, q.options().dtype(at::kByte)); };
    if (need > 0 && capturing(st)) {
      buf = bytes();
    } else if (need > 0) {
      Workspace& ws = workspace(q, st);
      lock = std::unique_lock<std::mutex>(ws.mu);
      if (!ws.buf.defined() || ws.buf.numel() < need) ws.buf = bytes();
      buf = ws.buf;
    }
    void* wsp = buf.defined() ? buf.data_ptr() : nullptr;
    const int64_t ws_bytes = buf.defined() ? buf.numel() : 0;
    if (!own_bs) return general(api.flash_attn_fwd, wsp, ws_bytes, st);
    return api.flash_attn_fwd_plain(ptr(&q), B, Lq, H, D, q.stride(0), q.stride(1), q.stride(2), (int64_t)n, kp, vp,
                                    lens, seg_bs, k0.stride(1), k0.stride(2), ptr(&out), out.stride(0),
                                    out.stride(1), out.stride(2), ptr_as(lse), scale, wsp, ws_bytes, st);
  });
}

// ---------------------------------------------------------------------- AdaLN
// (x, y, gate, x_out, n_out, scale, shift, eps)
void adaln(PyObject* const* a) {
  static const char* const names[7] = {"x", "y", "gate", "x_out", "n_out", "scale", "shift"};
  Opt t[7] = {&tensor(a[0])};
  for (int i = 1; i < 7; ++i) t[i] = optional(a[i]);
  for (Opt o : t) need_gpu(o);
  const at::Tensor& x = *t[0];
  if (x.dim() != 3 || x.scalar_type() != at::kBFloat16) value_error("adaln: x must be bf16 [B, L, C]");
  const int64_t B = x.size(0), L = x.size(1), C = x.size(2);
  struct {
    void* p;
    int64_t bs, ls;
  } r[7] = {};
  for (int i = 0; i < 7; ++i) {
    if (t[i] == nullptr) continue;
    const at::Tensor& o = *t[i];
    if (o.scalar_type() != at::kBFloat16 || o.dim() != 3 || o.size(0) != B || o.size(2) != C || o.stride(2) != 1)
      value_error(std::string("adaln: ") + names[i] + " must be bf16 [B, L or 1, C] with contiguous channels");
    if (o.size(1) == L)
      r[i] = {o.data_ptr(), o.stride(0), L > 1 ? o.stride(1) : 0};
    else if (o.size(1) == 1)
      r[i] = {o.data_ptr(), o.stride(0), 0};
    else
      value_error(std::string("adaln: ") + names[i] + " rows " + std::to_string(o.size(1)) +
                  " vs L=" + std::to_string(L));
  }
  for (int i : {1, 3, 4})
    if (t[i] != nullptr && t[i]->size(1) != L)
      value_error(std::string("adaln: ") + names[i] + " must have L=" + std::to_string(L) + " rows");
  call("ltx_adaln", api.adaln, B, L, C, r[0].p, r[0].bs, r[0].ls, r[1].p, r[1].bs, r[1].ls, r[2].p, r[2].bs, r[2].ls,
       r[3].p, r[3].bs, r[3].ls, r[4].p, r[4].bs, r[4].ls, r[5].p, r[5].bs, r[5].ls, r[6].p, r[6].bs, r[6].ls,
       (float)real(a[7]), stream_of(x));
}

// -------------------------------------------------------------- skinny linear
// (x, weight, bias, y, silu)
void skinny_linear(PyObject* const* a) {
  const at::Tensor &x = tensor(a[0]), &w = tensor(a[1]), &y = tensor(a[3]);
  const Opt bias = optional(a[2]);
  for (Opt t : {Opt(&x), Opt(&w), bias, Opt(&y)}) {
    need_gpu(t);
    if (t != nullptr && t->scalar_type() != at::kBFloat16) type_error("skinny_linear: every tensor must be bf16");
  }
  if (x.dim() != 2 || w.dim() != 2 || y.dim() != 2 || x.size(1) != w.size(1) || y.size(0) != x.size(0) ||
      y.size(1) != w.size(0) || x.stride(1) != 1 || w.stride(1) != 1 || y.stride(1) != 1)
    value_error("skinny_linear: x " + shape(x) + ", weight " + shape(w) + ", y " + shape(y));
  if (bias != nullptr && (bias->dim() != 1 || bias->size(0) != w.size(0) || bias->stride(0) != 1))
    value_error("skinny_linear: bias must be a contiguous [N] vector");
  call("ltx_skinny_linear", api.skinny_linear, x.size(0), w.size(0), x.size(1), ptr(&x), x.stride(0),
       (int)truth(a[4]), ptr(&w), w.stride(0), ptr(bias), ptr(&y), y.stride(0), stream_of(x));
}

// is_eager(): whether an op on plain tensors would run as it is written, as far
// as the thread's state tells: no gradients, autocast, torch function or dispatch
// mode, function transform or trace (the last two and dispatch modes add keys to
// the thread's included set).
PyObject* is_eager(PyObject*, PyObject*) {
  const auto tls = c10::impl::tls_local_dispatch_key_set();
  return PyBool_FromLong(!c10::GradMode::is_enabled() && !at::autocast::is_autocast_enabled(at::kCUDA) &&
                         at::impl::PythonTorchFunctionTLS::stack_len() == 0 &&
                         c10::impl::TorchDispatchModeTLS::stack_len() == 0 &&
                         (tls.included_ - c10::default_included_set).empty());
}

// row_operands(x, weight, bias): whether skinny_linear takes them, and they are
// tensors or parameters without a subclass.
PyObject* row_operands(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 3) {
    PyErr_Format(PyExc_TypeError, "expected 3 arguments, got %zd", nargs);
    return nullptr;
  }
  auto plain = [&](PyObject* o) {
    return THPVariable_CheckExact(o) && THPVariable_Unpack(o).layout() == at::kStrided &&
           THPVariable_Unpack(o).scalar_type() == at::kBFloat16 && !THPVariable_Unpack(o).is_neg();
  };
  bool ok = false;
  try {
    ok = plain(args[0]) && plain(args[1]) && (args[2] == Py_None || plain(args[2]));
    if (ok) {
      const at::Tensor &x = THPVariable_Unpack(args[0]), &w = THPVariable_Unpack(args[1]);
      auto aligned = [](const at::Tensor& t) { return (uintptr_t)t.data_ptr() % 16 == 0; };
      ok = x.is_cuda() && x.dim() == 2 && x.size(0) >= 1 && x.size(0) <= LTX_SKINNY_MAX_ROWS && x.size(1) >= 8 &&
           x.size(1) <= LTX_SKINNY_MAX_K && x.size(1) % 8 == 0 && x.stride(1) == 1 && x.stride(0) % 8 == 0 &&
           aligned(x) && w.dim() == 2 && w.size(1) == x.size(1) && w.is_contiguous() && w.device() == x.device() &&
           aligned(w);
      if (ok && args[2] != Py_None) {
        const at::Tensor& b = THPVariable_Unpack(args[2]);
        ok = b.dim() == 1 && b.size(0) == w.size(0) && b.is_contiguous() && b.device() == x.device();
      }
    }
  } catch (const std::exception&) {
    ok = false;  // a tensor without storage
  }
  return PyBool_FromLong(ok);
}

// ------------------------------------------------------------------- bindings
template <void (*Fn)(PyObject* const*), Py_ssize_t N>
PyObject* entry(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != N) {
    PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", N, nargs);
    return nullptr;
  }
  try {
    Fn(args);
    Py_RETURN_NONE;
  } catch (const Refused& r) {
    if (r.type != nullptr) PyErr_SetString(r.type, r.msg.c_str());
  } catch (const c10::IndexError& e) {
    PyErr_SetString(PyExc_IndexError, e.what_without_backtrace());
  } catch (const std::exception& e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
  }
  return nullptr;
}

// bind(addresses by entry point name, NativeCallError)
PyObject* bind(PyObject*, PyObject* args) {
  PyObject *dict, *error;
  if (!PyArg_ParseTuple(args, "O!O", &PyDict_Type, &dict, &error)) return nullptr;
  Api next{};
  bool ok = true;
  auto get = [&](const char* name, auto& fn) {
    PyObject* o = PyDict_GetItemString(dict, name);
    void* p = o != nullptr ? PyLong_AsVoidPtr(o) : nullptr;
    ok = ok && p != nullptr;
    fn = reinterpret_cast<std::remove_reference_t<decltype(fn)>>(p);
  };
  get("ltx_last_error", next.last_error);
  get("ltx_qk_rmsnorm_rope", next.qk_rmsnorm_rope);
  get("ltx_qk_rmsnorm_rope_v", next.qk_rmsnorm_rope_v);
  get("ltx_kv_append", next.kv_append);
  get("ltx_kv_append_fp8_pair", next.kv_append_fp8_pair);
  get("ltx_flash_attn_fwd", next.flash_attn_fwd);
  get("ltx_flash_attn_fwd_noalloc", next.flash_attn_fwd_noalloc);
  get("ltx_flash_attn_fwd_plain", next.flash_attn_fwd_plain);
  get("ltx_flash_attn_workspace_size", next.flash_attn_workspace_size);
  get("ltx_adaln", next.adaln);
  get("ltx_skinny_linear", next.skinny_linear);
  if (!ok) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "bind: missing entry point addresses");
    return nullptr;
  }
  api = next;
  Py_INCREF(error);
  Py_XSETREF(native_call_error, error);
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"bind", bind, METH_VARARGS, nullptr},
    {"qk_rmsnorm_rope", (PyCFunction)(void*)&entry<qk_rmsnorm_rope, 14>, METH_FASTCALL, nullptr},
    {"kv_append", (PyCFunction)(void*)&entry<kv_append, 4>, METH_FASTCALL, nullptr},
    {"kv_append_fp8_pair", (PyCFunction)(void*)&entry<kv_append_fp8_pair, 7>, METH_FASTCALL, nullptr},
    {"flash_attn", (PyCFunction)(void*)&entry<flash_attn, 10>, METH_FASTCALL, nullptr},
    {"skinny_linear", (PyCFunction)(void*)&entry<skinny_linear, 5>, METH_FASTCALL, nullptr},
    {"adaln", (PyCFunction)(void*)&entry<adaln, 8>, METH_FASTCALL, nullptr},
    {"is_eager", is_eager, METH_NOARGS, nullptr},
    {"row_operands", (PyCFunction)(void*)&row_operands, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_ltx_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__ltx_host() {
  str_k = PyUnicode_InternFromString("k");
  str_v = PyUnicode_InternFromString("v");
  str_ks = PyUnicode_InternFromString("k_scales");
  str_vs = PyUnicode_InternFromString("v_scales");
  return PyModule_Create(&module);
}
