// The eager host path of the attention backend: one Python call takes the tensors of a pass to the C ABI.
//
// A pass of a few microseconds of GPU time (a short prompt, one user's decode step) is bound by the host:
// through Python views, the operator registry and ctypes it issues in 33 .. 55 us.  This module reads
// addresses, sizes and strides from the tensors directly and calls the same entry points with the same
// arguments.  It serves exactly the ordinary form of a pass (plain bfloat16 rows on the current device, the
// caches' layouts, int32 tables; nobody watching operators: no dispatch mode, function mode or trace); for anything else it answers None before it has issued anything, and the
// caller's general path takes the pass, raises what is to be raised and converts what is to be
// converted.  Scratch comes from the caching allocator on the current stream, call by call: nothing is kept
// between calls, so streams, threads and graph captures need no care of their own.  (A latent step takes the operators', which
// belongs to the calling thread and to the default stream outside a capture.)
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/TracerMode.h>
#include <ATen/core/grad_mode.h>
#include <ATen/record_function.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>

#include "ttpa.h"

namespace {

// Largest scratch a pass may ask for (the operators' limit).
constexpr int64_t kScratchLimit = int64_t(8) << 30;

constexpr c10::DispatchKeySet kWrapped({c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                        c10::DispatchKey::Functionalize, c10::DispatchKey::Python, c10::DispatchKey::ZeroTensor,
                                        c10::DispatchKey::Negative, c10::DispatchKey::Conjugate});

struct Pass {
  int device;
  bool grad;

  // A plain tensor on the current device that autograd does not watch; null otherwise.  (A tensor inside vmap or
  // a functional transform, one to be functionalized and one with a lazy sign are plain Python tensors whose memory is not theirs to read;
  // one with a forward-mode tangent would lose it.)
  const at::Tensor *plain(PyObject *o) const {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor &t = THPVariable_Unpack(o);
    if (!t.defined() || !t.is_cuda() || t.get_device() != device || t.layout() != at::kStrided) return nullptr;
    if (t.unsafeGetTensorImpl()->key_set().has_any(kWrapped) || !t.has_storage()) return nullptr;
    if (grad && t.requires_grad()) return nullptr;
    if (t.unsafeGetTensorImpl()->autograd_meta() && t._fw_grad(0).defined()) return nullptr;
    return &t;
  }
  // [rows, cols] bfloat16 with contiguous, 16-byte aligned rows.
  const at::Tensor *rows(PyObject *o, int64_t cols) const {
    const at::Tensor *t = plain(o);
    if (!t || t->scalar_type() != at::kBFloat16 || t->dim() != 2 || t->size(1) != cols || t->stride(1) != 1 || t->stride(0) % 8 ||
        reinterpret_cast<uintptr_t>(t->data_ptr()) % 16)
      return nullptr;
    return t;
  }
  const at::Tensor *table(PyObject *o) const {
    const at::Tensor *t = plain(o);
    return t && t->scalar_type() == at::kInt && t->dim() == 2 && t->stride(1) == 1 ? t : nullptr;
  }
  // `n` whole numbers, int32 or int64.
  const at::Tensor *numbers(PyObject *o, int64_t n) const {
    const at::Tensor *t = plain(o);
    if (!t || (t->scalar_type() != at::kInt && t->scalar_type() != at::kLong) || t->dim() != 1 || t->size(0) != n || !t->is_contiguous())
      return nullptr;
    return t;
  }
};

inline void *at_ptr(const at::Tensor *t) { return t ? t->data_ptr() : nullptr; }
inline int is_i64(const at::Tensor *t) { return t && t->scalar_type() == at::kLong; }
inline void written(const at::Tensor *t) {
  if (!t->is_inference()) t->unsafeGetTensorImpl()->bump_version();
}
// The interpreter lock is not held while scratch is allocated and kernels are launched: either may wait (a launch for a
// full queue, as long as the GPU takes), and other Python threads run meanwhile, as they do through ctypes.
class Unlocked {
 public:
  Unlocked() : state_(PyEval_SaveThread()) {}
  ~Unlocked() { PyEval_RestoreThread(state_); }
  Unlocked(const Unlocked &) = delete;

 private:
  PyThreadState *state_;
};
inline at::Tensor scratch(int64_t bytes, const at::Tensor *like) {
  return at::empty({bytes}, like->options().dtype(at::kByte));
}

PyObject *result(const char *entry, int rc) { return rc == TTPA_OK ? PyLong_FromLong(0) : Py_BuildValue("(si)", entry, rc); }

// attention_pass(query, key, value, k_cache, v_cache, page_table, cache_position, fill_page_table, batch_idx, chunk_start,
//                sinks, output, users, heads, kv_heads, head_size, scale, window, chunk_end)
// -> 0, (name, status) of the entry point that failed, or None: not an ordinary pass, nothing was issued.  A profiler
// sees the names of the operators that the pass stands for.
PyObject *attention_pass(PyObject *, PyObject *const *v, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 19) {
    PyErr_SetString(PyExc_TypeError, "attention_pass takes 19 arguments");
    return nullptr;
  }
  if (c10::impl::TorchDispatchModeTLS::any_modes_set() || at::impl::torch_function_mode_enabled() ||
      at::tracer::impl::is_dispatch_enabled())
    Py_RETURN_NONE;
  if (!THPVariable_CheckExact(v[0]) || !THPVariable_Unpack(v[0]).is_cuda()) Py_RETURN_NONE;  // (ahead of any question to the device)
  for (int i = 12; i < 18; ++i)
    if (i == 16 ? !PyFloat_Check(v[i]) : !PyLong_Check(v[i])) Py_RETURN_NONE;
  const int64_t users = PyLong_AsLongLong(v[12]), hq = PyLong_AsLongLong(v[13]), hkv = PyLong_AsLongLong(v[14]);
  const int64_t d = PyLong_AsLongLong(v[15]), window = PyLong_AsLongLong(v[17]);
  const float scale = (float)PyFloat_AsDouble(v[16]);
  int64_t most_keys = PyLong_Check(v[18]) ? PyLong_AsLongLong(v[18]) : 0;
  if (PyErr_Occurred()) {  // a number that does not fit 64 bits
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  if (users <= 0 || hq <= 0 || hkv <= 0 || d <= 0 || d % 8 || hq % hkv || window < 0) Py_RETURN_NONE;

  const Pass p{(int)c10::hip::current_device(), at::GradMode::is_enabled()};
  const at::Tensor *q = p.rows(v[0], hq * d), *k = p.rows(v[1], hkv * d), *val = p.rows(v[2], hkv * d);
  if (!q || !k || !val) Py_RETURN_NONE;
  const int64_t tokens = q->size(0);
  if (tokens == 0 || tokens % users || k->size(0) != tokens || val->size(0) != tokens || k->stride(0) != val->stride(0)) Py_RETURN_NONE;
  const int64_t s = tokens / users;
  const at::Tensor *out = p.plain(v[11]);
  if (!out || out->scalar_type() != at::kBFloat16 || !out->is_contiguous() || out->numel() != tokens * hq * d ||
      reinterpret_cast<uintptr_t>(out->data_ptr()) % 16)
    Py_RETURN_NONE;

  const at::Tensor *kc = p.plain(v[3]), *vc = p.plain(v[4]);
  if (!kc || !vc || kc->dim() != 4 || kc->sizes() != vc->sizes() || kc->scalar_type() != vc->scalar_type() || !kc->is_contiguous() ||
      !vc->is_contiguous() || kc->size(0) == 0 || kc->size(1) != hkv || kc->size(3) != d)
    Py_RETURN_NONE;
  const bool bfp8 = kc->scalar_type() == at::kByte;
  if (!bfp8 && kc->scalar_type() != at::kBFloat16) Py_RETURN_NONE;
  const int64_t nb = kc->size(0);
  int64_t bs = kc->size(2);
  if (bfp8) {
    if (bs % 17) Py_RETURN_NONE;
    bs = bs / 17 * 16;
  }
  const int fmt = bfp8 ? TTPA_KV_BFP8 : TTPA_KV_BF16;
  void *stream = c10::hip::getCurrentHIPStream((c10::DeviceIndex)p.device).stream();

  if (s == 1) {  // decode step: cache update and attention
    const at::Tensor *pt = p.table(v[5]), *pos = p.numbers(v[6], users), *sinks = nullptr;
    if (!pt || pt->size(0) != users || !pos) Py_RETURN_NONE;
    if (v[10] != Py_None) {
      sinks = p.plain(v[10]);
      if (!sinks || sinks->scalar_type() != at::kFloat || sinks->numel() != hq || !sinks->is_contiguous()) Py_RETURN_NONE;
    }
    const size_t bytes = ttpa_paged_decode_workspace_bytes((int32_t)users, (int32_t)hq, (int32_t)hkv, (int32_t)d);
    if (bytes == 0) Py_RETURN_NONE;
    RECORD_FUNCTION("tt::paged_update_kv_decode_out_", std::vector<c10::IValue>());
    written(kc), written(vc), written(out);
    const auto launch = [&] {
      const Unlocked unlocked;
      const at::Tensor ws = scratch((int64_t)bytes, out);
      return ttpa_paged_update_decode(
          out->data_ptr(), hq * d, d, q->data_ptr(), q->stride(0), d, kc->data_ptr(), vc->data_ptr(), k->data_ptr(), val->data_ptr(),
          k->stride(0), d, static_cast<const int32_t *>(pt->data_ptr()), pt->stride(0), pos->data_ptr(), is_i64(pos), (int32_t)users,
          (int32_t)hq, (int32_t)hkv, (int32_t)d, (int32_t)bs, (int32_t)pt->size(1), (int32_t)nb, scale, fmt, (int32_t)window,
          static_cast<const float *>(at_ptr(sinks)), ws.data_ptr(), bytes, stream);
    };
    return result("ttpa_paged_update_decode", launch());
  }

  // prefill: fill through the fill table, attention on the fresh K / V or on the cache
  if (v[10] != Py_None || !(scale > 0.f)) Py_RETURN_NONE;
  const at::Tensor *fill = p.table(v[7]), *bidx = p.numbers(v[8], users);
  if (!fill || !bidx || fill->size(0) == 0 || s > fill->size(1) * bs) Py_RETURN_NONE;
  const int32_t *fill_pt = static_cast<const int32_t *>(fill->data_ptr());
  const auto fill_caches = [&] {
    RECORD_FUNCTION("tt::paged_fill_kv_cache_", std::vector<c10::IValue>());
    const Unlocked unlocked;
    return ttpa_paged_fill_cache_kv(
        kc->data_ptr(), vc->data_ptr(), k->data_ptr(), val->data_ptr(), s * k->stride(0), d, k->stride(0), fill_pt, fill->stride(0),
        bidx->data_ptr(), is_i64(bidx), (int32_t)users, (int32_t)fill->size(0), (int32_t)hkv, (int32_t)s, (int32_t)bs, (int32_t)d,
        (int32_t)fill->size(1), (int32_t)nb, fmt, stream);
  };
  if (v[9] == Py_None) {
    if (s % 32) Py_RETURN_NONE;
    if (bfp8) {  // (a quantising fill is a launch of its own)
      written(kc), written(vc), written(out);
      if (const int rc = fill_caches()) return result("ttpa_paged_fill_cache_kv", rc);
      RECORD_FUNCTION("tt::scaled_dot_product_attention_out", std::vector<c10::IValue>());
      const auto launch = [&] {
        const Unlocked unlocked;
        return ttpa_sdpa_prefill_expanded(
            out->data_ptr(), s * hq * d, d, hq * d, q->data_ptr(), s * q->stride(0), d, q->stride(0), k->data_ptr(), val->data_ptr(),
            s * k->stride(0), d, k->stride(0), nullptr, 0, nullptr, nullptr, 0, 0, (int32_t)users, (int32_t)hq, (int32_t)hkv, (int32_t)s,
            (int32_t)s, (int32_t)d, 0, 0, 0, 1, scale, (int32_t)window, TTPA_KV_BF16, nullptr, 0, stream);
      };
      return result("ttpa_sdpa_prefill_expanded", launch());
    }
    RECORD_FUNCTION("tt::paged_fill_kv_prefill_out_", std::vector<c10::IValue>());
    written(kc), written(vc), written(out);
    const auto launch = [&] {
      const Unlocked unlocked;
      return ttpa_sdpa_prefill_fill(
          out->data_ptr(), s * hq * d, d, hq * d, q->data_ptr(), s * q->stride(0), d, q->stride(0), k->data_ptr(), val->data_ptr(),
          s * k->stride(0), d, k->stride(0), (int32_t)users, (int32_t)hq, (int32_t)hkv, (int32_t)s, (int32_t)s, (int32_t)d, 1, scale,
          (int32_t)window, kc->data_ptr(), vc->data_ptr(), fill_pt, fill->stride(0), bidx->data_ptr(), is_i64(bidx),
          (int32_t)fill->size(0), (int32_t)bs, (int32_t)fill->size(1), (int32_t)nb, stream);
    };
    return result("ttpa_sdpa_prefill_fill", launch());
  }
  const at::Tensor *pt = p.table(v[5]), *start = p.numbers(v[9], 1);
  if (!pt || pt->size(0) != users || !start || is_i64(start)) Py_RETURN_NONE;
  // (what a graph captures is replayed for other chunks)
  if (most_keys <= 0 || c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None) most_keys = 0;
  int64_t bytes = ttpa_sdpa_prefill_bounded_scratch_bytes((int32_t)users, (int32_t)hq, (int32_t)hkv, (int32_t)s, (int32_t)d, (int32_t)bs,
                                                          (int32_t)pt->size(1), fmt, most_keys);
  if (bytes < 0 || bytes > kScratchLimit) bytes = 0;
  written(kc), written(vc), written(out);
  if (const int rc = fill_caches()) return result("ttpa_paged_fill_cache_kv", rc);
  RECORD_FUNCTION("tt::chunked_scaled_dot_product_attention_out", std::vector<c10::IValue>());
  const auto launch = [&] {
    const Unlocked unlocked;
    at::Tensor ws;
    if (bytes) {
      try {
        ws = scratch(bytes, out);
      } catch (const c10::OutOfMemoryError &) {  // sized by the page table, not by the pass: it runs without, too
        bytes = 0;
      }
    }
    return ttpa_sdpa_prefill_bounded(
        out->data_ptr(), s * hq * d, d, hq * d, q->data_ptr(), s * q->stride(0), d, q->stride(0), kc->data_ptr(), vc->data_ptr(), 0, 0,
        0, static_cast<const int32_t *>(pt->data_ptr()), pt->stride(0), static_cast<const int32_t *>(start->data_ptr()), nullptr, 0, 0,
        (int32_t)users, (int32_t)hq, (int32_t)hkv, (int32_t)s, (int32_t)(pt->size(1) * bs), (int32_t)d, (int32_t)bs,
        (int32_t)pt->size(1), (int32_t)nb, 1, scale, 0, fmt, most_keys, bytes ? ws.data_ptr() : nullptr, bytes, stream);
  };
  return result("ttpa_sdpa_prefill_expanded", launch());  // (its bounded form; an error reads as the operators')
  END_HANDLE_TH_ERRORS
}

// A weight [heads, rows, columns] as the latent kernels read it: rows or columns contiguous, every other stride whole
// 16-byte pieces, aligned.
const at::Tensor *weight(const Pass &p, PyObject *o, int64_t heads, int64_t rows, int64_t columns) {
  const at::Tensor *t = p.plain(o);
  if (!t || t->scalar_type() != at::kBFloat16 || t->dim() != 3 || t->size(0) != heads || t->size(1) != rows || t->size(2) != columns) return nullptr;
  const int64_t rs = t->stride(1), cs = t->stride(2), other = cs == 1 ? rs : cs;
  if ((rs != 1 && cs != 1) || t->stride(0) % 8 || other % 8 || other <= 0 || other >= (1 << 23) || reinterpret_cast<uintptr_t>(t->data_ptr()) % 16)
    return nullptr;
  return t;
}

// latent_pass(q_nope, q_rope, latent, rope, cache, page_table, cache_position, fill_page_table, w_uk_t, w_uv, output, heads, scale,
//             workspace)
// The pass of a latent layer (128 + 64 query features, latent width 512, values of 128; causal): decode step or prompt.
// -> as attention_pass.  workspace(bytes, device) is the operators' own scratch of a decode step, a thread's (the interpreter lock
// is not held between the launches that hand data through it) and sized for the largest grid, not for the pass.
PyObject *latent_pass(PyObject *, PyObject *const *v, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 14) {
    PyErr_SetString(PyExc_TypeError, "latent_pass takes 14 arguments");
    return nullptr;
  }
  if (c10::impl::TorchDispatchModeTLS::any_modes_set() || at::impl::torch_function_mode_enabled() ||
      at::tracer::impl::is_dispatch_enabled())
    Py_RETURN_NONE;
  if (!THPVariable_CheckExact(v[0]) || !THPVariable_Unpack(v[0]).is_cuda()) Py_RETURN_NONE;  // (ahead of any question to the device)
  if (!PyLong_Check(v[11]) || !PyFloat_Check(v[12])) Py_RETURN_NONE;
  const int64_t heads = PyLong_AsLongLong(v[11]);
  const float scale = (float)PyFloat_AsDouble(v[12]);
  if (PyErr_Occurred()) {  // a number that does not fit 64 bits
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  if (heads <= 0 || heads > 65535) Py_RETURN_NONE;
  const Pass p{(int)c10::hip::current_device(), at::GradMode::is_enabled()};
  // [tokens, heads, width] with contiguous, 16-byte aligned rows
  const auto parts = [&](PyObject *o, int64_t per_token, int64_t width) -> const at::Tensor * {
    const at::Tensor *t = p.plain(o);
    return t && t->scalar_type() == at::kBFloat16 && t->dim() == 3 && t->size(1) == per_token && t->size(2) == width && t->stride(2) == 1 &&
                   t->stride(0) % 8 == 0 && t->stride(1) % 8 == 0 && reinterpret_cast<uintptr_t>(t->data_ptr()) % 16 == 0
               ? t
               : nullptr;
  };
  const at::Tensor *qn = parts(v[0], heads, 128), *qr = parts(v[1], heads, 64), *lat = p.rows(v[2], 512), *rope = parts(v[3], 1, 64);
  if (!qn || !qr || !lat || !rope) Py_RETURN_NONE;
  const int64_t tokens = qn->size(0);
  if (tokens == 0 || qr->size(0) != tokens || lat->size(0) != tokens || rope->size(0) != tokens) Py_RETURN_NONE;
  const at::Tensor *pos = p.plain(v[6]);
  if (!pos || pos->dim() != 1 || pos->size(0) == 0 || tokens % pos->size(0)) Py_RETURN_NONE;
  const int64_t users = pos->size(0), s = tokens / users;
  const at::Tensor *cache = p.plain(v[4]);
  if (!cache || cache->scalar_type() != at::kBFloat16 || cache->dim() != 4 || cache->size(0) == 0 || cache->size(1) != 1 || cache->size(2) == 0 ||
      cache->size(3) != 576 || !cache->is_contiguous() || reinterpret_cast<uintptr_t>(cache->data_ptr()) % 16)
    Py_RETURN_NONE;
  const int64_t nb = cache->size(0), bs = cache->size(2);
  const at::Tensor *uk = weight(p, v[8], heads, 128, 512), *uv = weight(p, v[9], heads, 512, 128), *out = p.plain(v[10]);
  if (!uk || !uv || !out || out->scalar_type() != at::kBFloat16 || !out->is_contiguous() || out->numel() != tokens * heads * 128) Py_RETURN_NONE;
  // (an output that the kernels' stores cannot take is copied to)
  const bool storable = reinterpret_cast<uintptr_t>(out->data_ptr()) % 16 == 0;
  void *stream = c10::hip::getCurrentHIPStream((c10::DeviceIndex)p.device).stream();

  if (s == 1) {
    const at::Tensor *pt = p.table(v[5]);
    pos = p.numbers(v[6], users);
    if (!pt || pt->size(0) != users || pt->size(1) == 0 || !pos || users > 1024) Py_RETURN_NONE;
    const size_t bytes = ttpa_latent_decode_step_workspace_bytes((int32_t)users, (int32_t)heads);
    if (bytes == 0) Py_RETURN_NONE;
    PyObject *const device = PyObject_GetAttrString(v[10], "device");
    if (!device) return nullptr;
    PyObject *const kept = PyObject_CallFunction(v[13], "nO", (Py_ssize_t)bytes, device);
    Py_DECREF(device);
    if (!kept) return nullptr;
    const at::Tensor ws = THPVariable_Check(kept) ? THPVariable_Unpack(kept) : at::Tensor();
    Py_DECREF(kept);
    if (!ws.defined() || !ws.is_cuda() || ws.get_device() != p.device || ws.nbytes() < bytes) Py_RETURN_NONE;
    RECORD_FUNCTION("tt::latent_decode_step_", std::vector<c10::IValue>());
    written(cache), written(out);
    const auto launch = [&] {
      const Unlocked unlocked;
      const at::Tensor target = storable ? *out : at::empty(out->sizes(), out->options());
      const int rc = ttpa_latent_decode_step_strided(
          target.data_ptr(), heads * 128, 128, qn->data_ptr(), qn->stride(0), qn->stride(1), qr->data_ptr(), qr->stride(0), qr->stride(1),
          lat->data_ptr(), lat->stride(0), rope->data_ptr(), rope->stride(0), uk->data_ptr(), uk->stride(0), uk->stride(1), uk->stride(2),
          uv->data_ptr(), uv->stride(0), uv->stride(1), uv->stride(2), cache->data_ptr(), static_cast<const int32_t *>(pt->data_ptr()),
          pt->stride(0), pos->data_ptr(), is_i64(pos), (int32_t)users, (int32_t)heads, (int32_t)bs, (int32_t)pt->size(1), (int32_t)nb, scale,
          ws.data_ptr(), bytes, stream);
      if (!storable && rc == TTPA_OK) out->copy_(target);
      return rc;
    };
    return result("ttpa_latent_decode_step_strided", launch());
  }

  const at::Tensor *fill = p.table(v[7]);
  if (!(scale > 0.f) || s % 32 || !fill || fill->size(0) == 0 || s > fill->size(1) * bs || lat->stride(0) <= 0 || lat->stride(0) >= (1 << 23))
    Py_RETURN_NONE;
  const int64_t bytes = ttpa_latent_prompt_workspace_bytes((int32_t)users, (int32_t)heads, (int32_t)s);
  if (tokens > 65535 * 32 || bytes <= 0 || bytes > kScratchLimit) Py_RETURN_NONE;
  RECORD_FUNCTION("tt::latent_prompt", std::vector<c10::IValue>());
  written(cache), written(out);
  const auto launch = [&] {
    const Unlocked unlocked;
    const at::Tensor ws = scratch(bytes, out), target = storable ? *out : at::empty(out->sizes(), out->options());
    const int rc = ttpa_latent_prompt(
        target.data_ptr(), heads * 128, 128, qn->data_ptr(), qn->stride(0), qn->stride(1), qr->data_ptr(), qr->stride(0), qr->stride(1),
        lat->data_ptr(), lat->stride(0), rope->data_ptr(), rope->stride(0), uk->data_ptr(), uk->stride(0), uk->stride(1), uk->stride(2),
        uv->data_ptr(), uv->stride(0), uv->stride(1), uv->stride(2), cache->data_ptr(), static_cast<const int32_t *>(fill->data_ptr()),
        fill->stride(0), (int32_t)users, (int32_t)fill->size(0), (int32_t)heads, (int32_t)s, (int32_t)bs, (int32_t)fill->size(1), (int32_t)nb,
        scale, ws.data_ptr(), bytes, stream);
    if (!storable && rc == TTPA_OK) out->copy_(target);
    return rc;
  };
  return result("ttpa_latent_prompt", launch());
  END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"latent_pass", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(latent_pass)), METH_FASTCALL,
     "One pass of a latent layer from its tensors; None if it is not an ordinary one."},
    {"attention_pass", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(attention_pass)), METH_FASTCALL,
     "One pass of an attention layer from its tensors; None if it is not an ordinary one."},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "ttpa_host", "Eager host path of the attention backend.", -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit_ttpa_host() { return PyModule_Create(&module); }
