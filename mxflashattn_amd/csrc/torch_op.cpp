// Host-side torch operator in front of the C ABI (include/mxfa_mi355x.h): the
// decode calls and the cache writes without Python's per-argument marshalling
// (a call of several query tokens, an fp8 cache or options took 17-30 us of
// host time through ctypes, an append about 12; small calls were bound by it).
//
// decode(q, k_cache, v_cache, block_table, cache_seqlens, scale, out,
//        num_splits, seqlen_add) takes the common call (one query
// token per sequence, caches of q's 16-bit type, int32 table and lengths,
// every tensor on the current GPU with layouts the kernels read in place),
// launches it on torch's current HIP stream and returns the output.
// num_splits None is mxfa_split_heuristic's choice. For any
// other call it launches nothing and returns None; the Python binding then
// takes the call and gives its usual errors. decode_tokens (the general call),
// contiguous_decode, reshape_and_cache and append_kv below do the same.
//
// The workspace is grow-only per (device, stream): a buffer replaced by a
// larger one stays alive until the process ends, since a HIP graph captured
// earlier keeps its address. A replay therefore belongs on the stream of the
// capture, or ordered with it: on another stream, beside eager calls on that
// one, both write the workspace and give wrong numbers (never a read or write
// outside the tensors: what the kernels address by is in no workspace, or
// clamped where it is read).
//
// Reference counterpart: the pybind binding paged_decode_split of
// csrc_native/m1_binding.cpp:78-115 (checks, output and workspace, launch on
// the caller's stream).

#include <torch/extension.h>

#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <limits>
#include <map>
#include <mutex>
#include <string>
#include <utility>
#include <vector>

#include "mxfa_mi355x.h"
#include "mxfa_package.h"

namespace {

struct Workspaces {
  std::mutex mu;
  std::map<std::pair<int, void *>, at::Tensor> live;
  std::vector<at::Tensor> retired;
};

// Never destroyed: the tensors must outlive every graph that holds their
// address, and static destruction at exit would run after the HIP runtime.
Workspaces &workspaces() {
  static Workspaces *w = new Workspaces();
  return *w;
}

at::Tensor workspace(const at::Device &device, void *stream, size_t bytes) {
  Workspaces &w = workspaces();
  std::lock_guard<std::mutex> lock(w.mu);
  const auto key = std::make_pair((int)device.index(), stream);
  auto it = w.live.find(key);
  if (it == w.live.end() || (size_t)it->second.numel() < bytes) {
    int64_t size = std::max<int64_t>((int64_t)bytes, 1 << 20);
    if (it != w.live.end()) {
      size = std::max<int64_t>(size, 2 * it->second.numel());
      w.retired.push_back(it->second);
    }
    at::Tensor t = at::empty({size}, at::TensorOptions().dtype(at::kByte).device(device));
    w.live[key] = t;
    return t;
  }
  return it->second;
}

// First rows and lengths of a call on keys in consecutive rows: memory that no
// other call or graph writes before the decode has read it (mxfa_package.h). A
// graph gets memory of its own pool; eager calls of one stream, which follow each
// other, share at most 128 KB (16,000 sequences) that no graph holds (an
// allocation per call cost 1 us of a short call's 15).
at::Tensor rows_table(const at::Device &device, void *stream, int64_t batch, bool capturing) {
  const auto options = at::TensorOptions().dtype(at::kInt).device(device);
  if (capturing) return at::empty({2 * batch}, options);
  struct Tables {
    std::mutex mu;
    std::map<std::pair<int, void *>, at::Tensor> live;
  };
  static Tables *tables = new Tables();  // never destroyed, as the workspaces
  std::lock_guard<std::mutex> lock(tables->mu);
  at::Tensor &t = tables->live[std::make_pair((int)device.index(), stream)];
  if (!t.defined() || t.numel() < 2 * batch)
    t = at::empty({std::max<int64_t>(2 * batch, 1024)}, options);
  return t;
}

// MXFA_POISON_OUTPUTS=1 (a debugging aid, read once; the Python binding reads
// the same variable): outside graph capture the output of a call is filled with
// NaN and the workspace of each of its launches with 0xff bytes, so a row or a
// piece the kernels fail to write shows up as NaN rather than as a stale value.
bool poison_outputs() {
  static const bool on = [] {
    const char *e = std::getenv("MXFA_POISON_OUTPUTS");
    return e != nullptr && std::string(e) == "1";
  }();
  return on;
}

void poison(void *stream, at::Tensor *out, at::Tensor *ws) {
  // An output whose rows overlap is refused by the launch; it is not filled.
  if (!poison_outputs() || (out && at::has_internal_overlap(*out) != at::MemOverlap::No)) return;
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing((hipStream_t)stream, &status) != hipSuccess ||
      status != hipStreamCaptureStatusNone)
    return;
  if (out) out->fill_(std::numeric_limits<float>::quiet_NaN());
  if (ws) ws->fill_(0xff);
}

// (bytes of the live workspaces, bytes of the retired ones)
std::pair<int64_t, int64_t> workspace_bytes() {
  Workspaces &w = workspaces();
  std::lock_guard<std::mutex> lock(w.mu);
  int64_t live = 0, retired = 0;
  for (const auto &kv : w.live) live += kv.second.numel();
  for (const auto &t : w.retired) retired += t.numel();
  return {live, retired};
}

bool aligned(const void *p, uintptr_t n) { return ((uintptr_t)p & (n - 1)) == 0; }

// Compute units of a device, looked up once (the split heuristic's input).
int num_cus(int device) {
  static std::mutex mu;
  static std::map<int, int> cus;
  std::lock_guard<std::mutex> lock(mu);
  auto it = cus.find(device);
  if (it != cus.end()) return it->second;
  int n = 0;
  if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess)
    n = 0;
  cus[device] = n;
  return n;
}

// q or out as [B, HQ, HD] strides (batch, head), or false when the layout is
// not [B, HQ, HD] / [B, 1, HQ, HD] with a contiguous last dim.
bool bhd_strides(const at::Tensor &t, int64_t &sb, int64_t &sh) {
  if (t.dim() == 3) {
    sb = t.stride(0);
    sh = t.stride(1);
  } else if (t.dim() == 4 && t.size(1) == 1) {
    sb = t.stride(0);
    sh = t.stride(2);
  } else {
    return false;
  }
  return t.stride(-1) == 1;
}

py::object decode(const at::Tensor &q, const at::Tensor &k_cache, const at::Tensor &v_cache,
                  const at::Tensor &block_table, const at::Tensor &cache_seqlens, double scale,
                  const c10::optional<at::Tensor> &out_arg,
                  const c10::optional<int64_t> &num_splits_arg, int64_t seqlen_add) {
  const at::ScalarType dt = q.scalar_type();
  if (dt != at::kHalf && dt != at::kBFloat16) return py::none();
  if (!q.is_cuda() || k_cache.scalar_type() != dt || v_cache.scalar_type() != dt) return py::none();
  if (k_cache.dim() != 4 || !v_cache.sizes().equals(k_cache.sizes())) return py::none();
  if (!v_cache.strides().equals(k_cache.strides()) || k_cache.stride(3) != 1) return py::none();
  if (block_table.scalar_type() != at::kInt || cache_seqlens.scalar_type() != at::kInt)
    return py::none();
  if (block_table.dim() != 2 || block_table.stride(1) != 1 || cache_seqlens.dim() != 1 ||
      !cache_seqlens.is_contiguous())
    return py::none();
  const at::Device device = q.device();
  if (k_cache.device() != device || v_cache.device() != device ||
      block_table.device() != device || cache_seqlens.device() != device)
    return py::none();
  if (device.index() != c10::hip::current_device()) return py::none();
  int64_t q_sb, q_sh;
  if (!bhd_strides(q, q_sb, q_sh)) return py::none();
  const int64_t batch = q.size(0), hq = q.size(-2), hd = q.size(-1);
  const int64_t pages = k_cache.size(0), ps = k_cache.size(1), hkv = k_cache.size(2);
  if (k_cache.size(3) != hd || block_table.size(0) != batch || cache_seqlens.size(0) != batch ||
      block_table.size(1) < 1)
    return py::none();
  // The kernels' 16-byte fragments: aligned pointers, strides of 8 elements.
  if (!aligned(q.data_ptr(), 16) || !aligned(k_cache.data_ptr(), 16) ||
      !aligned(v_cache.data_ptr(), 16) || ((q_sb | q_sh) & 7) || q_sb < 0 || q_sh < 0 ||
      (hq > 1 && q_sh < hd))
    return py::none();
  at::Tensor out;
  int64_t o_sb, o_sh;
  if (out_arg.has_value()) {
    out = *out_arg;
    if (out.scalar_type() != dt || out.device() != device || !out.sizes().equals(q.sizes()) ||
        !bhd_strides(out, o_sb, o_sh) || !aligned(out.data_ptr(), 8) || ((o_sb | o_sh) & 3))
      return py::none();
  } else {
    out = at::empty(q.sizes(), q.options());
    bhd_strides(out, o_sb, o_sh);
  }
  void *stream = (void *)c10::hip::getCurrentHIPStream(device.index()).stream();
  // No num_splits: the heuristic's choice. Values the C ABI rejects (0, below
  // MXFA_SPLITS_PER_SEQUENCE, above 65535) go to the binding's path, which
  // reports them.
  int ns = 0;
  if (num_splits_arg.has_value()) {
    const int64_t v = *num_splits_arg;
    if ((v <= 0 && v != MXFA_SPLITS_PER_SEQUENCE) || v > 65535) return py::none();
    ns = (int)v;
  } else if (mxfa_split_heuristic((int)batch, (int)hq, (int)hkv, (int)hd, (int)ps,
                                  (int)block_table.size(1), num_cus(device.index()),
                                  &ns) != MXFA_OK) {
    return py::none();
  }
  size_t ws_bytes = 0;
  if (mxfa_split_decode_workspace_size((int)batch, (int)hq, (int)hd, ns, &ws_bytes) != MXFA_OK)
    return py::none();
  at::Tensor ws_t;
  if (ws_bytes) ws_t = workspace(device, stream, ws_bytes);
  void *ws = ws_bytes ? ws_t.data_ptr() : nullptr;
  poison(stream, &out, ws_bytes ? &ws_t : nullptr);
  const int rc = mxfa_split_decode_launch(
      q.data_ptr(), q_sb, q_sh, k_cache.data_ptr(), v_cache.data_ptr(), k_cache.stride(0),
      k_cache.stride(1), k_cache.stride(2), block_table.data_ptr<int32_t>(), block_table.stride(0),
      cache_seqlens.data_ptr<int32_t>(), (int)seqlen_add, out.data_ptr(), o_sb, o_sh, ws, ws_bytes,
      (float)scale, (int)batch, (int)hq, (int)hkv, (int)hd, (int)ps, (int)block_table.size(1),
      (int)pages, dt == at::kBFloat16 ? MXFA_DTYPE_BF16 : MXFA_DTYPE_F16, ns, stream);
  if (rc == MXFA_EUNSUPPORTED || rc == MXFA_EINVAL) return py::none();  // nothing launched
  if (rc != MXFA_OK)
    throw std::runtime_error(std::string("mxfa_split_decode_launch failed (") +
                             std::to_string(rc) + "): " + mxfa_strerror(rc));
  return py::cast(out);
}

// Host copies of a packed call's offsets, written by the call's first (small)
// launch into pinned memory. get() waits for that launch only, not for the
// decode behind it, so the caller checks the offsets while the decode runs. The
// event releases the device's writes to the system: torch's pinned memory is
// coherent by default, but the process may ask for the other kind
// (HIP_HOST_COHERENT=0), and then nothing else shows the host these values.
// Against two blocking reads before the launch (each a copy kernel, and the GPU
// idle until the host had checked and launched), 32 packed sequences of 1k-8k
// keys, 32q/8kv HD 128, on MI355X: 157.8 -> 117.0 us a call.
class PackedOffsets {
 public:
  ~PackedOffsets() {
    if (recorded_) (void)hipEventSynchronize(event_);  // the device may still write the memory
    if (event_) (void)hipEventDestroy(event_);
  }
  // Memory and event for num_seqs sequences, or false.
  bool reserve(int64_t num_seqs) {
    if (recorded_ || event_) return false;  // one call each
    n_ = num_seqs + 1;
    values_ = at::empty({2 * n_}, at::TensorOptions().dtype(at::kLong).pinned_memory(true));
    return hipEventCreateWithFlags(&event_, hipEventDisableTiming | hipEventReleaseToSystem) ==
           hipSuccess;
  }
  int64_t *memory() {
    void *p = nullptr;
    return hipHostGetDevicePointer(&p, values_.data_ptr(), 0) == hipSuccess ? (int64_t *)p
                                                                            : nullptr;
  }
  hipEvent_t event() const { return event_; }
  void launched() { recorded_ = true; }
  // (cu_seqlens_q, cu_seqlens_k) as lists, or None when no call was launched.
  py::object get() {
    if (!recorded_) return py::none();
    hipError_t err;
    {
      py::gil_scoped_release release;
      err = hipEventSynchronize(event_);
    }
    if (err != hipSuccess)
      throw std::runtime_error(std::string("reading the offsets failed: ") +
                               hipGetErrorString(err));
    const int64_t *v = values_.data_ptr<int64_t>();
    return py::make_tuple(std::vector<int64_t>(v, v + n_), std::vector<int64_t>(v + n_, v + 2 * n_));
  }

 private:
  at::Tensor values_;
  hipEvent_t event_ = nullptr;
  int64_t n_ = 0;
  bool recorded_ = false;
};

// contiguous_decode(q, k, v, scale, causal, max_len, cu_seqlens_q,
// cu_seqlens_k, seqlens, out): decode over keys in consecutive rows, read in
// place (mxfa_package_contiguous_decode_launch).
//   dense: q [B, QL, HQ, HD], k and v [B, S, HKV, HD], every sequence max_len =
//     S keys, or seqlens (int32 [B]) of them;
//   packed (cu_seqlens_q and cu_seqlens_k given): q [B, HQ, HD], the B rows of
//     the sequences that have one, k and v [T, HKV, HD]. `offsets`, if given,
//     receives the offsets' values (PackedOffsets).
// Returns the output, or None (nothing launched) for calls whose tensors the
// kernels do not read in place.
py::object contiguous_decode(const at::Tensor &q, const at::Tensor &k, const at::Tensor &v,
                             double scale, bool causal, int64_t max_len,
                             const c10::optional<at::Tensor> &cu_q_arg,
                             const c10::optional<at::Tensor> &cu_k_arg,
                             const c10::optional<at::Tensor> &seqlens_arg,
                             const c10::optional<at::Tensor> &out_arg, PackedOffsets *offsets) {
  const bool packed = cu_q_arg.has_value();
  const int64_t rank = packed ? 3 : 4;
  const at::ScalarType dt = q.scalar_type();
  if ((dt != at::kHalf && dt != at::kBFloat16) || k.scalar_type() != dt || v.scalar_type() != dt)
    return py::none();
  if (!q.is_cuda() || q.dim() != rank || k.dim() != rank || !v.sizes().equals(k.sizes()) ||
      !v.strides().equals(k.strides()) || k.stride(-1) != 1 || q.stride(-1) != 1)
    return py::none();
  const at::Device device = q.device();
  if (k.device() != device || v.device() != device || device.index() != c10::hip::current_device())
    return py::none();
  const int64_t batch = q.size(0), ql = packed ? 1 : q.size(1);
  const int64_t hq = q.size(-2), hkv = k.size(-2), hd = q.size(-1);
  const int64_t firsts = k.size(0);
  if (batch < 1 || batch > 16000 || ql < 1 || hkv < 1 || hq % hkv || hq / hkv > 16 ||
      k.size(-1) != hd || max_len < 1 || max_len > 1 << 30 || firsts > std::numeric_limits<int>::max())
    return py::none();
  const auto vector_on_device = [&](const at::Tensor &t) {
    return t.device() == device && t.dim() == 1 && t.is_contiguous();
  };
  const void *cu_q = nullptr, *cu_k = nullptr;
  const int32_t *seqlens = nullptr;
  bool cu_q64 = false, cu_k64 = false;
  int64_t num_seqs = batch;
  if (packed) {
    if (!cu_k_arg.has_value()) return py::none();
    const at::Tensor &tq = *cu_q_arg, &tk = *cu_k_arg;
    for (const at::Tensor *t : {&tq, &tk})
      if (!vector_on_device(*t) || (t->scalar_type() != at::kInt && t->scalar_type() != at::kLong))
        return py::none();
    num_seqs = tq.numel() - 1;
    if (tk.numel() != tq.numel() || num_seqs < batch) return py::none();
    cu_q = tq.data_ptr();
    cu_k = tk.data_ptr();
    cu_q64 = tq.scalar_type() == at::kLong;
    cu_k64 = tk.scalar_type() == at::kLong;
  } else {
    if (firsts < batch || max_len > k.size(1)) return py::none();
    if (seqlens_arg.has_value()) {
      const at::Tensor &t = *seqlens_arg;
      if (!vector_on_device(t) || t.scalar_type() != at::kInt || t.numel() != batch)
        return py::none();
      seqlens = t.data_ptr<int32_t>();
    }
  }
  // q's and the output's strides (batch, token, head); a token stride of one
  // token is never used, so it need not suit the kernel.
  const auto strides = [&](const at::Tensor &t, int64_t (&s)[3]) {
    s[0] = t.stride(0);
    s[1] = ql > 1 ? t.stride(1) : 0;
    s[2] = t.stride(-2);
  };
  int64_t qs[3], os[3];
  strides(q, qs);
  if (!aligned(q.data_ptr(), 16) || ((qs[0] | qs[1] | qs[2]) & 7) || (hq > 1 && qs[2] < hd))
    return py::none();
  at::Tensor out;
  if (out_arg.has_value()) {
    out = *out_arg;
    if (out.scalar_type() != dt || out.device() != device || !out.sizes().equals(q.sizes()) ||
        out.stride(-1) != 1)
      return py::none();
    strides(out, os);
    if (!aligned(out.data_ptr(), 8) || ((os[0] | os[1] | os[2]) & 3)) return py::none();
  } else {
    out = at::empty(q.sizes(), q.options());
    strides(out, os);
  }
  // The pages that hold the same bytes (decode.py): one-token pages for packed
  // keys, for a dense cache of the largest power of two dividing its length, up
  // to 256. Splits as for those pages, or, pages of less than a tile being read
  // lane by lane there and as well as any here, as for pages of 16.
  const int64_t len = packed ? 1 : k.size(1);
  const int ps = (int)std::min<int64_t>(len & -len, 256), tile = std::max(ps, 16);
  const int width = (int)((max_len + tile - 1) / tile);
  const int wide = mxfa_package_launch_columns((int)hd, 16, 0, 0);
  int ns = 0;
  if (mxfa_package_num_splits((int)batch, (int)ql, (int)hq, (int)hkv, (int)hd, tile, width, 0, wide,
                              num_cus(device.index()), &ns) != MXFA_OK)
    return py::none();
  const int64_t tokens = mxfa_package_tokens_per_launch(
      (int)ql, (int)(hq / hkv), ns == MXFA_SPLITS_PER_SEQUENCE ? 16 : wide);
  if (tokens < ql && !causal) return py::none();
  size_t ws_bytes = 0;
  if (mxfa_package_contiguous_workspace_size((int)batch, (int)hq, (int)hkv, (int)ql, (int)hd, ns,
                                             &ws_bytes) != MXFA_OK)
    return py::none();
  void *stream = (void *)c10::hip::getCurrentHIPStream(device.index()).stream();
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing((hipStream_t)stream, &status) != hipSuccess) return py::none();
  const bool capturing = status != hipStreamCaptureStatusNone;
  int64_t *host_offsets = nullptr;
  // A capture cannot be waited for; the caller reads the offsets another way.
  if (offsets && (!packed || capturing || !offsets->reserve(num_seqs) ||
                  !(host_offsets = offsets->memory())))
    return py::none();
  at::Tensor ws_t;
  if (ws_bytes) ws_t = workspace(device, stream, ws_bytes);
  void *ws = ws_bytes ? ws_t.data_ptr() : nullptr;
  poison(stream, &out, ws_bytes ? &ws_t : nullptr);
  const at::Tensor rows_t = rows_table(device, stream, batch, capturing);
  const int64_t token_stride = k.stride(packed ? 0 : 1);
  for (int64_t t = 0; t < ql; t += tokens) {
    const int64_t n = std::min(tokens, ql - t);
    if (t > 0) poison(stream, nullptr, ws_bytes ? &ws_t : nullptr);
    // Tokens [t, t + n) as the last n tokens of sequences shortened by the
    // tokens after them.
    const int rc = mxfa_package_contiguous_decode_launch(
        (const char *)q.data_ptr() + t * qs[1] * 2, qs[0], qs[1], qs[2], (int)n, causal,
        k.data_ptr(), v.data_ptr(), k.stride(0), token_stride, k.stride(-2), firsts, (int)max_len,
        cu_q, cu_q64, cu_k, cu_k64, (int)num_seqs, rows_t.data_ptr<int32_t>(), t > 0,
        host_offsets, offsets ? offsets->event() : nullptr, seqlens, (int)(t + n - ql),
        (char *)out.data_ptr() + t * os[1] * 2, os[0], os[1], os[2], ws, ws_bytes, (float)scale,
        (int)batch, (int)hq, (int)hkv, (int)hd, ps,
        dt == at::kBFloat16 ? MXFA_DTYPE_BF16 : MXFA_DTYPE_F16, ns, stream);
    if (t == 0 && (rc == MXFA_EUNSUPPORTED || rc == MXFA_EINVAL))
      return py::none();  // nothing launched
    if (offsets) {  // one token
      if (rc != MXFA_OK) (void)hipStreamSynchronize((hipStream_t)stream);  // no event to wait for
      else offsets->launched();
    }
    if (rc != MXFA_OK)
      throw std::runtime_error(std::string("contiguous decode failed (") + std::to_string(rc) +
                               "): " + mxfa_strerror(rc));
  }
  return py::cast(out);
}

// A float32 [n] vector's address (sinks, ALiBi slopes), null for none; false
// for a tensor the kernels do not read in place.
bool head_vector(const c10::optional<at::Tensor> &t, int64_t n, const at::Device &device,
                 const float *&ptr) {
  ptr = nullptr;
  if (!t.has_value()) return true;
  if (t->scalar_type() != at::kFloat || t->device() != device || t->dim() != 1 ||
      t->size(0) != n || !t->is_contiguous())
    return false;
  ptr = t->data_ptr<float>();
  return true;
}

// A per-tensor scale's address (one float32, or one broadcast), null for none.
bool tensor_scale(const c10::optional<at::Tensor> &t, const at::Device &device,
                  const float *&ptr) {
  ptr = nullptr;
  if (!t.has_value()) return true;
  if (t->scalar_type() != at::kFloat || t->device() != device || t->numel() < 1) return false;
  if (t->numel() != 1)
    for (const int64_t st : t->strides())
      if (st != 0) return false;
  ptr = t->data_ptr<float>();
  return true;
}

// decode_tokens(q, k_cache, v_cache, block_table, cache_seqlens, scale, out,
// num_splits, seqlen_add, causal, window_left, softcap, k_scale, v_scale, sinks,
// alibi_slopes): the general paged call (several query tokens, fp8 caches,
// window, soft cap, sinks, ALiBi) with tensors the kernels read in place; a
// causal query of more columns than one launch takes runs as several.
// cache_seqlens moves on by `advance` once it has been read. Returns
// the output, or None (nothing launched) for any other call, which the Python
// binding then takes.
py::object decode_tokens(const at::Tensor &q, const at::Tensor &k_cache, const at::Tensor &v_cache,
                         const at::Tensor &block_table, const at::Tensor &cache_seqlens,
                         double scale, const c10::optional<at::Tensor> &out_arg,
                         const c10::optional<int64_t> &num_splits_arg, int64_t seqlen_add,
                         bool causal, int64_t window_left, double softcap,
                         const c10::optional<at::Tensor> &k_scale,
                         const c10::optional<at::Tensor> &v_scale,
                         const c10::optional<at::Tensor> &sinks,
                         const c10::optional<at::Tensor> &alibi_slopes, int64_t advance) {
  const at::ScalarType dt = q.scalar_type();
  const bool fp8 = k_cache.scalar_type() == at::kFloat8_e4m3fn;
  if ((dt != at::kHalf && dt != at::kBFloat16) || (!fp8 && k_cache.scalar_type() != dt) ||
      v_cache.scalar_type() != k_cache.scalar_type())
    return py::none();
  if (!q.is_cuda() || (q.dim() != 3 && q.dim() != 4) || q.stride(-1) != 1) return py::none();
  if (k_cache.dim() != 4 || !v_cache.sizes().equals(k_cache.sizes()) ||
      !v_cache.strides().equals(k_cache.strides()) || k_cache.stride(3) != 1)
    return py::none();
  if (block_table.scalar_type() != at::kInt || cache_seqlens.scalar_type() != at::kInt ||
      block_table.dim() != 2 || block_table.stride(1) != 1 || cache_seqlens.dim() != 1 ||
      !cache_seqlens.is_contiguous())
    return py::none();
  const at::Device device = q.device();
  if (k_cache.device() != device || v_cache.device() != device ||
      block_table.device() != device || cache_seqlens.device() != device ||
      device.index() != c10::hip::current_device())
    return py::none();
  const int64_t batch = q.size(0), ql = q.dim() == 4 ? q.size(1) : 1;
  const int64_t hq = q.size(-2), hd = q.size(-1);
  const int64_t pages = k_cache.size(0), ps = k_cache.size(1), hkv = k_cache.size(2);
  if (batch < 1 || ql < 1 || hkv < 1 || ps < 1 || hq % hkv || hq / hkv > 16 || hq < hkv ||
      k_cache.size(3) != hd || block_table.size(0) != batch || cache_seqlens.size(0) != batch ||
      block_table.size(1) < 1)
    return py::none();
  const int64_t limit = std::numeric_limits<int>::max() / 64;
  if (batch > limit || hq > limit || ql > limit || pages > std::numeric_limits<int>::max() ||
      ps > 4096 || block_table.size(1) > std::numeric_limits<int>::max())
    return py::none();
  const int64_t gq = hq / hkv;
  if ((ql * gq > 16 && !causal) || window_left < -1 || window_left > 1 << 30 ||
      !(softcap >= 0.0) || softcap == std::numeric_limits<double>::infinity())
    return py::none();
  if (advance < 0 || advance > 1 << 30) return py::none();
  if (seqlen_add < -(1 << 29) || seqlen_add > 1 << 30) return py::none();
  const float *ks, *vs, *sink_ptr, *alibi_ptr;
  if (!head_vector(sinks, hq, device, sink_ptr) || !head_vector(alibi_slopes, hq, device, alibi_ptr))
    return py::none();
  if (!tensor_scale(fp8 ? k_scale : c10::nullopt, device, ks) ||
      !tensor_scale(fp8 ? v_scale : c10::nullopt, device, vs))
    return py::none();
  // Strides (batch, token, head); the token stride of one token is not used.
  const auto strides = [&](const at::Tensor &t, int64_t (&s)[3]) {
    s[0] = t.stride(0);
    s[1] = ql > 1 ? t.stride(1) : 0;
    s[2] = t.stride(-2);
  };
  int64_t qs[3], os[3];
  strides(q, qs);
  if (!aligned(q.data_ptr(), 16) || ((qs[0] | qs[1] | qs[2]) & 7) || (hq > 1 && qs[2] < hd))
    return py::none();
  at::Tensor out;
  if (out_arg.has_value()) {
    out = *out_arg;
    if (out.scalar_type() != dt || out.device() != device || !out.sizes().equals(q.sizes()) ||
        out.stride(-1) != 1 || at::has_internal_overlap(out) == at::MemOverlap::Yes)
      return py::none();
    strides(out, os);
    if (!aligned(out.data_ptr(), 8) || ((os[0] | os[1] | os[2]) & 3)) return py::none();
  } else {
    out = at::empty(q.sizes(), q.options());
    strides(out, os);
  }
  const bool extras = window_left >= 0 || softcap > 0 || sink_ptr || alibi_ptr;
  // Only the entry point of several tokens or options takes shortened sequences;
  // one plain token is refused by the C ABI (mxfa_split_decode_launch).
  if (seqlen_add < 0 && ql == 1 && !extras) return py::none();
  const int width = (int)block_table.size(1);
  const int wide = mxfa_package_launch_columns((int)hd, (int)ps, fp8, extras);
  int ns = 0;
  if (num_splits_arg.has_value()) {
    const int64_t v = *num_splits_arg;
    if ((v <= 0 && v != MXFA_SPLITS_PER_SEQUENCE) || v > 65535) return py::none();
    ns = (int)v;
  } else if (mxfa_package_num_splits((int)batch, (int)ql, (int)hq, (int)hkv, (int)hd, (int)ps,
                                     width, fp8, wide, num_cus(device.index()), &ns) !=
             MXFA_OK) {
    return py::none();
  }
  const int64_t tokens = mxfa_package_tokens_per_launch(
      (int)ql, (int)gq, ns == MXFA_SPLITS_PER_SEQUENCE ? 16 : wide);
  size_t ws_bytes = 0;
  if (mxfa_split_decode_workspace_size((int)batch, (int)(hq * tokens), (int)hd, ns, &ws_bytes) !=
      MXFA_OK)
    return py::none();
  void *stream = (void *)c10::hip::getCurrentHIPStream(device.index()).stream();
  at::Tensor ws_t;
  if (ws_bytes) ws_t = workspace(device, stream, ws_bytes);
  void *ws = ws_bytes ? ws_t.data_ptr() : nullptr;
  poison(stream, &out, ws_bytes ? &ws_t : nullptr);
  const int64_t esz = 2;
  for (int64_t t = 0; t < ql; t += tokens) {
    const int64_t n = std::min(tokens, ql - t);
    if (t > 0) poison(stream, nullptr, ws_bytes ? &ws_t : nullptr);
    // Tokens [t, t + n) as the last n tokens of sequences shortened by the
    // tokens after them.
    const int rc = mxfa_package_decode_tokens_launch(
        (const char *)q.data_ptr() + t * qs[1] * esz, qs[0], qs[1], qs[2], (int)n, causal,
        (int)window_left, sink_ptr, (float)softcap, alibi_ptr, k_cache.data_ptr(),
        v_cache.data_ptr(), k_cache.stride(0), k_cache.stride(1), k_cache.stride(2),
        block_table.data_ptr<int32_t>(), block_table.stride(0),
        cache_seqlens.data_ptr<int32_t>(), (int)(seqlen_add - (ql - t - n)),
        (char *)out.data_ptr() + t * os[1] * esz, os[0], os[1], os[2], ws, ws_bytes, (float)scale,
        (int)batch, (int)hq, (int)hkv, (int)hd, (int)ps, width, (int)pages,
        dt == at::kBFloat16 ? MXFA_DTYPE_BF16 : MXFA_DTYPE_F16,
        fp8                  ? MXFA_DTYPE_FP8_E4M3
        : dt == at::kBFloat16 ? MXFA_DTYPE_BF16
                              : MXFA_DTYPE_F16,
        ks, vs, ns, advance && t + n == ql ? cache_seqlens.data_ptr<int32_t>() : nullptr,
        (int)advance, stream);
    if (t == 0 && (rc == MXFA_EUNSUPPORTED || rc == MXFA_EINVAL))
      return py::none();  // nothing launched
    if (rc != MXFA_OK)
      throw std::runtime_error(std::string("mxfa_split_decode_multi_launch failed (") +
                               std::to_string(rc) + "): " + mxfa_strerror(rc));
  }
  return py::cast(out);
}

// Source rows K and V (of `rank` dims) sharing strides with a contiguous last
// dim, and paged caches sharing theirs, all on the current GPU; cache_dt the
// caches' type.
bool append_tensors(const at::Tensor &key, const at::Tensor &value, const at::Tensor &key_cache,
                    const at::Tensor &value_cache, int64_t rank, at::ScalarType cache_dt) {
  const at::ScalarType dt = key.scalar_type();
  if ((dt != at::kHalf && dt != at::kBFloat16) || !key.is_cuda() || value.scalar_type() != dt ||
      key_cache.scalar_type() != cache_dt || value_cache.scalar_type() != cache_dt)
    return false;
  if (key.dim() != rank || !value.sizes().equals(key.sizes()) ||
      !value.strides().equals(key.strides()) || key.stride(-1) != 1)
    return false;
  if (key_cache.dim() != 4 || !value_cache.sizes().equals(key_cache.sizes()) ||
      !value_cache.strides().equals(key_cache.strides()) || key_cache.stride(3) != 1)
    return false;
  if (key.size(-2) != key_cache.size(2) || key.size(-1) != key_cache.size(3)) return false;
  const at::Device device = key.device();
  return value.device() == device && key_cache.device() == device &&
         value_cache.device() == device && device.index() == c10::hip::current_device();
}

// reshape_and_cache(key, value, key_cache, value_cache, slot_mapping, k_scale,
// v_scale): the vLLM-form append, 16-bit (mxfa_reshape_and_cache_launch) or
// into fp8 caches (mxfa_reshape_and_cache_fp8_launch), for the common call:
// key/value [T, HKV, HD], caches [pages, PS, HKV, HD], int64 contiguous slots
// (at least T of them), scales None or float32 device tensors.
// Returns true once launched on torch's current stream; false (nothing
// launched) for any other call, which the Python binding then takes.
bool reshape_and_cache(const at::Tensor &key, const at::Tensor &value,
                       const at::Tensor &key_cache, const at::Tensor &value_cache,
                       const at::Tensor &slot_mapping, const c10::optional<at::Tensor> &k_scale,
                       const c10::optional<at::Tensor> &v_scale) {
  const at::ScalarType dt = key.scalar_type();
  const bool fp8 = key_cache.scalar_type() == at::kFloat8_e4m3fn;
  if (!append_tensors(key, value, key_cache, value_cache, 3, fp8 ? at::kFloat8_e4m3fn : dt))
    return false;
  const at::Device device = key.device();
  if (slot_mapping.scalar_type() != at::kLong || slot_mapping.dim() != 1 ||
      !slot_mapping.is_contiguous() || slot_mapping.size(0) < key.size(0) ||
      slot_mapping.device() != device)
    return false;
  const float *ks, *vs;
  if (!tensor_scale(fp8 ? k_scale : c10::nullopt, device, ks) ||
      !tensor_scale(fp8 ? v_scale : c10::nullopt, device, vs))
    return false;
  void *stream = (void *)c10::hip::getCurrentHIPStream(device.index()).stream();
  const int code = dt == at::kBFloat16 ? MXFA_DTYPE_BF16 : MXFA_DTYPE_F16;
  const int rc =
      fp8 ? mxfa_reshape_and_cache_fp8_launch(
                key.data_ptr(), value.data_ptr(), key.stride(0), key.stride(1),
                key_cache.data_ptr(), value_cache.data_ptr(), key_cache.stride(0),
                key_cache.stride(1), key_cache.stride(2), slot_mapping.data_ptr<int64_t>(),
                (int)key.size(0), (int)key.size(1), (int)key.size(2), (int)key_cache.size(1),
                (int)key_cache.size(0), code, ks, vs, stream)
          : mxfa_reshape_and_cache_launch(
                key.data_ptr(), value.data_ptr(), key.stride(0), key.stride(1),
                key_cache.data_ptr(), value_cache.data_ptr(), key_cache.stride(0),
                key_cache.stride(1), key_cache.stride(2), slot_mapping.data_ptr<int64_t>(),
                (int)key.size(0), (int)key.size(1), (int)key.size(2), (int)key_cache.size(1),
                (int)key_cache.size(0), code, stream);
  if (rc == MXFA_EUNSUPPORTED || rc == MXFA_EINVAL) return false;  // nothing launched
  if (rc != MXFA_OK)
    throw std::runtime_error(std::string("mxfa_reshape_and_cache_launch failed (") +
                             std::to_string(rc) + "): " + mxfa_strerror(rc));
  return true;
}

// append_kv(k, v, k_cache, v_cache, block_table, cache_seqlens): the table-form
// append (mxfa_append_kv_launch) of 16-bit rows [B, S, HKV, HD], int32 table and
// lengths. True once launched, false (nothing launched) for any other call.
bool append_kv(const at::Tensor &k, const at::Tensor &v, const at::Tensor &k_cache,
               const at::Tensor &v_cache, const at::Tensor &block_table,
               const at::Tensor &cache_seqlens) {
  if (!append_tensors(k, v, k_cache, v_cache, 4, k.scalar_type())) return false;
  const at::Device device = k.device();
  if (block_table.scalar_type() != at::kInt || cache_seqlens.scalar_type() != at::kInt ||
      block_table.dim() != 2 || block_table.stride(1) != 1 || cache_seqlens.dim() != 1 ||
      !cache_seqlens.is_contiguous() || block_table.device() != device ||
      cache_seqlens.device() != device || block_table.size(0) != k.size(0) ||
      block_table.size(1) < 1 || cache_seqlens.size(0) != k.size(0))
    return false;
  void *stream = (void *)c10::hip::getCurrentHIPStream(device.index()).stream();
  const int rc = mxfa_append_kv_launch(
      k.data_ptr(), v.data_ptr(), k.stride(0), k.stride(1), k.stride(2), k_cache.data_ptr(),
      v_cache.data_ptr(), k_cache.stride(0), k_cache.stride(1), k_cache.stride(2),
      block_table.data_ptr<int32_t>(), block_table.stride(0), cache_seqlens.data_ptr<int32_t>(),
      (int)k.size(0), (int)k.size(1), (int)k.size(2), (int)k.size(3), (int)k_cache.size(1),
      (int)block_table.size(1), (int)k_cache.size(0),
      k.scalar_type() == at::kBFloat16 ? MXFA_DTYPE_BF16 : MXFA_DTYPE_F16, stream);
  if (rc == MXFA_EUNSUPPORTED || rc == MXFA_EINVAL) return false;  // nothing launched
  if (rc != MXFA_OK)
    throw std::runtime_error(std::string("mxfa_append_kv_launch failed (") + std::to_string(rc) +
                             "): " + mxfa_strerror(rc));
  return true;
}

}  // namespace

PYBIND11_MODULE(_mxfa_torch, m) {
  m.doc() = "torch operator in front of libmxfa_mi355x's split decode C ABI";
  py::class_<PackedOffsets>(m, "PackedOffsets").def(py::init<>()).def("get", &PackedOffsets::get);
  m.def("decode", &decode, py::arg("q"), py::arg("k_cache"), py::arg("v_cache"),
        py::arg("block_table"), py::arg("cache_seqlens"), py::arg("scale"),
        py::arg("out") = py::none(), py::arg("num_splits") = py::none(),
        py::arg("seqlen_add") = 0);
  m.def("contiguous_decode", &contiguous_decode, py::arg("q"), py::arg("k"), py::arg("v"),
        py::arg("scale"), py::arg("causal"), py::arg("max_len"),
        py::arg("cu_seqlens_q") = py::none(), py::arg("cu_seqlens_k") = py::none(),
        py::arg("seqlens") = py::none(), py::arg("out") = py::none(),
        py::arg("offsets") = py::none());
  m.def("decode_tokens", &decode_tokens, py::arg("q"), py::arg("k_cache"), py::arg("v_cache"),
        py::arg("block_table"), py::arg("cache_seqlens"), py::arg("scale"), py::arg("out"),
        py::arg("num_splits"), py::arg("seqlen_add"), py::arg("causal"), py::arg("window_left"),
        py::arg("softcap"), py::arg("k_scale"), py::arg("v_scale"), py::arg("sinks"),
        py::arg("alibi_slopes"), py::arg("advance") = 0);
  // The call without scales by itself: two optional arguments cost a small
  // append 0.1 us of its 4.1 us.
  m.def("reshape_and_cache",
        [](const at::Tensor &key, const at::Tensor &value, const at::Tensor &key_cache,
           const at::Tensor &value_cache, const at::Tensor &slot_mapping) {
          return reshape_and_cache(key, value, key_cache, value_cache, slot_mapping, c10::nullopt,
                                   c10::nullopt);
        },
        py::arg("key"), py::arg("value"), py::arg("key_cache"), py::arg("value_cache"),
        py::arg("slot_mapping"));
  m.def("reshape_and_cache_scaled", &reshape_and_cache, py::arg("key"), py::arg("value"),
        py::arg("key_cache"), py::arg("value_cache"), py::arg("slot_mapping"),
        py::arg("k_scale"), py::arg("v_scale"));
  m.def("append_kv", &append_kv, py::arg("k"), py::arg("v"), py::arg("k_cache"),
        py::arg("v_cache"), py::arg("block_table"), py::arg("cache_seqlens"));
  m.def("abi_version", &mxfa_abi_version);
  m.def("workspace_bytes", &workspace_bytes,
        "(bytes of live workspaces, bytes of workspaces replaced by larger ones)");
}
