// Compiled PyTorch-ROCm operator layer over the C ABI of libsdk_mapped_ops.so.
//
// Registers, for the CUDA (= HIP on ROCm) dispatch key, the operators of the `sdk_mapped_ops`
// namespace whose per-call cost matters: each checks its tensors the way the reference's
// pybind entry points do (contiguous, all on the GPU: ext_modules/include/cuda_helper.h:12-18;
// ext_modules/include/layers/mapped_convolution_layer.h:62-143 is the shape of such an entry
// point), allocates the outputs, fetches the current HIP stream, looks up or builds the plan of
// the map and makes one call into the C ABI.  The schemas are defined from Python
// (_spherical_distortion_ext/_ops.py), which loads this library when it is built and registers
// its own implementations of the same operators when it is not; both keep the same plan cache
// rules: keyed on the map's storage, offset, version counter, shape and the geometry; least
// recently used entry dropped first; maps without a version counter (inference tensors) and
// keys that miss during a stream capture go to the entry points that build what they need
// inside the call.
//
// Built with the host compiler against the torch headers; no device code here.
#include <ATen/ATen.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>
#include <torch/library.h>

#include <algorithm>
#include <cstdint>
#include <iterator>
#include <list>
#include <mutex>
#include <string>
#include <utility>
#include <vector>

#include "sdk_mapped_ops.h"

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;

// ----------------------------------------------------------------------------- state
std::mutex g_mu;
int g_default_mode = SDK_COMPUTE_NATIVE;
thread_local int t_mode = -1;   // -1: no override on this thread
bool g_cache_enabled = true;
size_t g_cache_max = 16;
bool g_unpool_workspace = true;

int current_mode() { return t_mode >= 0 ? t_mode : g_default_mode; }

struct TensorKey {
  bool present = false;
  const void* storage = nullptr;
  int64_t offset = 0, version = 0;
  std::vector<int64_t> shape;
  bool operator==(const TensorKey& o) const {
    return present == o.present && storage == o.storage && offset == o.offset &&
           version == o.version && shape == o.shape;
  }
};

// false: the tensor's changes cannot be tracked (no version counter)
bool tensor_key(const OptTensor& t, TensorKey* k) {
  if (!t.has_value() || !t->defined()) return true;
  if (t->is_inference()) return false;
  k->present = true;
  k->storage = t->storage().data();
  k->offset = t->storage_offset();
  k->version = (int64_t)t->_version();
  k->shape = t->sizes().vec();
  return true;
}

enum Kind { kConv = 0, kResample = 1, kAvgUnpool = 2, kMaxUnpool = 3, kAvgUnpoolLists = 4,
            kUvScatter = 5 };

struct Key {
  int kind = 0, device = 0, dtype = 0;
  TensorKey map, wts;
  int64_t a = 0, b = 0, K = 0, P = 0, interp = 0;
  bool operator==(const Key& o) const {
    return kind == o.kind && device == o.device && dtype == o.dtype && map == o.map &&
           wts == o.wts && a == o.a && b == o.b && K == o.K && P == o.P && interp == o.interp;
  }
};

struct Buffer {
  Tensor plan;
  size_t nbytes = 0;
  int built = 0;   // parts of the buffer that are filled (each by the first call that reads it)
};
// kSide: the inverted map that convolutions by columns read (much smaller than the plan of the others
// on the same map).
enum Slot { kMain = 0, kSide = 1 };

struct Entry {
  Key key;
  Buffer buffers[2];   // by Slot, each made by the first call that reads it
  c10::Storage keep_map, keep_wts;   // an address cannot be reused while its entry lives
  hipStream_t stream = nullptr;      // last user: a call on another stream is ordered behind it
  int complete = 0;
  bool captured = false;             // a graph reads the plan
};
// Most recently used last.  Never destroyed: at the process's end the GPU runtime may be gone before this
// library's statics, and freeing a plan that several streams used (an event is recorded for each)
// then throws, which aborts the process.
std::list<Entry>& g_cache = *new std::list<Entry>;

// Lets go of the least recently used entries until `most` are left.  A plan that a captured graph reads
// by its address stays as long as anyone beside the cache holds its map (the graph's owner has to).
void shrink_cache(size_t most) {
  for (auto it = g_cache.begin(); g_cache.size() > most && it != g_cache.end();)
    it = it->captured && it->keep_map.use_count() > 1 ? std::next(it) : g_cache.erase(it);
}

struct PlanRef {
  Tensor plan;   // undefined: none
  size_t nbytes = 0;
  int complete = 0;
  void* ptr() const { return plan.defined() ? plan.data_ptr() : nullptr; }
};

void order_behind(hipStream_t cur, hipStream_t last) {
  hipEvent_t ev = nullptr;
  if (hipEventCreateWithFlags(&ev, hipEventDisableTiming) != hipSuccess) return;
  if (hipEventRecord(ev, last) == hipSuccess) (void)hipStreamWaitEvent(cur, ev, 0);
  (void)hipEventDestroy(ev);
}

bool capturing(hipStream_t s) {
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &st) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return st != hipStreamCaptureStatusNone;
}

void fail_call(const char* name, int rc) {
  TORCH_CHECK(false, name, " failed (status ", rc, "): ", sdk_last_error());
}
#define SDK_CALL(name, ...)              \
  do {                                   \
    const int rc__ = name(__VA_ARGS__);  \
    if (rc__ != 0) fail_call(#name, rc__); \
  } while (0)

const void* cptr(const OptTensor& t) {
  return (t.has_value() && t->defined()) ? t->data_ptr() : nullptr;
}

int dtype_code(const Tensor& ref) {
  if (ref.scalar_type() == at::kFloat) return SDK_F32;
  if (ref.scalar_type() == at::kDouble) return SDK_F64;
  TORCH_CHECK(false, "unsupported dtype ", ref.scalar_type(), " (float32 and float64 only)");
}

void check_first(const Tensor& ref) {
  TORCH_CHECK(ref.is_cuda(), "this backend runs on the GPU only: tensors must be CUDA/HIP tensors");
  (void)dtype_code(ref);
}
void check_one(const Tensor& ref, const char* name, const Tensor& t, bool any_dtype = false) {
  TORCH_CHECK(t.is_contiguous(), name, " must be contiguous");
  TORCH_CHECK(t.is_cuda() && t.device() == ref.device(), name, " must be a CUDA tensor on ",
              ref.device());
  TORCH_CHECK(any_dtype || t.scalar_type() == ref.scalar_type(), name, " must have dtype ",
              ref.scalar_type(), " (got ", t.scalar_type(), ")");
}
void check_opt(const Tensor& ref, const char* name, const OptTensor& t) {
  if (t.has_value() && t->defined()) check_one(ref, name, *t);
}

// 0 for the unweighted map layout, P for the weighted one.
int64_t npts(const Tensor& map, const OptTensor& w, int64_t rank_unweighted) {
  if (!w.has_value() || !w->defined()) {
    TORCH_CHECK(map.dim() == rank_unweighted && map.size(-1) == 2, "sample_map must have ",
                rank_unweighted, " dimensions ending in 2, got ", map.sizes());
    return 0;
  }
  TORCH_CHECK(map.dim() == rank_unweighted + 1 && map.size(-1) == 2,
              "weighted sample_map must have ", rank_unweighted + 1,
              " dimensions ending in 2, got ", map.sizes());
  TORCH_CHECK(w->sizes() == map.sizes().slice(0, map.dim() - 1), "interp_weights shape ",
              w->sizes(), " does not match sample_map ", map.sizes());
  return w->size(-1);
}

hipStream_t stream_of(const Tensor& ref) {
  return c10::hip::getCurrentHIPStream(ref.device().index()).stream();
}

Tensor bytes_on(const Tensor& ref, size_t n) {
  return at::empty({(int64_t)n}, ref.options().dtype(at::kByte));
}

// The kept plan of `key`, or one built by `build` (which returns the plan's size, 0 for none,
// and fills the buffer it is handed on `stream`).  needed: the parts of the plan (bits) that this call
// reads; build fills the parts it is asked for.  A call that reads none leaves the cache as it is: an
// entry for it would hold nothing but its map, and push out a plan.
template <typename Size, typename Build>
PlanRef plan_for(Key key, const Tensor& ref, const Tensor& map, const OptTensor& wts,
                 hipStream_t stream, Size size, Build build, int needed = 1, Slot slot = kMain) {
  PlanRef out;
  if (!g_cache_enabled || needed == 0) return out;
  if (!tensor_key(map, &key.map) || !tensor_key(wts, &key.wts)) return out;
  std::lock_guard<std::mutex> lock(g_mu);
  for (auto it = g_cache.begin(); it != g_cache.end(); ++it) {
    if (!(it->key == key)) continue;
    g_cache.splice(g_cache.end(), g_cache, it);   // most recently used
    Entry& e = g_cache.back();
    Buffer& buf = e.buffers[slot];
    const int missing = needed & ~buf.built;
    const bool captured = capturing(stream);
    if (missing != 0) {
      if (captured) return out;
      if (!buf.plan.defined()) {
        buf.nbytes = size();
        if (buf.nbytes == 0) return out;
        buf.plan = bytes_on(ref, buf.nbytes);
      }
    }
    if (stream != e.stream) {
      order_behind(stream, e.stream);
      e.stream = stream;
      // once let go, the buffers' memory waits for the calls of this stream too
      const auto here = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(ref.device().index());
      for (Buffer& b : e.buffers)
        if (b.plan.defined()) b.plan.record_stream(here.unwrap());
    }
    if (missing != 0) {
      e.complete = build(buf.plan.data_ptr(), buf.nbytes, missing);
      buf.built |= missing;
    }
    e.captured |= captured;
    out.plan = buf.plan;
    out.nbytes = buf.nbytes;
    out.complete = e.complete;
    return out;
  }
  if (capturing(stream)) return out;
  const size_t n = size();
  if (n == 0) return out;
  Entry e;
  e.key = key;
  Buffer& buf = e.buffers[slot];
  buf.nbytes = n;
  buf.plan = bytes_on(ref, n);
  e.complete = build(buf.plan.data_ptr(), n, needed);
  buf.built = needed;
  e.keep_map = map.storage();
  if (wts.has_value() && wts->defined()) e.keep_wts = wts->storage();
  e.stream = stream;
  out.plan = buf.plan;
  out.nbytes = n;
  out.complete = e.complete;
  shrink_cache(g_cache_max - 1);
  g_cache.push_back(std::move(e));
  return out;
}

struct ConvDims {
  int64_t B, Cin, Cout, K;
};

// The plan of a (transposed) convolution call.  gather: the call samples the image (the forward of
// a convolution, the backward-input of a transposed one); weights: it forms a weight gradient;
// scatter: it splats into the image (the other two).  Each reads its part of the plan, a layer
// of a few image channels none; of the calls that run as columns and products only scatters
// read one, the inverted map.  A forward whose input requires a gradient asks for what the input's
// gradient reads too: a backward captured into a graph after it finds its plan whole, where
// nothing could be built.  (Measured, first step on a new map, all parts of a plan built ->
// those that are read: 4 x 512 x 1024, 3 -> 32 channels, no picture gradient 694 -> 342 us,
// 64 x 128, 3 -> 16 547 -> 175 us.)
PlanRef conv_plan(const Tensor& ref, const Tensor& map, const OptTensor& wts, const ConvDims& d,
                  int64_t img_h, int64_t img_w, int64_t P, int64_t interp, bool transposed,
                  bool gather, bool weights, bool scatter, hipStream_t stream) {
  if (ref.scalar_type() != at::kFloat) return PlanRef();
  const int64_t MH = map.size(0), MW = map.size(1), K = d.K;
  const bool columns =
      sdk_mapped_conv_by_columns(d.B, d.Cin, d.Cout, img_h, img_w, MH, MW, K, (int32_t)P,
                                 (int32_t)interp, SDK_F32, current_mode(), transposed ? 1 : 0) == 1;
  Key key;
  key.kind = kConv;
  key.device = ref.device().index();
  key.a = img_h;
  key.b = img_w;
  key.K = K;
  key.P = P;
  key.interp = interp;
  return plan_for(
      key, ref, map, wts, stream,
      [&] {
        return columns ? sdk_mapped_conv_columns_bytes(img_h, img_w, MH, MW, K, (int32_t)P,
                                                       (int32_t)interp, SDK_F32)
                       : sdk_mapped_conv_plan_bytes(img_h, img_w, MH, MW, K, (int32_t)P,
                                                    (int32_t)interp, SDK_F32);
      },
      [&](void* buf, size_t n, int parts) {
        if (columns)
          SDK_CALL(sdk_mapped_conv_plan_build_columns, map.data_ptr(), cptr(wts), buf, n, img_h,
                   img_w, MH, MW, K, (int32_t)P, (int32_t)interp, SDK_F32, stream);
        else
          SDK_CALL(sdk_mapped_conv_plan_build_parts, map.data_ptr(), cptr(wts), buf, n, img_h, img_w,
                   MH, MW, K, (int32_t)P, (int32_t)interp, SDK_F32, parts, stream);
        return 0;
      },
      columns ? (scatter ? 1 : 0)
              : sdk_mapped_conv_plan_parts(d.B, d.Cin, d.Cout, img_h, img_w, MH, MW, K, (int32_t)P,
                                           (int32_t)interp, SDK_F32, current_mode(),
                                           transposed ? 1 : 0, gather, weights, scatter),
      columns ? kSide : kMain);
}

PlanRef scatter_plan(Kind kind, const Tensor& ref, const Tensor& map, const OptTensor& wts,
                     int64_t out_h, int64_t out_w, int64_t K, int64_t P, int64_t interp,
                     hipStream_t stream) {
  const int dt = dtype_code(ref);
  const int64_t MH = map.size(0), MW = map.size(1);
  Key key;
  key.kind = kind;
  key.device = ref.device().index();
  key.dtype = dt;
  key.a = out_h;
  key.b = out_w;
  key.K = K;
  key.P = P;
  key.interp = interp;
  return plan_for(
      key, ref, map, wts, stream,
      [&] {
        if (kind == kAvgUnpoolLists)
          return sdk_mapped_avg_unpool_lists_bytes(out_h, out_w, MH, MW, K, (int32_t)P,
                                                   (int32_t)interp, dt);
        return kind == kMaxUnpool ? sdk_mapped_max_unpool_workspace_bytes(out_h, out_w, dt)
                                  : sdk_resample_to_map_workspace_bytes(out_h, out_w, dt);
      },
      [&](void* buf, size_t n, int) {
        if (kind == kAvgUnpoolLists) {
          SDK_CALL(sdk_mapped_avg_unpool_lists_build, map.data_ptr(), cptr(wts), buf, n, out_h,
                   out_w, MH, MW, K, (int32_t)P, (int32_t)interp, dt, stream);
          return 1;
        }
        if (kind == kMaxUnpool) {
          SDK_CALL(sdk_mapped_max_unpool_plan_build, map.data_ptr(), buf, n, out_h, out_w, MH, MW,
                   K, (int32_t)P, (int32_t)interp, dt, stream);
          int32_t bands = 0;
          SDK_CALL(sdk_mapped_max_unpool_plan_bands, buf, n, out_h, out_w, dt, stream, &bands);
          return (int)bands;
        }
        SDK_CALL(sdk_resample_to_map_plan_build, map.data_ptr(), cptr(wts), buf, n, MH, MW, out_h,
                 out_w, K, (int32_t)P, (int32_t)interp, dt, stream);
        int32_t flag = 0;
        SDK_CALL(sdk_resample_plan_complete, buf, n, stream, &flag);
        return (int)flag;
      });
}

// ----------------------------------------------------------------------------- resample
Tensor resample_from_map(const Tensor& x, const Tensor& map, const OptTensor& wts, int64_t interp) {
  check_first(x);
  check_one(x, "x", x);
  check_one(x, "sample_map", map);
  check_opt(x, "interp_weights", wts);
  const int64_t P = npts(map, wts, 3);
  TORCH_CHECK(x.dim() == 4, "x must be [B, C, H, W]");
  const int64_t B = x.size(0), C = x.size(1), H = x.size(2), W = x.size(3);
  const int64_t MH = map.size(0), MW = map.size(1);
  Tensor out = at::empty({B, C, MH, MW}, x.options());
  c10::DeviceGuard guard(x.device());
  SDK_CALL(sdk_resample_from_map, x.data_ptr(), map.data_ptr(), cptr(wts), out.data_ptr(), B, C, H,
           W, MH, MW, (int32_t)P, (int32_t)interp, dtype_code(x), stream_of(x));
  return out;
}

std::tuple<Tensor, Tensor> resample_to_map_impl(const Tensor& x, const Tensor& map,
                                                const OptTensor& wts, int64_t out_h,
                                                int64_t out_w, int64_t interp, bool normalize,
                                                double eps) {
  check_first(x);
  check_one(x, "x", x);
  check_one(x, "sample_map", map);
  check_opt(x, "interp_weights", wts);
  const int64_t P = npts(map, wts, 3);
  TORCH_CHECK(x.dim() == 4, "x must be [B, C, MH, MW]");
  const int64_t B = x.size(0), C = x.size(1), MH = x.size(2), MW = x.size(3);
  TORCH_CHECK(map.size(0) == MH && map.size(1) == MW, "sample_map grid ",
              map.sizes().slice(0, 2), " must match the input's ", x.sizes().slice(2));
  const int dt = dtype_code(x);
  Tensor out = at::empty({B, C, out_h, out_w}, x.options());
  Tensor wsum;
  if (normalize) wsum = at::empty({out_h, out_w}, x.options());
  c10::DeviceGuard guard(x.device());
  hipStream_t s = stream_of(x);
  PlanRef plan = scatter_plan(kResample, x, map, wts, out_h, out_w, 1, P, interp, s);
  if (plan.plan.defined()) {
    SDK_CALL(sdk_resample_to_map_planned, x.data_ptr(), map.data_ptr(), cptr(wts), out.data_ptr(),
             normalize ? wsum.data_ptr() : nullptr, plan.ptr(), plan.nbytes, plan.complete,
             normalize ? 1 : 0, eps, B, C, MH, MW, out_h, out_w, (int32_t)P, (int32_t)interp, dt, s);
    return {out, wsum};
  }
  const size_t nws = sdk_resample_to_map_workspace_bytes(out_h, out_w, dt);
  Tensor ws;
  if (nws) ws = bytes_on(x, nws);
  if (normalize)
    SDK_CALL(sdk_resample_to_map_normalized, x.data_ptr(), map.data_ptr(), cptr(wts),
             out.data_ptr(), wsum.data_ptr(), nws ? ws.data_ptr() : nullptr, nws, eps, B, C, MH, MW,
             out_h, out_w, (int32_t)P, (int32_t)interp, dt, s);
  else
    SDK_CALL(sdk_resample_to_map, x.data_ptr(), map.data_ptr(), cptr(wts), out.data_ptr(), nullptr,
             nws ? ws.data_ptr() : nullptr, nws, B, C, MH, MW, out_h, out_w, (int32_t)P,
             (int32_t)interp, dt, s);
  return {out, wsum};
}

Tensor resample_to_map(const Tensor& x, const Tensor& map, const OptTensor& wts, int64_t out_h,
                       int64_t out_w, int64_t interp) {
  return std::get<0>(resample_to_map_impl(x, map, wts, out_h, out_w, interp, false, 0.0));
}
std::tuple<Tensor, Tensor> resample_to_map_normalized(const Tensor& x, const Tensor& map,
                                                      const OptTensor& wts, int64_t out_h,
                                                      int64_t out_w, int64_t interp, double eps) {
  return resample_to_map_impl(x, map, wts, out_h, out_w, interp, true, eps);
}

// ----------------------------------------------------------------------------- pooling
void check_kernel(const Tensor& map, int64_t kernel_size) {
  TORCH_CHECK(map.dim() >= 3 && map.size(2) == kernel_size, "kernel_size ", kernel_size,
              " does not match sample_map ", map.sizes());
}

std::tuple<Tensor, Tensor> mapped_max_pool(const Tensor& x, const Tensor& map, const OptTensor& wts,
                                           int64_t kernel_size, int64_t interp) {
  check_first(x);
  check_one(x, "x", x);
  check_one(x, "sample_map", map);
  check_opt(x, "interp_weights", wts);
  const int64_t P = npts(map, wts, 4);
  TORCH_CHECK(x.dim() == 4, "x must be [B, C, H, W]");
  check_kernel(map, kernel_size);
  const int64_t B = x.size(0), C = x.size(1), H = x.size(2), W = x.size(3);
  const int64_t OH = map.size(0), OW = map.size(1);
  Tensor out = at::empty({B, C, OH, OW}, x.options());
  Tensor idx = at::empty({B, C, OH, OW}, x.options().dtype(at::kLong));
  c10::DeviceGuard guard(x.device());
  SDK_CALL(sdk_mapped_max_pool, x.data_ptr(), map.data_ptr(), cptr(wts), out.data_ptr(),
           idx.data_ptr<int64_t>(), B, C, H, W, OH, OW, kernel_size, (int32_t)P, (int32_t)interp,
           dtype_code(x), stream_of(x));
  return {out, idx};
}

Tensor mapped_avg_pool(const Tensor& x, const Tensor& map, const OptTensor& wts,
                       int64_t kernel_size, int64_t interp) {
  check_first(x);
  check_one(x, "x", x);
  check_one(x, "sample_map", map);
  check_opt(x, "interp_weights", wts);
  const int64_t P = npts(map, wts, 4);
  TORCH_CHECK(x.dim() == 4, "x must be [B, C, H, W]");
  check_kernel(map, kernel_size);
  const int64_t B = x.size(0), C = x.size(1), H = x.size(2), W = x.size(3);
  const int64_t OH = map.size(0), OW = map.size(1);
  Tensor out = at::empty({B, C, OH, OW}, x.options());
  c10::DeviceGuard guard(x.device());
  SDK_CALL(sdk_mapped_avg_pool, x.data_ptr(), map.data_ptr(), cptr(wts), out.data_ptr(), B, C, H, W,
           OH, OW, kernel_size, (int32_t)P, (int32_t)interp, dtype_code(x), stream_of(x));
  return out;
}

Tensor mapped_max_unpool(const Tensor& g, const Tensor& idx, const Tensor& map,
                         const OptTensor& wts, int64_t in_h, int64_t in_w, int64_t kernel_size,
                         int64_t interp) {
  check_first(g);
  check_one(g, "grad_output", g);
  check_one(g, "idx_mask", idx, true);
  check_one(g, "sample_map", map);
  check_opt(g, "interp_weights", wts);
  TORCH_CHECK(idx.scalar_type() == at::kLong && idx.sizes() == g.sizes(),
              "idx_mask must be an int64 tensor shaped like grad_output");
  const int64_t P = npts(map, wts, 4);
  TORCH_CHECK(g.dim() == 4, "grad_output must be [B, C, OH, OW]");
  const int64_t B = g.size(0), C = g.size(1), OH = g.size(2), OW = g.size(3);
  TORCH_CHECK(map.size(0) == OH && map.size(1) == OW && map.size(2) == kernel_size, "sample_map ",
              map.sizes(), " does not match grad_output ", g.sizes(), " / kernel_size ",
              kernel_size);
  const int dt = dtype_code(g);
  Tensor gin = at::empty({B, C, in_h, in_w}, g.options());
  c10::DeviceGuard guard(g.device());
  hipStream_t s = stream_of(g);
  if (g_unpool_workspace) {
    PlanRef plan = scatter_plan(kMaxUnpool, g, map, wts, in_h, in_w, kernel_size, P, interp, s);
    if (plan.plan.defined() && plan.complete) {
      SDK_CALL(sdk_mapped_max_unpool_planned_bands, g.data_ptr(), idx.data_ptr<int64_t>(),
               map.data_ptr(), gin.data_ptr(), plan.ptr(), plan.nbytes, B, C, in_h, in_w, OH, OW,
               kernel_size, (int32_t)interp, dt, s);
      return gin;
    }
    if (plan.plan.defined()) {
      SDK_CALL(sdk_mapped_max_unpool_planned, g.data_ptr(), idx.data_ptr<int64_t>(), map.data_ptr(),
               cptr(wts), gin.data_ptr(), plan.ptr(), plan.nbytes, B, C, in_h, in_w, OH, OW,
               kernel_size, (int32_t)P, (int32_t)interp, dt, s);
      return gin;
    }
  }
  const size_t nws = g_unpool_workspace ? sdk_mapped_max_unpool_workspace_bytes(in_h, in_w, dt) : 0;
  Tensor ws;
  if (nws) ws = bytes_on(g, nws);
  SDK_CALL(sdk_mapped_max_unpool, g.data_ptr(), idx.data_ptr<int64_t>(), map.data_ptr(), cptr(wts),
           gin.data_ptr(), nws ? ws.data_ptr() : nullptr, nws, B, C, in_h, in_w, OH, OW,
           kernel_size, (int32_t)P, (int32_t)interp, dt, s);
  return gin;
}

Tensor mapped_avg_unpool(const Tensor& g, const Tensor& map, const OptTensor& wts, int64_t in_h,
                         int64_t in_w, int64_t kernel_size, int64_t interp) {
  check_first(g);
  check_one(g, "grad_output", g);
  check_one(g, "sample_map", map);
  check_opt(g, "interp_weights", wts);
  const int64_t P = npts(map, wts, 4);
  TORCH_CHECK(g.dim() == 4, "grad_output must be [B, C, OH, OW]");
  const int64_t B = g.size(0), C = g.size(1), OH = g.size(2), OW = g.size(3);
  TORCH_CHECK(map.size(0) == OH && map.size(1) == OW && map.size(2) == kernel_size, "sample_map ",
              map.sizes(), " does not match grad_output ", g.sizes(), " / kernel_size ",
              kernel_size);
  const int dt = dtype_code(g);
  Tensor gin = at::empty({B, C, in_h, in_w}, g.options());
  c10::DeviceGuard guard(g.device());
  hipStream_t s = stream_of(g);
  if (sdk_mapped_avg_unpool_lists_bytes(in_h, in_w, OH, OW, kernel_size, (int32_t)P,
                                        (int32_t)interp, dt) != 0) {
    PlanRef lists = scatter_plan(kAvgUnpoolLists, g, map, wts, in_h, in_w, kernel_size, P, interp, s);
    if (lists.plan.defined()) {
      SDK_CALL(sdk_mapped_avg_unpool_from_lists, g.data_ptr(), gin.data_ptr(), lists.ptr(),
               lists.nbytes, B, C, in_h, in_w, OH, OW, kernel_size, (int32_t)P, (int32_t)interp, dt,
               s);
      return gin;
    }
  }
  PlanRef plan = scatter_plan(kAvgUnpool, g, map, wts, in_h, in_w, kernel_size, P, interp, s);
  if (plan.plan.defined()) {
    SDK_CALL(sdk_mapped_avg_unpool_planned, g.data_ptr(), map.data_ptr(), cptr(wts), gin.data_ptr(),
             plan.ptr(), plan.nbytes, plan.complete, B, C, in_h, in_w, OH, OW, kernel_size,
             (int32_t)P, (int32_t)interp, dt, s);
    return gin;
  }
  const size_t nws = sdk_resample_to_map_workspace_bytes(in_h, in_w, dt);
  Tensor ws;
  if (nws) ws = bytes_on(g, nws);
  SDK_CALL(sdk_mapped_avg_unpool, g.data_ptr(), map.data_ptr(), cptr(wts), gin.data_ptr(),
           nws ? ws.data_ptr() : nullptr, nws, B, C, in_h, in_w, OH, OW, kernel_size, (int32_t)P,
           (int32_t)interp, dt, s);
  return gin;
}

// ----------------------------------------------------------------------------- convolution
ConvDims conv_dims(const Tensor& x, const Tensor& weight, const Tensor& map, int64_t kernel_size,
                   bool transposed) {
  TORCH_CHECK(x.dim() == 4 && weight.dim() == 3 && map.dim() >= 4, "bad tensor ranks");
  TORCH_CHECK(map.size(2) == kernel_size && weight.size(2) == kernel_size, "kernel_size ",
              kernel_size, " does not match sample_map ", map.sizes(), " / weight ",
              weight.sizes());
  ConvDims d;
  d.B = x.size(0);
  d.Cin = x.size(1);
  d.K = kernel_size;
  TORCH_CHECK(weight.size(transposed ? 0 : 1) == d.Cin, "weight ", weight.sizes(),
              " does not match ", d.Cin, " input channels");
  d.Cout = weight.size(transposed ? 1 : 0);
  return d;
}

Tensor workspace(const Tensor& ref, const ConvDims& d, int64_t img_h, int64_t img_w, int64_t map_h,
                 int64_t map_w, int64_t P, int64_t interp, size_t* n) {
  *n = sdk_mapped_conv_workspace_bytes(d.B, d.Cin, d.Cout, img_h, img_w, map_h, map_w, d.K,
                                       (int32_t)P, (int32_t)interp, dtype_code(ref), current_mode());
  return *n ? bytes_on(ref, *n) : Tensor();
}

Tensor mapped_conv_forward(const Tensor& x, const Tensor& map, const OptTensor& wts,
                           const Tensor& weight, const Tensor& bias, int64_t kernel_size,
                           int64_t interp) {
  check_first(x);
  check_one(x, "input", x);
  check_one(x, "sample_map", map);
  check_opt(x, "interp_weights", wts);
  check_one(x, "weight", weight);
  check_one(x, "bias", bias);
  const int64_t P = npts(map, wts, 4);
  const ConvDims d = conv_dims(x, weight, map, kernel_size, false);
  const int64_t H = x.size(2), W = x.size(3), OH = map.size(0), OW = map.size(1);
  Tensor out = at::empty({d.B, d.Cout, OH, OW}, x.options());
  c10::DeviceGuard guard(x.device());
  hipStream_t s = stream_of(x);
  size_t nws = 0;
  Tensor ws = workspace(x, d, H, W, OH, OW, P, interp, &nws);
  PlanRef plan = conv_plan(x, map, wts, d, H, W, P, interp, false, true, false, x.requires_grad(), s);
  const int dt = dtype_code(x), mode = current_mode();
  void* wsp = nws ? ws.data_ptr() : nullptr;
  if (!plan.plan.defined())
    SDK_CALL(sdk_mapped_conv_forward, x.data_ptr(), map.data_ptr(), cptr(wts), weight.data_ptr(),
             bias.data_ptr(), out.data_ptr(), wsp, nws, d.B, d.Cin, H, W, d.Cout, OH, OW, d.K,
             (int32_t)P, (int32_t)interp, dt, mode, s);
  else
    SDK_CALL(sdk_mapped_conv_forward_planned, x.data_ptr(), map.data_ptr(), cptr(wts),
             weight.data_ptr(), bias.data_ptr(), out.data_ptr(), wsp, nws, plan.ptr(), plan.nbytes,
             d.B, d.Cin, H, W, d.Cout, OH, OW, d.K, (int32_t)P, (int32_t)interp, dt, mode, s);
  return out;
}

std::tuple<Tensor, Tensor, Tensor> mapped_conv_backward(const Tensor& grad_output,
                                                        const Tensor& map, const OptTensor& wts,
                                                        const Tensor& x, const Tensor& weight,
                                                        const Tensor& bias, int64_t kernel_size,
                                                        int64_t interp) {
  // The reference checks input, sample_map, weight and bias here, not grad_output
  // (include/layers/mapped_convolution_layer.h:93-96); the kernels need it dense too.
  const Tensor g = grad_output.contiguous();
  check_first(g);
  check_one(g, "grad_output", g);
  check_one(g, "input", x);
  check_one(g, "sample_map", map);
  check_opt(g, "interp_weights", wts);
  check_one(g, "weight", weight);
  check_one(g, "bias", bias);
  const int64_t P = npts(map, wts, 4);
  const ConvDims d = conv_dims(x, weight, map, kernel_size, false);
  const int64_t H = x.size(2), W = x.size(3), OH = map.size(0), OW = map.size(1);
  Tensor gi = at::empty_like(x), gw = at::empty_like(weight);
  Tensor gb = at::empty({d.Cout}, x.options());
  c10::DeviceGuard guard(x.device());
  hipStream_t s = stream_of(x);
  size_t nws = 0;
  Tensor ws = workspace(x, d, H, W, OH, OW, P, interp, &nws);
  PlanRef plan = conv_plan(x, map, wts, d, H, W, P, interp, false, false, true, true, s);
  const int dt = dtype_code(x), mode = current_mode();
  void* wsp = nws ? ws.data_ptr() : nullptr;
  if (!plan.plan.defined())
    SDK_CALL(sdk_mapped_conv_backward, g.data_ptr(), map.data_ptr(), cptr(wts), x.data_ptr(),
             weight.data_ptr(), gi.data_ptr(), gw.data_ptr(), gb.data_ptr(), wsp, nws, d.B, d.Cin,
             H, W, d.Cout, OH, OW, d.K, (int32_t)P, (int32_t)interp, dt, mode, s);
  else
    SDK_CALL(sdk_mapped_conv_backward_planned, g.data_ptr(), map.data_ptr(), cptr(wts),
             x.data_ptr(), weight.data_ptr(), gi.data_ptr(), gw.data_ptr(), gb.data_ptr(), wsp, nws,
             plan.ptr(), plan.nbytes, d.B, d.Cin, H, W, d.Cout, OH, OW, d.K, (int32_t)P,
             (int32_t)interp, dt, mode, s);
  return {gi, gw, gb};
}

Tensor mapped_transposed_conv_forward(const Tensor& x, const Tensor& map, const OptTensor& wts,
                                      const Tensor& weight, const Tensor& bias, int64_t out_h,
                                      int64_t out_w, int64_t kernel_size, int64_t interp) {
  check_first(x);
  check_one(x, "input", x);
  check_one(x, "sample_map", map);
  check_opt(x, "interp_weights", wts);
  check_one(x, "weight", weight);
  check_one(x, "bias", bias);
  const int64_t P = npts(map, wts, 4);
  const ConvDims d = conv_dims(x, weight, map, kernel_size, true);
  const int64_t IH = x.size(2), IW = x.size(3);
  TORCH_CHECK(map.size(0) == IH && map.size(1) == IW, "sample_map grid ", map.sizes().slice(0, 2),
              " must match the input's ", x.sizes().slice(2));
  Tensor out = at::empty({d.B, d.Cout, out_h, out_w}, x.options());
  c10::DeviceGuard guard(x.device());
  hipStream_t s = stream_of(x);
  size_t nws = 0;
  Tensor ws = workspace(x, d, out_h, out_w, IH, IW, P, interp, &nws);
  PlanRef plan = conv_plan(x, map, wts, d, out_h, out_w, P, interp, true, x.requires_grad(), false,
                           true, s);
  const int dt = dtype_code(x), mode = current_mode();
  void* wsp = nws ? ws.data_ptr() : nullptr;
  if (!plan.plan.defined())
    SDK_CALL(sdk_mapped_transposed_conv_forward, x.data_ptr(), map.data_ptr(), cptr(wts),
             weight.data_ptr(), bias.data_ptr(), out.data_ptr(), wsp, nws, d.B, d.Cin, IH, IW,
             d.Cout, out_h, out_w, d.K, (int32_t)P, (int32_t)interp, dt, mode, s);
  else
    SDK_CALL(sdk_mapped_transposed_conv_forward_planned, x.data_ptr(), map.data_ptr(), cptr(wts),
             weight.data_ptr(), bias.data_ptr(), out.data_ptr(), wsp, nws, plan.ptr(), plan.nbytes,
             d.B, d.Cin, IH, IW, d.Cout, out_h, out_w, d.K, (int32_t)P, (int32_t)interp, dt, mode,
             s);
  return out;
}

std::tuple<Tensor, Tensor, Tensor> mapped_transposed_conv_backward(
    const Tensor& grad_output, const Tensor& map, const OptTensor& wts, const Tensor& x,
    const Tensor& weight, const Tensor& bias, int64_t kernel_size, int64_t interp) {
  const Tensor g = grad_output.contiguous();
  check_first(g);
  check_one(g, "grad_output", g);
  check_one(g, "input", x);
  check_one(g, "sample_map", map);
  check_opt(g, "interp_weights", wts);
  check_one(g, "weight", weight);
  check_one(g, "bias", bias);
  const int64_t P = npts(map, wts, 4);
  const ConvDims d = conv_dims(x, weight, map, kernel_size, true);
  TORCH_CHECK(g.dim() == 4, "grad_output must be [B, C, OH, OW]");
  const int64_t IH = x.size(2), IW = x.size(3), OH = g.size(2), OW = g.size(3);
  Tensor gi = at::empty_like(x), gw = at::empty_like(weight);
  Tensor gb = at::empty({d.Cout}, x.options());
  c10::DeviceGuard guard(x.device());
  hipStream_t s = stream_of(x);
  size_t nws = 0;
  Tensor ws = workspace(x, d, OH, OW, IH, IW, P, interp, &nws);
  PlanRef plan = conv_plan(x, map, wts, d, OH, OW, P, interp, true, true, true, false, s);
  const int dt = dtype_code(x), mode = current_mode();
  void* wsp = nws ? ws.data_ptr() : nullptr;
  if (!plan.plan.defined())
    SDK_CALL(sdk_mapped_transposed_conv_backward, g.data_ptr(), map.data_ptr(), cptr(wts),
             x.data_ptr(), weight.data_ptr(), gi.data_ptr(), gw.data_ptr(), gb.data_ptr(), wsp, nws,
             d.B, d.Cin, IH, IW, d.Cout, OH, OW, d.K, (int32_t)P, (int32_t)interp, dt, mode, s);
  else
    SDK_CALL(sdk_mapped_transposed_conv_backward_planned, g.data_ptr(), map.data_ptr(), cptr(wts),
             x.data_ptr(), weight.data_ptr(), gi.data_ptr(), gw.data_ptr(), gb.data_ptr(), wsp, nws,
             plan.ptr(), plan.nbytes, d.B, d.Cin, IH, IW, d.Cout, OH, OW, d.K, (int32_t)P,
             (int32_t)interp, dt, mode, s);
  return {gi, gw, gb};
}

// The gradients that are wanted, undefined tensors for the others (what the plain backward
// operators return, without the work nobody asks for).
std::tuple<Tensor, Tensor, Tensor> mapped_conv_backward_select(
    const Tensor& grad_output, const Tensor& map, const OptTensor& wts, const Tensor& x,
    const Tensor& weight, int64_t kernel_size, int64_t interp, bool transposed, bool need_input,
    bool need_params) {
  const Tensor g = grad_output.contiguous();
  check_first(g);
  check_one(g, "input", x);
  check_one(g, "sample_map", map);
  check_opt(g, "interp_weights", wts);
  check_one(g, "weight", weight);
  const int64_t P = npts(map, wts, 4);
  const ConvDims d = conv_dims(x, weight, map, kernel_size, transposed);
  TORCH_CHECK(g.dim() == 4, "grad_output must be [B, C, OH, OW]");
  const int64_t IH = x.size(2), IW = x.size(3), OH = g.size(2), OW = g.size(3);
  const int64_t img_h = transposed ? OH : IH, img_w = transposed ? OW : IW;
  Tensor gi, gw, gb;
  if (need_input) gi = at::empty_like(x);
  if (need_params) {
    gw = at::empty_like(weight);
    gb = at::empty({d.Cout}, x.options());
  }
  c10::DeviceGuard guard(x.device());
  hipStream_t s = stream_of(x);
  size_t nws = 0;
  Tensor ws = workspace(x, d, img_h, img_w, map.size(0), map.size(1), P, interp, &nws);
  PlanRef plan = conv_plan(x, map, wts, d, img_h, img_w, P, interp, transposed,
                           transposed && need_input, need_params, !transposed && need_input, s);
  const auto ptr = [](const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; };
  const auto call = transposed ? sdk_mapped_transposed_conv_backward_select
                               : sdk_mapped_conv_backward_select;
  const int rc =
      call(g.data_ptr(), map.data_ptr(), cptr(wts), x.data_ptr(), weight.data_ptr(), ptr(gi),
           ptr(gw), ptr(gb), ptr(ws), nws, plan.ptr(), plan.nbytes, d.B, d.Cin, IH, IW, d.Cout, OH,
           OW, d.K, (int32_t)P, (int32_t)interp, dtype_code(x), current_mode(), s);
  if (rc != 0) fail_call("sdk_mapped_conv_backward_select", rc);
  return {gi, gw, gb};
}

// ----------------------------------------------------------------------------- textures, labels
void check_uv(const Tensor& ref, const Tensor& quad, const Tensor& uv) {
  check_one(ref, "quad_idx", quad, true);
  check_one(ref, "tex_uv", uv);
  TORCH_CHECK(quad.scalar_type() == at::kLong && quad.dim() == 2,
              "quad_idx must be a 2-D int64 tensor, got ", quad.scalar_type(), " ", quad.sizes());
  TORCH_CHECK(uv.dim() == 3 && uv.size(0) == quad.size(0) && uv.size(1) == quad.size(1) &&
                  uv.size(2) == 2,
              "tex_uv ", uv.sizes(), " must be quad_idx ", quad.sizes(), " + (2,)");
}

Tensor resample_from_uv_maps(const Tensor& textures, const Tensor& quad, const Tensor& uv,
                             int64_t interp) {
  check_first(textures);
  check_one(textures, "textures", textures);
  check_uv(textures, quad, uv);
  TORCH_CHECK(textures.dim() == 5, "textures must be [B, C, T, TH, TW], got ", textures.sizes());
  const int64_t B = textures.size(0), C = textures.size(1), H = quad.size(0), W = quad.size(1);
  Tensor out = at::empty({B, C, H, W}, textures.options());
  c10::DeviceGuard guard(textures.device());
  SDK_CALL(sdk_resample_from_uv_maps, textures.data_ptr(), quad.data_ptr<int64_t>(), uv.data_ptr(),
           out.data_ptr(), B, C, textures.size(2), textures.size(3), textures.size(4), H, W,
           (int32_t)interp, dtype_code(textures), stream_of(textures));
  return out;
}

Tensor resample_to_uv_maps(const Tensor& x, const Tensor& quad, const Tensor& uv, int64_t NT,
                           int64_t TH, int64_t TW, int64_t interp) {
  check_first(x);
  check_one(x, "x", x);
  check_uv(x, quad, uv);
  const int64_t H = quad.size(0), W = quad.size(1);
  TORCH_CHECK(x.dim() == 4 && x.size(2) == H && x.size(3) == W, "input ", x.sizes(),
              " must be [B, C, ", H, ", ", W, "]");
  const int64_t B = x.size(0), C = x.size(1);
  const int dt = dtype_code(x);
  Tensor out = at::empty({B, C, NT, TH, TW}, x.options());
  c10::DeviceGuard guard(x.device());
  hipStream_t s = stream_of(x);
  const size_t nws = sdk_resample_to_uv_maps_workspace_bytes(NT, TH, TW, H, W, dt);
  // the pixels bucketed by texture, a function of quad_idx alone
  Key key;
  key.kind = kUvScatter;
  key.device = x.device().index();
  key.dtype = dt;
  key.a = NT;
  key.b = TH;
  key.K = TW;
  PlanRef plan = plan_for(
      key, x, quad, OptTensor(), s, [&] { return nws; },
      [&](void* buf, size_t n, int) {
        SDK_CALL(sdk_resample_to_uv_maps_plan_build, quad.data_ptr<int64_t>(), buf, n, NT, TH, TW,
                 H, W, dt, s);
        return 1;
      });
  if (plan.plan.defined()) {
    SDK_CALL(sdk_resample_to_uv_maps_planned, x.data_ptr(), quad.data_ptr<int64_t>(), uv.data_ptr(),
             out.data_ptr(), plan.ptr(), plan.nbytes, B, C, NT, TH, TW, H, W, (int32_t)interp, dt,
             s);
    return out;
  }
  Tensor ws;
  if (nws) ws = bytes_on(x, nws);
  SDK_CALL(sdk_resample_to_uv_maps, x.data_ptr(), quad.data_ptr<int64_t>(), uv.data_ptr(),
           out.data_ptr(), nws ? ws.data_ptr() : nullptr, nws, B, C, NT, TH, TW, H, W,
           (int32_t)interp, dt, s);
  return out;
}

Tensor voting_resample_to_map(const Tensor& labels, const Tensor& map, int64_t out_h, int64_t out_w,
                              int64_t candidates) {
  const std::pair<const char*, const Tensor*> named[2] = {{"input", &labels}, {"sample_map", &map}};
  for (const auto& t : named) {
    TORCH_CHECK(t.second->is_cuda(), "this backend runs on the GPU only: ", t.first,
                " must be a CUDA/HIP tensor");
    TORCH_CHECK(t.second->scalar_type() == at::kLong, t.first, " must be int64 (got ",
                t.second->scalar_type(), ")");
    TORCH_CHECK(t.second->is_contiguous(), t.first, " must be contiguous");
  }
  TORCH_CHECK(labels.dim() == 4 && map.dim() == 3 && map.size(0) == labels.size(2) &&
                  map.size(1) == labels.size(3) && map.size(2) == 2,
              "input ", labels.sizes(), " must be [B, C, IH, IW] and sample_map ", map.sizes(),
              " [IH, IW, 2]");
  const int64_t B = labels.size(0), C = labels.size(1);
  Tensor out = at::empty({B, C, out_h, out_w}, labels.options());
  c10::DeviceGuard guard(labels.device());
  // room for several batch elements per pass, within 256 MiB
  size_t nws = sdk_voting_resample_workspace_bytes(C, out_h, out_w, candidates);
  const int64_t fit = (int64_t)(((size_t)256 << 20) / std::max<size_t>(nws, 1));
  nws *= (size_t)std::max<int64_t>(1, std::min<int64_t>(B, fit));
  Tensor ws = bytes_on(labels, std::max<size_t>(nws, 16));
  SDK_CALL(sdk_voting_resample_to_map, labels.data_ptr<int64_t>(), map.data_ptr<int64_t>(),
           out.data_ptr<int64_t>(), ws.data_ptr(), nws, B, C, labels.size(2), labels.size(3), out_h,
           out_w, candidates, stream_of(labels));
  return out;
}

}  // namespace

TORCH_LIBRARY_IMPL(sdk_mapped_ops, CUDA, m) {
  m.impl("resample_from_map", &resample_from_map);
  m.impl("resample_to_map", &resample_to_map);
  m.impl("resample_to_map_normalized", &resample_to_map_normalized);
  m.impl("resample_from_uv_maps", &resample_from_uv_maps);
  m.impl("resample_to_uv_maps", &resample_to_uv_maps);
  m.impl("voting_resample_to_map", &voting_resample_to_map);
  m.impl("mapped_max_pool", &mapped_max_pool);
  m.impl("mapped_max_unpool", &mapped_max_unpool);
  m.impl("mapped_avg_pool", &mapped_avg_pool);
  m.impl("mapped_avg_unpool", &mapped_avg_unpool);
  m.impl("mapped_conv_forward", &mapped_conv_forward);
  m.impl("mapped_conv_backward", &mapped_conv_backward);
  m.impl("mapped_transposed_conv_forward", &mapped_transposed_conv_forward);
  m.impl("mapped_transposed_conv_backward", &mapped_transposed_conv_backward);
  m.impl("mapped_conv_backward_select", &mapped_conv_backward_select);
}

// Controls, called from Python (ctypes): the compute mode (process default and per-thread
// override), the plan cache and the unpool workspace switch.
extern "C" {
const char* sdk_torch_native_ops(void) {
  return "resample_from_map,resample_to_map,resample_to_map_normalized,mapped_max_pool,"
         "mapped_max_unpool,mapped_avg_pool,mapped_avg_unpool,mapped_conv_forward,"
         "mapped_conv_backward,mapped_transposed_conv_forward,mapped_transposed_conv_backward";
}
// ... and those for textures and labels, and the backward that forms only the gradients asked for
const char* sdk_torch_native_more(void) {
  return "mapped_conv_backward_select,resample_from_uv_maps,resample_to_uv_maps,"
         "voting_resample_to_map";
}
void sdk_torch_set_default_mode(int mode) { g_default_mode = mode; }
// mode < 0 removes the override; returns the previous override (-1: none)
int sdk_torch_set_thread_mode(int mode) {
  const int prev = t_mode;
  t_mode = mode;
  return prev;
}
int sdk_torch_current_mode(void) { return current_mode(); }
void sdk_torch_set_plan_cache(int enabled, int max_entries) {
  std::lock_guard<std::mutex> lock(g_mu);
  g_cache_enabled = enabled != 0;
  if (max_entries > 0) g_cache_max = (size_t)max_entries;
  if (!g_cache_enabled) g_cache.clear();
  shrink_cache(g_cache_max);
}
int sdk_torch_plan_cache_size(void) {
  std::lock_guard<std::mutex> lock(g_mu);
  return (int)g_cache.size();
}
void sdk_torch_set_unpool_workspace(int enabled) { g_unpool_workspace = enabled != 0; }
}
