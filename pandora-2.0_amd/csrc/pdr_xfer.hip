// pdr_xfer.hip -- fields between the device and the caller's host arrays (FP64 on the
// host; the device holds FP64 or FP32), through pinned memory of the context.
//
// A pageable hipMemcpy stages through the runtime's own buffers on one thread, and an
// FP32-mixed field was converted after it on the same thread, which also took the page
// faults of the caller's array.  Here chunks of 1 MB go by DMA into pinned slots and as many
// threads as the size warrants copy or convert them out, two slots each, so that DMA,
// conversion and page faults overlap: 512^3 FP32-mixed velocity read back into arrays in use
// 145 -> 15.3 ms, 324 -> 190 into fresh pages, 256^3 FP64 7.0 -> 3.9 and 33 -> 21.  A small
// box's fields go in one kernel that writes them into the pinned memory: one launch and one
// wait instead of three copies (32^3 FP64 0.05 to 0.13 -> 0.03 ms, 48^3 0.074 -> 0.054).
#include <algorithm>
#include <cstring>
#include <string>
#include <thread>
#include <vector>

#include "pdr_internal.hpp"

namespace pdr {

namespace {

constexpr size_t kChunk = size_t(1) << 20;  // device bytes of a chunk
constexpr size_t kSmall = size_t(1) << 20;  // fields that go in one kernel
constexpr int kMaxThreads = 8;

// Copies up to three fields of n words into one pinned array, one after another.
template <typename W>
__global__ void __launch_bounds__(256)
    k_xfer(W* __restrict__ host, const W* d0, const W* d1, const W* d2, int fields, long long n) {
  const long long step = (long long)gridDim.x * blockDim.x;
  for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < fields * n; e += step) {
    const int f = int(e / n);
    host[e] = (f == 0 ? d0 : (f == 1 ? d1 : d2))[e - f * n];
  }
}

hipError_t launch_xfer(pdr_ctx* c, void* host, void* const* dev, int fields, long long n, bool f32) {
  const unsigned nb = unsigned(std::min<long long>((fields * n + 255) / 256, 512));
  void *a = dev[0], *b = dev[fields > 1 ? 1 : 0], *d = dev[fields > 2 ? 2 : 0];
  if (f32)
    k_xfer<float><<<nb, 256, 0, c->stream>>>((float*)host, (float*)a, (float*)b, (float*)d, fields, n);
  else
    k_xfer<double><<<nb, 256, 0, c->stream>>>((double*)host, (double*)a, (double*)b, (double*)d, fields, n);
  return hipGetLastError();
}

// The context's pinned memory, at least `bytes` of it.
hipError_t stage_reserve(pdr_ctx* c, size_t bytes) {
  if (c->stage_bytes >= bytes) return hipSuccess;
  if (c->stage) (void)hipHostFree(c->stage);
  c->stage = nullptr;
  c->stage_bytes = 0;
  const hipError_t e = hipHostMalloc(&c->stage, bytes, hipHostMallocDefault);
  if (e != hipSuccess) {
    (void)hipGetLastError();  // the caller goes on without: later launch checks read it
    c->stage = nullptr;
    return e;
  }
  c->stage_bytes = bytes;
  return hipSuccess;
}

void words_out(double* dst, const void* src, size_t n, bool f32) {
  if (!f32) {
    std::memcpy(dst, src, n * sizeof(double));
    return;
  }
  const float* s = static_cast<const float*>(src);
  for (size_t q = 0; q < n; ++q) dst[q] = double(s[q]);
}
void words_in(void* dst, const double* src, size_t n, bool f32) {
  if (!f32) {
    std::memcpy(dst, src, n * sizeof(double));
    return;
  }
  float* d = static_cast<float*>(dst);
  for (size_t q = 0; q < n; ++q) d[q] = float(src[q]);
}

// Straight to or from the caller's arrays, through the runtime's own buffers.
template <bool OUT>
hipError_t pageable(pdr_ctx* c, int fields, void* const* dev, double* const* host, long long n, bool f32) {
  const size_t fbytes = size_t(n) * (f32 ? sizeof(float) : sizeof(double));
  hipError_t e = hipStreamSynchronize(c->stream);
  std::vector<float> tmp(f32 ? size_t(n) : 0);
  for (int f = 0; f < fields && e == hipSuccess; ++f) {
    void* h = f32 ? (void*)tmp.data() : (void*)host[f];
    if (!OUT && f32) words_in(h, host[f], size_t(n), true);
    e = OUT ? hipMemcpy(h, dev[f], fbytes, hipMemcpyDeviceToHost) : hipMemcpy(dev[f], h, fbytes, hipMemcpyHostToDevice);
    if (OUT && f32 && e == hipSuccess) words_out(host[f], h, size_t(n), true);
  }
  return e;
}

template <bool OUT>
hipError_t transfer(pdr_ctx* c, int fields, void* const* dev, double* const* host, long long n, bool f32) {
  const OnDevice on(c);
  const size_t w = f32 ? sizeof(float) : sizeof(double);
  const size_t fbytes = size_t(n) * w, total = fbytes * size_t(fields);
  // Pinning costs 0.3 ms for a small box's fields and up to 4 ms for the chunks: not spent
  // on what is often done once, a small box's uploads and first download and FP64 uploads.
  // Where the host has no pinned memory to give, every transfer goes this way.
  if (OUT ? total <= kSmall && c->small_downloads++ == 0 : total <= kSmall || !f32)
    return pageable<OUT>(c, fields, dev, host, n, f32);
  if (OUT && total <= kSmall) {
    if (stage_reserve(c, total) != hipSuccess) return pageable<OUT>(c, fields, dev, host, n, f32);
    hipError_t e = launch_xfer(c, c->stage, dev, fields, n, f32);
    if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
    if (e == hipSuccess)
      for (int f = 0; f < fields; ++f) words_out(host[f], (char*)c->stage + fbytes * size_t(f), size_t(n), f32);
    return e;
  }
  // chunk k of the fields one after another; thread t takes k = t, t + T, ...
  const size_t per = (fbytes + kChunk - 1) / kChunk, chunks = per * size_t(fields);
  const int hw = int(std::max(1u, std::thread::hardware_concurrency()));
  const int T = std::max(1, std::min({kMaxThreads, hw, int(chunks / 8)}));
  if (stage_reserve(c, 2 * size_t(T) * kChunk) != hipSuccess) return pageable<OUT>(c, fields, dev, host, n, f32);
  // the threads start when there is something to move: waiting for the steps queued
  // before, each would hold a core
  hipError_t e = hipStreamSynchronize(c->stream);
  if (e != hipSuccess) return e;
  std::vector<hipError_t> err(size_t(T), hipSuccess);
  auto work = [&](int t) {
    hipError_t r = hipSetDevice(c->device);
    hipEvent_t ev[2] = {nullptr, nullptr};
    for (hipEvent_t& x : ev)
      if (r == hipSuccess) r = hipEventCreateWithFlags(&x, hipEventDisableTiming);
    auto where = [&](size_t i, size_t* off, size_t* bytes, int* f) {
      const size_t k = size_t(t) + size_t(T) * i;
      *f = int(k / per);
      *off = (k % per) * kChunk;
      *bytes = std::min(kChunk, fbytes - *off);
      return k < chunks;
    };
    auto slot = [&](size_t i) { return (char*)c->stage + (2 * size_t(t) + (i & 1)) * kChunk; };
    auto dma = [&](size_t i) {
      size_t off, bytes;
      int f;
      if (!where(i, &off, &bytes, &f)) return;
      char* d = (char*)dev[f] + off;
      if (r == hipSuccess)
        r = OUT ? hipMemcpyAsync(slot(i), d, bytes, hipMemcpyDeviceToHost, c->stream)
                : hipMemcpyAsync(d, slot(i), bytes, hipMemcpyHostToDevice, c->stream);
      if (r == hipSuccess) r = hipEventRecord(ev[i & 1], c->stream);
    };
    size_t off, bytes;
    int f;
    if (OUT) {
      dma(0);
      dma(1);
    }
    for (size_t i = 0; r == hipSuccess && where(i, &off, &bytes, &f); ++i) {
      // out: the chunk has arrived; in: the slot's chunk before last has left
      if (OUT || i >= 2) r = hipEventSynchronize(ev[i & 1]);
      if (r != hipSuccess) break;
      if (OUT) {
        words_out(host[f] + off / w, slot(i), bytes / w, f32);
        dma(i + 2);
      } else {
        words_in(slot(i), host[f] + off / w, bytes / w, f32);
        dma(i);
      }
    }
    for (hipEvent_t x : ev)
      if (x) (void)hipEventDestroy(x);
    err[size_t(t)] = r;
  };
  std::vector<std::thread> threads;
  int started = 1;
  try {
    for (; started < T; ++started) threads.emplace_back(work, started);
  } catch (...) {  // no more threads to be had: this one does their share
  }
  for (int t = started; t < T; ++t) work(t);
  work(0);
  for (std::thread& x : threads) x.join();
  e = hipStreamSynchronize(c->stream);
  for (hipError_t x : err)
    if (e == hipSuccess) e = x;
  return e;
}

}  // namespace

void xfer_free(pdr_ctx* c) {
  if (c->stage) (void)hipHostFree(c->stage);
  c->stage = nullptr;
  c->stage_bytes = 0;
}

int xfer_to_host(pdr_ctx* c, int fields, const void* const* dev, double* const* host, long long n, bool f32) {
  for (int f = 0; f < fields; ++f)
    if (!host[f]) return set_error(PDR_ERR_ARG, "null host array");
  const hipError_t e = transfer<true>(c, fields, const_cast<void* const*>(dev), host, n, f32);
  if (e != hipSuccess) return set_error(PDR_ERR_HIP, std::string("download: ") + hipGetErrorString(e));
  return PDR_OK;
}

int xfer_from_host(pdr_ctx* c, int fields, void* const* dev, const double* const* host, long long n, bool f32) {
  for (int f = 0; f < fields; ++f)
    if (!host[f]) return set_error(PDR_ERR_ARG, "null host array");
  const hipError_t e = transfer<false>(c, fields, dev, const_cast<double* const*>(host), n, f32);
  if (e != hipSuccess) return set_error(PDR_ERR_HIP, std::string("upload: ") + hipGetErrorString(e));
  return PDR_OK;
}

}  // namespace pdr
