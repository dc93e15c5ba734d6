// gp_xfer.h -- transfers between a caller's ordinary (pageable) memory and
// the device.
//
// A plain copy of pageable memory is staged by one host thread: it reaches
// 5-15 GB/s, less where the destination's pages are touched for the first
// time, against about 50 GB/s of the link.  Here a transfer is cut into
// chunks of at most XFER_CHUNK bytes that several workers take in turn, each
// with its own page-locked buffer: while one chunk is on the link the others
// are copied (and their pages touched) by the other workers.
//
// The buffers belong to the object that makes the transfers (a particle
// context, a fluid state), at most XFER_WORKERS x XFER_CHUNK bytes on either
// side, and go with it.  The workers live within one call.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstddef>
#include <cstring>
#include <thread>

namespace gpx {

constexpr int XFER_WORKERS = 8;
constexpr size_t XFER_CHUNK = (size_t)4 << 20;
// below this a chunk is not worth a worker of its own (starting one costs
// about 30 us, in which one thread copies some 300 KB)
constexpr size_t XFER_SPLIT = (size_t)1 << 20;

struct Xfer {
  char* pin[XFER_WORKERS] = {};
  char* dev[XFER_WORKERS] = {};
  hipEvent_t ev[XFER_WORKERS] = {};
  size_t pin_n[XFER_WORKERS] = {}, dev_n[XFER_WORKERS] = {};

  void release() {
    for (int b = 0; b < XFER_WORKERS; ++b) {
      if (pin[b]) (void)hipHostFree(pin[b]);
      if (dev[b]) (void)hipFree(dev[b]);
      if (ev[b]) (void)hipEventDestroy(ev[b]);
      pin[b] = dev[b] = nullptr;
      ev[b] = nullptr;
      pin_n[b] = dev_n[b] = 0;
    }
  }

  // buffers of the first n workers (device ones on request); one that is too
  // small is followed by one of twice its size or more, up to XFER_CHUNK, so
  // that lists that grow from call to call do not allocate each time (the
  // first is as large as asked: page-locking takes 0.35 ms a MB).  The
  // transfers that used the old ones are complete
  hipError_t reserve(int n, size_t bytes, bool device) {
    auto size = [&](size_t had) { return std::max(bytes, std::min(XFER_CHUNK, 2 * had)); };
    for (int b = 0; b < n; ++b) {
      hipError_t e;
      if (!ev[b] && (e = hipEventCreateWithFlags(&ev[b], hipEventDisableTiming)) != hipSuccess)
        return e;
      if (pin_n[b] < bytes) {
        const size_t m = size(pin_n[b]);
        if (pin[b]) (void)hipHostFree(pin[b]);
        pin[b] = nullptr;
        pin_n[b] = 0;
        if ((e = hipHostMalloc((void**)&pin[b], m)) != hipSuccess) return e;
        pin_n[b] = m;
      }
      if (device && dev_n[b] < bytes) {
        const size_t m = size(dev_n[b]);
        if (dev[b]) (void)hipFree(dev[b]);
        dev[b] = nullptr;
        dev_n[b] = 0;
        if ((e = hipMalloc((void**)&dev[b], m)) != hipSuccess) return e;
        dev_n[b] = m;
      }
    }
    return hipSuccess;
  }

  // f(worker, chunk) for every chunk, workers in parallel (a chunk's number
  // modulo n is its worker); the first error ends it, when what was queued on
  // the stream by then (it uses the buffers) is complete
  template <typename F>
  static hipError_t run(int n, long long chunks, hipStream_t st, F&& f) {
    std::atomic<int> err{(int)hipSuccess};
    int device = 0;
    (void)hipGetDevice(&device);
    auto work = [&](int b) {
      for (long long q = b; q < chunks && err.load() == (int)hipSuccess; q += n) {
        const hipError_t e = f(b, q);
        if (e != hipSuccess) err.store((int)e);
      }
    };
    std::thread th[XFER_WORKERS];
    int started = 1;
    for (; started < n; ++started) {
      const int b = started;
      try {
        th[b] = std::thread([&, b] {
          (void)hipSetDevice(device);   // a thread starts on device 0
          work(b);
        });
      } catch (...) {
        break;   // no more threads, or no memory for one: their chunks are taken below
      }
    }
    work(0);
    for (int b = started; b < n; ++b) work(b);
    for (int b = 1; b < started; ++b) th[b].join();
    if (err.load() != (int)hipSuccess) (void)hipStreamSynchronize(st);
    return (hipError_t)err.load();
  }

  static int workers(size_t total) {
    const unsigned hw = std::thread::hardware_concurrency();
    const int most = std::min<int>(XFER_WORKERS, hw > 2 ? (int)hw / 2 : 1);
    return std::max(1, std::min<int>(most, (int)std::min<size_t>(total / XFER_SPLIT, 64)));
  }
  static size_t chunk_of(size_t total, int n) {
    return std::min(XFER_CHUNK, ((total + n - 1) / n + 4095) / 4096 * 4096);
  }

  // device memory to host memory, complete on return
  hipError_t d2h(void* dst, const void* src, size_t bytes, hipStream_t st) {
    if (!bytes) return hipStreamSynchronize(st);
    const int n = workers(bytes);
    const size_t ch = chunk_of(bytes, n);
    hipError_t e = reserve(n, ch, false);
    if (e != hipSuccess) return e;
    return run(n, (long long)((bytes + ch - 1) / ch), st, [&](int b, long long q) {
      const size_t o = (size_t)q * ch, m = std::min(ch, bytes - o);
      hipError_t r = hipMemcpyAsync(pin[b], (const char*)src + o, m, hipMemcpyDeviceToHost, st);
      if (r == hipSuccess) r = hipEventRecord(ev[b], st);
      if (r == hipSuccess) r = hipEventSynchronize(ev[b]);
      if (r == hipSuccess) std::memcpy((char*)dst + o, pin[b], m);
      return r;
    });
  }

  // host memory to device memory, complete on return
  hipError_t h2d(void* dst, const void* src, size_t bytes, hipStream_t st) {
    if (!bytes) return hipStreamSynchronize(st);
    const int n = workers(bytes);
    const size_t ch = chunk_of(bytes, n);
    hipError_t e = reserve(n, ch, false);
    if (e != hipSuccess) return e;
    e = run(n, (long long)((bytes + ch - 1) / ch), st, [&](int b, long long q) {
      const size_t o = (size_t)q * ch, m = std::min(ch, bytes - o);
      // the buffer's last chunk has left it
      hipError_t r = q >= n ? hipEventSynchronize(ev[b]) : hipSuccess;
      if (r != hipSuccess) return r;
      std::memcpy(pin[b], (const char*)src + o, m);
      r = hipMemcpyAsync((char*)dst + o, pin[b], m, hipMemcpyHostToDevice, st);
      if (r == hipSuccess) r = hipEventRecord(ev[b], st);
      return r;
    });
    const hipError_t s = hipStreamSynchronize(st);
    return e != hipSuccess ? e : s;
  }
};

}  // namespace gpx
