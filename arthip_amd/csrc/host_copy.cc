#include "host_copy.h"

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <thread>

namespace arthip {

namespace {

constexpr size_t kMinChunk = static_cast<size_t>(2) << 20;
constexpr size_t kMaxChunks = 8;
constexpr size_t kMaxThreads = 4;
constexpr size_t kPage = 4096;

// f(destination, staged offset, length) over the staged byte range [a, b).
template <class F>
void for_rows(const std::vector<HostRows>& planes, size_t a, size_t b, F&& f) {
  size_t off = 0;  // staged offset of the plane
  for (const HostRows& p : planes) {
    const size_t len = p.row * static_cast<size_t>(p.rows);
    const size_t lo = std::max(a, off), hi = std::min(b, off + len);
    if (lo < hi) {
      if (p.stride == static_cast<ptrdiff_t>(p.row)) {
        f(p.base + (lo - off), lo, hi - lo);
      } else {
        for (size_t x = lo; x < hi;) {
          const size_t y = (x - off) / p.row, c = (x - off) % p.row;
          const size_t n = std::min(p.row - c, hi - x);
          f(p.base + static_cast<ptrdiff_t>(y) * p.stride + static_cast<ptrdiff_t>(c), x, n);
          x += n;
        }
      }
    }
    off += len;
  }
}

// Writes one byte per page back to itself, so that the page is mapped.
void touch(uint8_t* p, size_t n) {
  for (size_t i = 0; i < n; i += kPage) {
    volatile uint8_t* q = p + i;
    *q = *q;
  }
}

}  // namespace

ChunkedDownload::~ChunkedDownload() {
  for (hipEvent_t e : events_)
    if (e) hipEventDestroy(e);
}

hipError_t ChunkedDownload::Enqueue(int device, hipStream_t s, void* pinned, const void* dev, size_t bytes) {
  const hipError_t r = Send(device, s, pinned, dev, bytes);
  if (r != hipSuccess) (void)hipStreamSynchronize(s);
  return r;
}

hipError_t ChunkedDownload::Send(int device, hipStream_t s, void* pinned, const void* dev, size_t bytes) {
  const size_t want = std::min(kMaxChunks, std::max<size_t>(1, bytes / kMinChunk));
  const size_t chunk = ((bytes + want - 1) / want + kPage - 1) / kPage * kPage;
  events_.reserve(kMaxChunks);
  while (events_.size() < want) {
    hipEvent_t e = nullptr;
    const hipError_t r = hipEventCreateWithFlags(&e, hipEventDisableTiming);
    if (r != hipSuccess) return r;
    events_.push_back(e);
  }
  device_ = device;
  stream_ = s;
  pinned_ = static_cast<const uint8_t*>(pinned);
  bytes_ = bytes;
  chunk_ = chunk;
  n_chunks_ = 0;
  for (size_t o = 0; o < bytes; o += chunk) {
    const size_t n = std::min(chunk, bytes - o);
    hipError_t r = hipMemcpyAsync(static_cast<uint8_t*>(pinned) + o, static_cast<const uint8_t*>(dev) + o, n,
                                  hipMemcpyDeviceToHost, s);
    if (r == hipSuccess) r = hipEventRecord(events_[n_chunks_], s);
    if (r != hipSuccess) return r;
    ++n_chunks_;
  }
  return hipSuccess;
}

hipError_t ChunkedDownload::CopyOut(const std::vector<HostRows>& planes) {
  const size_t parts = std::min(kMaxThreads, static_cast<size_t>(std::max(n_chunks_, 1)));
  std::atomic<int> failed{hipSuccess};
  // Waiting for an event keeps a core busy, so until the first chunk is there,
  // which is most of a frame's GPU time, only the caller does; the helpers sleep.
  std::mutex mu;
  std::condition_variable cv;
  bool first_seen = false;
  auto first_done = [&] {
    {
      std::lock_guard<std::mutex> g(mu);
      first_seen = true;
    }
    cv.notify_all();
  };
  // Chunks w, w + parts, ...: whole chunks, so that no two threads fault the
  // same (huge) page of the destination at once, and nobody touches bytes that
  // another thread copies.
  auto work = [&](size_t w) {
    for (size_t k = w; k < static_cast<size_t>(n_chunks_); k += parts)
      for_rows(planes, k * chunk_, std::min((k + 1) * chunk_, bytes_), [](uint8_t* d, size_t, size_t n) { touch(d, n); });
    if (w != 0) {
      std::unique_lock<std::mutex> g(mu);
      cv.wait(g, [&] { return first_seen; });
    }
    for (size_t k = w; k < static_cast<size_t>(n_chunks_); k += parts) {
      const hipError_t r = hipEventSynchronize(events_[k]);
      if (k == 0) first_done();
      if (r != hipSuccess) {
        failed.store(r);
        return;
      }
      for_rows(planes, k * chunk_, std::min((k + 1) * chunk_, bytes_),
               [&](uint8_t* d, size_t at, size_t n) { std::memcpy(d, pinned_ + at, n); });
    }
  };
  std::thread helpers[kMaxThreads];
  size_t started = 1;  // parts taken by the caller and the helpers
  for (; started < parts; ++started) {
    try {
      helpers[started] = std::thread([&, started] {
        const hipError_t r = hipSetDevice(device_);
        if (r != hipSuccess)
          failed.store(r);
        else
          work(started);
      });
    } catch (...) {
      break;  // no thread or no memory for one: the caller copies that part too
    }
  }
  work(0);
  for (size_t w = started; w < parts; ++w) work(w);
  for (std::thread& t : helpers)
    if (t.joinable()) t.join();
  const hipError_t r = static_cast<hipError_t>(failed.load());
  // Chunks that nobody waited for may still be on their way into the staging.
  if (r != hipSuccess) (void)hipStreamSynchronize(stream_);
  return r;
}

}  // namespace arthip
