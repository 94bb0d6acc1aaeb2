// ChunkedDownload (host_copy.cc) on a simulated HIP runtime: transfers sent to a
// stream land only when something waits for them. Each scenario makes one call
// fail; the download must not report the failure while a chunk that was sent
// could still write the staging buffer. argv[1]: scenario.
#include <chrono>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

#include "host_copy.h"

namespace {

struct Copy {
  void* dst;
  const void* src;
  size_t n;
};

std::mutex mu;
std::vector<Copy> queued;  // in stream order, from `landed` on still under way
size_t landed = 0;
std::vector<size_t> recorded;  // per event: copies queued before its record
int copies_sent = 0;
int fail_copy = -1;
size_t fail_event = 0;  // 1-based, as handed out
bool fail_device = false;
bool slow_frame = false;  // the frame takes a while until its first chunk is there
int early_waits = 0;      // waits for later chunks begun before that

void land(size_t upto) {
  for (; landed < upto; ++landed) std::memcpy(queued[landed].dst, queued[landed].src, queued[landed].n);
}

}  // namespace

extern "C" {

hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  std::lock_guard<std::mutex> g(mu);
  recorded.push_back(0);
  *e = reinterpret_cast<hipEvent_t>(recorded.size());
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  std::lock_guard<std::mutex> g(mu);
  if (copies_sent++ == fail_copy) return hipErrorUnknown;
  queued.push_back(Copy{d, s, n});
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
  std::lock_guard<std::mutex> g(mu);
  recorded[reinterpret_cast<size_t>(e) - 1] = queued.size();
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  if (slow_frame && reinterpret_cast<size_t>(e) == 1) std::this_thread::sleep_for(std::chrono::milliseconds(300));
  std::lock_guard<std::mutex> g(mu);
  if (reinterpret_cast<size_t>(e) != 1 && !landed) ++early_waits;
  if (reinterpret_cast<size_t>(e) == fail_event) return hipErrorUnknown;
  land(recorded[reinterpret_cast<size_t>(e) - 1]);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
  std::lock_guard<std::mutex> g(mu);
  land(queued.size());
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return fail_device ? hipErrorInvalidDevice : hipSuccess; }

}  // extern "C"

int main(int argc, char** argv) {
  const std::string what = argc > 1 ? argv[1] : "ok";
  const size_t bytes = (static_cast<size_t>(9) << 20) + 4242;  // four chunks
  std::vector<uint8_t> dev(bytes), pinned(bytes), out(bytes);
  for (size_t i = 0; i < bytes; ++i) dev[i] = static_cast<uint8_t>(i * 131 + (i >> 12));
  if (what == "copy") fail_copy = 2;
  if (what == "first_wait") fail_event = 1;
  if (what == "last_wait") fail_event = 4;
  slow_frame = what == "slow";
  fail_device = what == "device";  // in the helper threads

  arthip::ChunkedDownload d;
  hipStream_t s = reinterpret_cast<hipStream_t>(&queued);
  hipError_t e = d.Enqueue(0, s, pinned.data(), dev.data(), bytes);
  // One plane of 1021-byte rows, 1100 apart, and the remaining bytes as another.
  const size_t row = 1021;
  const int rows = static_cast<int>(bytes / row);
  const size_t rest = bytes - row * rows;
  std::vector<uint8_t> strided(static_cast<size_t>(rows) * 1100);
  if (e == hipSuccess)
    e = d.CopyOut({arthip::HostRows{strided.data(), 1100, row, rows},
                   arthip::HostRows{out.data(), static_cast<ptrdiff_t>(rest), rest, 1}});
  std::printf("status %d queued %zu landed %zu\n", static_cast<int>(e), queued.size(), landed);
  if (e != hipSuccess) return landed == queued.size() ? 2 : 1;
  if (slow_frame && early_waits != 0) return 1;
  for (int y = 0; y < rows; ++y)
    if (std::memcmp(&strided[static_cast<size_t>(y) * 1100], &dev[y * row], row) != 0) return 1;
  return std::memcmp(out.data(), &dev[rows * row], rest) == 0 ? 0 : 1;
}
