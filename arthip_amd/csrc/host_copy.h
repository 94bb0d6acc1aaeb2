// Device-to-host download of a frame through pinned staging, copied out to the
// caller's rows as it arrives.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <vector>

namespace arthip {

// Transfers up to this size go by a copy kernel on the launch stream between
// pinned and device memory: a copy engine's start and the waits between its
// stream and the kernels cost more than the bytes (through the filter, copy
// streams and kernels with everything else alike: C4F32 at 96x128 85 -> 51 us a
// frame, at 270x480 140 -> 119, the shipped architecture at 270x480 454 -> 424).
constexpr size_t kKernelCopyBytes = static_cast<size_t>(1) << 20;
// The filter's limit for uploads while other frames are in flight.
constexpr size_t kSharedKernelUploadBytes = static_cast<size_t>(256) << 10;

// `rows` rows of `row` bytes, `stride` bytes apart, of the caller's memory.
struct HostRows {
  uint8_t* base;
  ptrdiff_t stride;
  size_t row;
  int rows;
};

// One download in flight. Enqueue sends it in chunks with an event after each;
// CopyOut waits for the chunks in order and copies each out while the next ones
// travel. The copy out of memory that the GPU has just written runs at about
// half the link's rate on one thread, and the first write to a fresh
// destination page faults, so larger frames are shared with up to three helper
// threads, which touch the destination and then sleep while the GPU still works;
// they end with the call. Through the filter, one chunk on the caller's thread
// against this: one caller, C4F32 at 1080p (16.6 MB out) 1130 -> 790 us a frame,
// R8F64 there 2700 -> 2370, the shipped architecture at 720p (7.4 MB out) 1830 ->
// 1720; two callers, C4F32 610 -> 425, R8F64 the same (1790). CPU time a frame
// grows by the helpers: R8F64 3.0 -> 3.7 ms, with two callers 3.9 -> 4.9.
class ChunkedDownload {
 public:
  ChunkedDownload() = default;
  ChunkedDownload(const ChunkedDownload&) = delete;
  ChunkedDownload& operator=(const ChunkedDownload&) = delete;
  ~ChunkedDownload();

  // Both wait for the stream before they report a failure, so that no chunk
  // still writes the staging, which the caller may then reuse or free.
  hipError_t Enqueue(int device, hipStream_t s, void* pinned, const void* dev, size_t bytes);
  // The staged bytes are the planes' rows, plane after plane. Blocks until they
  // are all copied; on failure the destination's content is unspecified.
  hipError_t CopyOut(const std::vector<HostRows>& planes);

 private:
  hipError_t Send(int device, hipStream_t s, void* pinned, const void* dev, size_t bytes);

  std::vector<hipEvent_t> events_;
  int device_ = 0;
  hipStream_t stream_ = nullptr;
  const uint8_t* pinned_ = nullptr;
  size_t bytes_ = 0, chunk_ = 0;
  int n_chunks_ = 0;
};

}  // namespace arthip
