// lbm_host_copy.hpp -- device results into the caller's ordinary host memory.
#pragma once
#include <hip/hip_runtime.h>

#include <mutex>

#include "lbm_internal.hpp"

namespace lbm {

// Pinned staging of one handle (24 MiB), allocated at its first large readback
// and freed with the handle.
struct HostStage {
  static constexpr int kBuffers = 3;
  static constexpr size_t kChunk = (size_t)8 << 20;
  char* pinned = nullptr;  // kBuffers chunks
  hipEvent_t ready[kBuffers] = {};
  std::mutex mu;           // one readback of a handle at a time
};
void free_stage(HostStage& s);

// Whether copy_to_host would stage a copy of this size.  Pinning the staging takes
// 4-5 ms, so only a large first copy pays for it (moments of a new handle, start
// -> staged: 100^3, 32 MB, 4.5 -> 9 ms; 128^3, 67 MB, 10.6 -> 5.3 ms).
inline bool worth_staging(const HostStage& s, size_t bytes) {
  return bytes >= (s.pinned ? (size_t)4 << 20 : (size_t)32 << 20);
}

// Copies `bytes` of device memory to `dst` after the work on `stream`, and waits.
// F32_TO_F64: the source is float, the destination double (twice the bytes).
enum class HostCopy { PLAIN, F32_TO_F64 };
hipError_t copy_to_host(HostStage& s, hipStream_t stream, void* dst, const void* src, size_t bytes,
                        HostCopy how = HostCopy::PLAIN);

}  // namespace lbm
