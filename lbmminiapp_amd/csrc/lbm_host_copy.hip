// lbm_host_copy.hip -- staged, threaded copy of device results to host memory.
//
// A readback goes to memory the caller has just allocated: its pages do not
// exist yet, and the runtime's copy to pageable memory faults them in and copies
// on one thread, at 9 GB/s (512^3 moments, 4.3 GB: 0.46 s, as long as 100 time
// steps).  Here a kernel of a few workgroups writes chunks into pinned memory
// (48 GB/s over PCIe; the DMA engine reached 28) and threads move them on, so
// that page faults and copies run in parallel and beside the transfer.  Moments
// of FP64 boxes, runtime's copy -> staged: 128^3 5.9 -> 1.9 ms, 256^3 58 -> 12 ms,
// 384^3 38 ms (48 GB/s; 4 threads: 38 GB/s, 16: no more).
#include "lbm_host_copy.hpp"

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstdint>
#include <cstring>
#include <memory>
#include <new>
#include <thread>

namespace lbm {

// Device to pinned host memory, 16 bytes a lane, then the last few bytes.  The
// source is aligned to its elements only (moments start at ncell doubles), which
// 16-byte loads from global memory allow; the pinned chunks are aligned.
__global__ void __launch_bounds__(256)
    k_to_pinned(const char* __restrict__ src, char* __restrict__ dst, size_t bytes) {
  using v4 = unsigned int __attribute__((ext_vector_type(4)));
  typedef unsigned int v4_by4 __attribute__((ext_vector_type(4), aligned(4)));
  const size_t n16 = bytes / 16, t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  for (size_t i = t; i < n16; i += (size_t)gridDim.x * blockDim.x)
    __builtin_nontemporal_store((v4)__builtin_nontemporal_load(reinterpret_cast<const v4_by4*>(src) + i),
                                reinterpret_cast<v4*>(dst) + i);
  if (t < bytes % 16) dst[n16 * 16 + t] = src[n16 * 16 + t];
}

namespace {

constexpr size_t kPiece = (size_t)1 << 20;  // what a thread moves at a time
constexpr size_t kThreads = 8;
constexpr unsigned kBlocks = 16;  // workgroups of the copy kernel: enough for the link

// `n` source bytes at offset `at`; src holds them, dst is the whole destination
void move_piece(char* dst, const char* src, size_t at, size_t n, HostCopy how) {
  if (how == HostCopy::PLAIN) {
    std::memcpy(dst + at, src, n);
    return;
  }
  const float* f = reinterpret_cast<const float*>(src);
  double* d = reinterpret_cast<double*>(dst) + at / sizeof(float);
  for (size_t i = 0; i < n / sizeof(float); i++) d[i] = f[i];
}

hipError_t prepare_stage(HostStage& s) {
  if (s.pinned) return hipSuccess;
  for (hipEvent_t& e : s.ready)
    if (!e)
      if (hipError_t err = hipEventCreateWithFlags(&e, hipEventDisableTiming)) return err;
  void* p = nullptr;
  const hipError_t err = hipHostMalloc(&p, HostStage::kBuffers * HostStage::kChunk, hipHostMallocDefault);
  if (err == hipSuccess) s.pinned = static_cast<char*>(p);
  return err;
}

// The runtime's copy, for small results and where there is no staging.
hipError_t copy_direct(hipStream_t stream, char* dst, const char* src, size_t bytes, HostCopy how) {
  if (how == HostCopy::PLAIN) {
    const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, stream);
    return e == hipSuccess ? hipStreamSynchronize(stream) : e;
  }
  std::unique_ptr<char[]> tmp(new (std::nothrow) char[std::min(bytes, HostStage::kChunk)]);
  if (!tmp) return hipErrorOutOfMemory;
  for (size_t at = 0; at < bytes; at += HostStage::kChunk) {
    const size_t n = std::min(HostStage::kChunk, bytes - at);
    hipError_t e = hipMemcpyAsync(tmp.get(), src + at, n, hipMemcpyDeviceToHost, stream);
    if (e == hipSuccess) e = hipStreamSynchronize(stream);
    if (e != hipSuccess) return e;
    move_piece(dst, tmp.get(), at, n, how);
  }
  return hipSuccess;
}

// The transfer's progress, shared by the threads that move pieces.
struct Progress {
  std::mutex mu;
  std::condition_variable cv;
  size_t arrived = 0;                      // chunks that are in pinned memory
  size_t moved[HostStage::kBuffers] = {};  // bytes moved out of each buffer's chunk
  bool stop = false;
};

}  // namespace

void free_stage(HostStage& s) {
  if (s.pinned) (void)hipHostFree(s.pinned);
  s.pinned = nullptr;
  for (hipEvent_t& e : s.ready) {
    if (e) (void)hipEventDestroy(e);
    e = nullptr;
  }
}

hipError_t copy_to_host(HostStage& s, hipStream_t stream, void* dst_, const void* src_, size_t bytes,
                        HostCopy how) {
  constexpr size_t B = HostStage::kBuffers, C = HostStage::kChunk;
  char* dst = static_cast<char*>(dst_);
  const char* src = static_cast<const char*>(src_);
  std::lock_guard<std::mutex> one(s.mu);
  if (!worth_staging(s, bytes)) return copy_direct(stream, dst, src, bytes, how);
  if (prepare_stage(s) != hipSuccess) {
    (void)hipGetLastError();
    return copy_direct(stream, dst, src, bytes, how);
  }
  const size_t chunks = (bytes + C - 1) / C;
  Progress pr;
  std::atomic<size_t> next{0};
  auto work = [&]() {
    for (;;) {
      const size_t at = next.fetch_add(kPiece);
      if (at >= bytes) return;
      const size_t k = at / C, n = std::min(kPiece, bytes - at);
      {
        std::unique_lock<std::mutex> l(pr.mu);
        pr.cv.wait(l, [&] { return pr.arrived > k || pr.stop; });
        if (pr.stop) return;
      }
      move_piece(dst, s.pinned + k % B * C + at % C, at, n, how);
      std::lock_guard<std::mutex> l(pr.mu);
      pr.moved[k % B] += n;
      pr.cv.notify_all();
    }
  };
  std::thread pool[kThreads];
  size_t started = 0;
  try {
    const size_t cpus = std::max(1u, std::thread::hardware_concurrency());
    for (; started < std::min(kThreads, cpus); started++) pool[started] = std::thread(work);
  } catch (...) {  // the threads there are will do
  }
  if (!started) return copy_direct(stream, dst, src, bytes, how);
  hipError_t err = hipSuccess;
  for (size_t k = 0; k <= chunks && err == hipSuccess; k++) {
    if (k < chunks) {
      if (k >= B) {  // until the buffer's last chunk has been moved on
        std::unique_lock<std::mutex> l(pr.mu);
        pr.cv.wait(l, [&] { return pr.moved[k % B] == C; });
        pr.moved[k % B] = 0;
      }
      hipLaunchKernelGGL(k_to_pinned, dim3(kBlocks), dim3(256), 0, stream, src + k * C,
                         s.pinned + k % B * C, std::min(C, bytes - k * C));
      err = hipGetLastError();
      if (err == hipSuccess) err = hipEventRecord(s.ready[k % B], stream);
    }
    if (k > 0 && err == hipSuccess) {
      err = hipEventSynchronize(s.ready[(k - 1) % B]);
      std::lock_guard<std::mutex> l(pr.mu);
      if (err == hipSuccess) pr.arrived = k;
      pr.cv.notify_all();
    }
  }
  if (err != hipSuccess) {
    {
      std::lock_guard<std::mutex> l(pr.mu);
      pr.stop = true;
      pr.cv.notify_all();
    }
    (void)hipStreamSynchronize(stream);  // nothing writes to the staging any more
  }
  for (size_t i = 0; i < started; i++) pool[i].join();
  return err;
}

}  // namespace lbm
