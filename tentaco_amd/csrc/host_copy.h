// Copies from the device to pageable host memory through pinned slabs.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <cstring>

#include "internal.h"

namespace tt {

// n words from src to dst, one of them in pinned host memory.
static __global__ __launch_bounds__(256) void stage_copy_kernel(const uint32_t* src, uint32_t* dst, int32_t n) {
  const int32_t tid = int32_t(blockIdx.x * 256 + threadIdx.x), nt = int32_t(gridDim.x * 256);
  const bool wide = ((reinterpret_cast<uintptr_t>(src) | reinterpret_cast<uintptr_t>(dst)) & 15) == 0;
  const int32_t n4 = wide ? n / 4 : 0;
  for (int32_t i = tid; i < n4; i += nt)
    reinterpret_cast<uint4*>(dst)[i] = reinterpret_cast<const uint4*>(src)[i];
  for (int32_t i = 4 * n4 + tid; i < n; i += nt) dst[i] = src[i];
}

// A pageable hipMemcpy from the device moves 17 GB/s here and takes 70 us however
// small it is; pinned memory moves at 50 GB/s. So a copy is cut into slabs of
// pinned memory, and the core empties one while the device fills others. The
// device fills a slab with stage_copy_kernel: a hipMemcpyAsync of 512 KB costs
// 24 us in a row of them (8 MB: 389 us), a kernel 12 (263). One core empties
// 512 KB in 16 us. Twelve factors of 0.3 to 3.8 MB and their weights, 22 MB:
// 1.86 -> 0.96 ms.
// The slabs (kSlabs x kSlab bytes) belong to the object that copies through
// them, which has to live for several copies (allocating them takes 0.1 ms, and
// several now and then), and are freed with it. Pinned or device operands, an
// object used from another device than its own, and a failed allocation take
// hipMemcpy. Sizes are in bytes, whole words.
class HostStage {
 public:
  HostStage() = default;
  HostStage(const HostStage&) = delete;
  HostStage& operator=(const HostStage&) = delete;
  ~HostStage() {
    if (!mem_) return;
    (void)drain();
    for (int i = 0; i < kSlabs; ++i)
      if (ev_[i]) (void)hipEventDestroy(ev_[i]);
    (void)hipHostFree(mem_);
  }

  // dst[0..n) = src[0..n) and, if given, dst2[0..n2) = src2[0..n2) (at most a
  // slab) behind it; returns when both are whole. The core reads a slab that the
  // device has written from memory, which bounds this (two threads emptying
  // slabs gained nothing over 22 MB in copies of 2).
  int to_host(void* dst, const void* src, size_t n, void* dst2 = nullptr, const void* src2 = nullptr,
              size_t n2 = 0) {
    if (n + n2 == 0) return TENTACO_OK;
    if (n2 > kSlab || !usable(n ? dst : dst2) || (n2 && !usable(dst2))) {
      if (n) TT_HIP_CHECK(hipMemcpy(dst, src, n, hipMemcpyDeviceToHost));
      if (n2) TT_HIP_CHECK(hipMemcpy(dst2, src2, n2, hipMemcpyDeviceToHost));
      return TENTACO_OK;
    }
    int rc = drain();
    if (rc) return rc;
    const size_t body = (n + kSlab - 1) / kSlab, chunks = body + (n2 ? 1 : 0);
    auto len = [&](size_t c) { return c < body ? std::min(kSlab, n - c * kSlab) : n2; };
    auto queue = [&](size_t c) -> int {
      const int i = int(c % kSlabs);
      const char* from = c < body ? static_cast<const char*>(src) + c * kSlab : static_cast<const char*>(src2);
      TT_HIP_CHECK(copy(slab(i), from, len(c)));
      TT_HIP_CHECK(hipEventRecord(ev_[i], nullptr));
      busy_[i] = true;
      return TENTACO_OK;
    };
    for (size_t c = 0; c < std::min<size_t>(chunks, kSlabs); ++c)
      if ((rc = queue(c))) return rc;
    for (size_t c = 0; c < chunks; ++c) {
      const int i = int(c % kSlabs);
      TT_HIP_CHECK(hipEventSynchronize(ev_[i]));
      busy_[i] = false;
      std::memcpy(c < body ? static_cast<char*>(dst) + c * kSlab : static_cast<char*>(dst2), slab(i), len(c));
      if (c + kSlabs < chunks && (rc = queue(c + kSlabs))) return rc;
    }
    return TENTACO_OK;
  }

  // Waits for the slabs that a failed copy left in flight.
  int drain() {
    for (int i = 0; i < kSlabs; ++i) {
      if (busy_[i]) TT_HIP_CHECK(hipEventSynchronize(ev_[i]));
      busy_[i] = false;
    }
    return TENTACO_OK;
  }

 private:
  static constexpr size_t kSlab = size_t(1) << 19;
  static constexpr int kSlabs = 4;

  hipError_t copy(void* dst, const void* src, size_t n) {
    stage_copy_kernel<<<64, 256, 0, nullptr>>>(static_cast<const uint32_t*>(src), static_cast<uint32_t*>(dst),
                                               int32_t(n / 4));
    return hipGetLastError();
  }

  char* slab(int i) { return mem_ + size_t(i) * kSlab; }

  // Whether a copy to `host` goes through the slabs.
  bool usable(const void* host) {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess) return false;
    if (!tried_) {
      tried_ = true;
      dev_ = dev;
      void* p = nullptr;
      if (hipHostMalloc(&p, kSlab * kSlabs, hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        return false;
      }
      mem_ = static_cast<char*>(p);
      for (int i = 0; i < kSlabs; ++i)
        if (hipEventCreateWithFlags(&ev_[i], hipEventDisableTiming) != hipSuccess) {
          (void)hipGetLastError();
          ev_[i] = nullptr;
          failed_ = true;
        }
    }
    if (!mem_ || failed_ || dev != dev_) return false;
    hipPointerAttribute_t at{};
    if (hipPointerGetAttributes(&at, host) != hipSuccess) {
      (void)hipGetLastError();
      return true;  // memory the runtime does not know
    }
    return at.type == hipMemoryTypeUnregistered;
  }

  char* mem_ = nullptr;
  hipEvent_t ev_[kSlabs] = {};
  bool busy_[kSlabs] = {};
  int dev_ = -1;
  bool tried_ = false, failed_ = false;
};

}  // namespace tt
