// Host-side helpers shared by the C-ABI entry points (see include/dryft_decode.h).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <atomic>
#include "../../include/dryft_decode.h"

#define DD_API extern "C" __attribute__((visibility("default")))

namespace dd {

constexpr int DD_ABI_VERSION = 17;

inline bool aligned16(const void* p) { return (((uintptr_t)p) & 15u) == 0; }

// Launch result: the error of the last launch on this thread (0 when it went through).
inline int launch_status() { return (int)hipGetLastError(); }

// Compute units of the current device (0 when it cannot be asked), remembered per device.
inline int cu_count() {
  static std::atomic<int> known[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
  int n = known[dev].load(std::memory_order_relaxed);
  if (n == 0) {
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
    known[dev].store(n, std::memory_order_relaxed);
  }
  return n;
}

// Lets a kernel use `bytes` of dynamic LDS on the current device; `done` (one per kernel) holds the
// devices where that has been set.
inline hipError_t allow_lds(const void* kernel, int bytes, std::atomic<unsigned long long>& done) {
  int dev = 0;
  const hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  const unsigned long long bit = 1ull << (dev & 63);
  if (done.load(std::memory_order_relaxed) & bit) return hipSuccess;
  const hipError_t r = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  if (r == hipSuccess) done.fetch_or(bit, std::memory_order_relaxed);
  return r;
}

// GEMV launch helpers (gemv.hip): split-K choice, k per split, workspace size, and the launch
// (h != nullptr selects the residual + RMSNorm epilogue; returns the number of splits).
int pick_splitk(int M, int N, int K);
int kps_for(int K, int sk);
int gemv_nsplit(int K, int sk);
size_t gemv_ws_floats(int M, int N, int K, int sk, bool add_rms);
int launch_gemv(const void* x, const void* W, void* y, void* ws, int* counters, int M, int N,
                int K, int sk, const void* h, const void* lnw, void* hn, float eps,
                hipStream_t stream);

// Residual add + RMSNorm of a product left as S fp32 sums [S][M][N] (norm.hip; N <= 4096).
int launch_sum_add_rmsnorm(const void* part, int S, const void* h, const void* w, void* hn, void* y, int M, int N,
                           float eps, hipStream_t stream);

}  // namespace dd

#define DD_REQUIRE(cond)                         \
  do {                                           \
    if (!(cond)) return (int)hipErrorInvalidValue; \
  } while (0)
