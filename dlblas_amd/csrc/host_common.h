// Host-side helpers shared by the translation units of the library.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include <mutex>

namespace dlb {

// Records the thread-local message dlb_last_error() returns and hands `code` back (defined in dlblas_fp8_gemm.hip).
int fail(int code, const char* fmt, ...) __attribute__((format(printf, 2, 3)));
void clear_error();

// Compute units of the current device (cached per device); -1 if hipGetDevice fails.  *dev_out = device ordinal.
int device_cu_count(int* dev_out);

// A call that goes through a workspace enqueues several kernels that hand data on in it, so the launches of two threads on one
// stream must not interleave.  One lock per workspace address, out of a fixed set (an address keeps its lock; two may share
// one).  Recursive: dlb_workspace_lock() holds it over several calls.
inline std::recursive_mutex& workspace_mutex(const void* workspace) {
  static std::recursive_mutex locks[64];
  return locks[(reinterpret_cast<uintptr_t>(workspace) >> 8) * 0x9E3779B97F4A7C15ull >> 58];
}
class WorkspaceLock {
 public:
  explicit WorkspaceLock(const void* workspace) : m_(workspace ? &workspace_mutex(workspace) : nullptr) {
    if (m_) m_->lock();
  }
  ~WorkspaceLock() {
    if (m_) m_->unlock();
  }
  WorkspaceLock(const WorkspaceLock&) = delete;
  WorkspaceLock& operator=(const WorkspaceLock&) = delete;

 private:
  std::recursive_mutex* m_;
};

inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }
inline bool misaligned(const void* ptr, size_t a) { return (reinterpret_cast<uintptr_t>(ptr) & (a - 1)) != 0; }

}  // namespace dlb
