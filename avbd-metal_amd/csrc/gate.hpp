// gate.hpp -- graph captures kept apart from calls on the default stream.
//
// A synchronous copy or fill, an allocation or a free in any thread ends the
// captures under way in the process, whatever their mode and stream, and fails
// itself.  A solver captures when its frames first take a form -- also in the
// middle of a run, beside another solver's frames -- while other threads create
// solvers or read and write states.  So the library makes those calls through
// here, and a capture waits for the ones under way and holds back the next.
#pragma once
#include <hip/hip_runtime.h>

#include <mutex>
#include <shared_mutex>

namespace avbd {

inline std::shared_mutex& capture_gate() {
  static std::shared_mutex* m = new std::shared_mutex();  // outlives every handle
  return *m;
}
// held from the begin of a capture to its end
struct CaptureApart {
  std::unique_lock<std::shared_mutex> lock{capture_gate()};
};

inline hipError_t copy_now(void* to, const void* from, size_t bytes, hipMemcpyKind kind) {
  std::shared_lock<std::shared_mutex> g(capture_gate());
  return hipMemcpy(to, from, bytes, kind);
}
inline hipError_t fill_now(void* to, int byte, size_t bytes) {
  std::shared_lock<std::shared_mutex> g(capture_gate());
  return hipMemset(to, byte, bytes);
}
template <typename T>
hipError_t alloc_now(T** p, size_t bytes) {
  std::shared_lock<std::shared_mutex> g(capture_gate());
  return hipMalloc((void**)p, bytes);
}
inline hipError_t free_now(void* p) {
  std::shared_lock<std::shared_mutex> g(capture_gate());
  return hipFree(p);
}
template <typename T>
hipError_t alloc_host_now(T** p, size_t bytes, unsigned flags) {
  std::shared_lock<std::shared_mutex> g(capture_gate());
  return hipHostMalloc((void**)p, bytes, flags);
}
inline hipError_t free_host_now(void* p) {
  std::shared_lock<std::shared_mutex> g(capture_gate());
  return hipHostFree(p);
}

}  // namespace avbd
