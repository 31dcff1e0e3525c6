// Memory that a handle keeps between calls: device workspaces, given back where an allocation of any handle
// finds no room, and pinned buffers.
#pragma once
#include <hip/hip_runtime.h>
#include <cstddef>
#include <mutex>
#include <vector>

namespace cvr {

// Workspaces that lie idle, by the pointers that hold them.  A handle claims its workspace before it uses it
// (it may be gone by then) and parks it afterwards; work that is queued on it may still run.
struct IdleWork {
  void** p;
  size_t* bytes;
  int device;
};
struct IdleList {
  std::mutex mu;
  std::vector<IdleWork> list;
};
inline IdleList& idle_work() {
  static IdleList& l = *new IdleList;  // until the process ends: handles may outlive static objects
  return l;
}
inline void claim_work(void** p) {
  IdleList& l = idle_work();
  std::lock_guard<std::mutex> lock(l.mu);
  for (size_t i = 0; i < l.list.size(); ++i)
    if (l.list[i].p == p) {
      l.list.erase(l.list.begin() + i);
      return;
    }
}
inline void park_work(void** p, size_t* bytes, int device) {
  if (!*p) return;
  IdleList& l = idle_work();
  std::lock_guard<std::mutex> lock(l.mu);
  l.list.push_back(IdleWork{p, bytes, device});
}

// hipMalloc on the current device; where it fails, once more without the device's idle workspaces (hipFree
// waits for the work queued on them).
template <class T> inline hipError_t device_alloc(T** p, size_t bytes) {
  void* q = nullptr;
  hipError_t e = hipMalloc(&q, bytes);
  int dev = -1;
  if (e != hipSuccess && hipGetDevice(&dev) == hipSuccess) {
    bool freed = false;
    IdleList& l = idle_work();
    std::lock_guard<std::mutex> lock(l.mu);
    for (size_t i = l.list.size(); i-- > 0;)
      if (l.list[i].device == dev) {
        (void)hipFree(*l.list[i].p);
        *l.list[i].p = nullptr;
        *l.list[i].bytes = 0;
        l.list.erase(l.list.begin() + i);
        freed = true;
      }
    if (freed) {
      (void)hipGetLastError();
      e = hipMalloc(&q, bytes);
    }
  }
  *p = e == hipSuccess ? static_cast<T*>(q) : nullptr;
  return e;
}

// A pinned buffer of at least `bytes`, which only grows; null where there is none to be had.
template <class T> inline T* pinned_buffer(T** p, size_t* have, size_t bytes) {
  if (*p && *have >= bytes) return *p;
  if (*p) (void)hipHostFree(*p);
  void* q = nullptr;
  const bool ok = hipHostMalloc(&q, bytes, hipHostMallocDefault) == hipSuccess;
  if (!ok) (void)hipGetLastError();
  *p = ok ? static_cast<T*>(q) : nullptr;
  *have = ok ? bytes : 0;
  return *p;
}

}  // namespace cvr
