// Host copies of large inputs.  A dense matrix keeps its values on the host; a
// plain vector writes them twice (zeros, then the copy) and faults 4 KB pages one
// by one on a single thread, longer than the device takes for a few rounds
// (262,144 x 64: 67 MB, some 8 ms; 1.7 ms by copy_large on large pages).
#pragma once
#include <sys/mman.h>

#include <algorithm>
#include <cstddef>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <new>
#include <thread>
#include <utility>
#include <vector>

namespace mgb {

// Leaves new elements uninitialized (resize), and asks for 2 MB pages from
// kLarge bytes on.
template <typename T>
struct HostAllocator {
  using value_type = T;
  static constexpr size_t kLarge = size_t(4) << 20, kPage = size_t(2) << 20;
  HostAllocator() = default;
  template <typename U>
  HostAllocator(const HostAllocator<U>&) {}

  T* allocate(size_t n) {
    if (n > (SIZE_MAX - kPage) / sizeof(T)) throw std::bad_alloc();
    const size_t bytes = n * sizeof(T);
    void* p = nullptr;
    if (bytes < kLarge) {
      p = std::malloc(bytes ? bytes : 1);
    } else {
      const size_t whole = (bytes + kPage - 1) / kPage * kPage;
      p = std::aligned_alloc(kPage, whole);
      if (p) (void)madvise(p, whole, MADV_HUGEPAGE);  // advice: 4 KB pages where it is not taken
    }
    if (!p) throw std::bad_alloc();
    return static_cast<T*>(p);
  }
  void deallocate(T* p, size_t) { std::free(p); }
  template <typename U>
  void construct(U* p) { ::new (static_cast<void*>(p)) U; }
  template <typename U, typename... Args>
  void construct(U* p, Args&&... args) { ::new (static_cast<void*>(p)) U(std::forward<Args>(args)...); }
  template <typename U>
  bool operator==(const HostAllocator<U>&) const { return true; }
  template <typename U>
  bool operator!=(const HostAllocator<U>&) const { return false; }
};

using HostFloats = std::vector<float, HostAllocator<float>>;

// memcpy, from 8 MB on over up to eight threads: first touches of the
// destination's pages are what it waits for.  A thread that cannot be started
// leaves its share to the caller.
inline void copy_large(void* dst, const void* src, size_t bytes) {
  constexpr size_t kShare = size_t(4) << 20;
  size_t n = std::min(bytes / kShare, size_t(8));
  if (n > 1) n = std::min(n, (size_t)std::max(1u, std::thread::hardware_concurrency()));  // a system call
  if (n <= 1) {
    if (bytes) std::memcpy(dst, src, bytes);
    return;
  }
  auto share = [=](size_t k) {
    const size_t begin = bytes / n * k, end = k + 1 == n ? bytes : bytes / n * (k + 1);
    std::memcpy(static_cast<char*>(dst) + begin, static_cast<const char*>(src) + begin, end - begin);
  };
  std::vector<std::thread> workers;
  workers.reserve(n);
  size_t k = 1;
  try {
    for (; k < n; ++k) workers.emplace_back(share, k);
  } catch (...) {
  }
  share(0);
  for (; k < n; ++k) share(k);
  for (auto& w : workers) w.join();
}

}  // namespace mgb
