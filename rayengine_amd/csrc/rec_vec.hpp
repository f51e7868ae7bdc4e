// Arrays of a tree's records.  resize() leaves new records uninitialised:
// every builder writes each record whole, and zeroing tens of megabytes first
// is a pass over memory that costs as much as the copy from the device.
#pragma once

#include <memory>
#include <utility>
#include <vector>

namespace re {

template <typename T>
struct DefaultInit : std::allocator<T> {
  template <typename U>
  struct rebind {
    using other = DefaultInit<U>;
  };
  DefaultInit() = default;
  template <typename U>
  DefaultInit(const DefaultInit<U>&) noexcept {}
  template <typename U>
  void construct(U* p) noexcept {
    ::new ((void*)p) U;
  }
  template <typename U, typename... A>
  void construct(U* p, A&&... a) {
    ::new ((void*)p) U(std::forward<A>(a)...);
  }
};

template <typename T>
using RecVec = std::vector<T, DefaultInit<T>>;

}  // namespace re
