// The window of a pass that runs over its paths or samples in windows.
#pragma once
#include <cstdint>

namespace trc {

// A window of 4,096 paths needs half a megabyte: below that the launches cost
// more than memory could.
constexpr uint64_t kMinWindow = 4096;

struct Window {
  void* ptr = nullptr;  // null: no window fits
  uint64_t size = 0;
  bool kept = false;
};

// The largest of the windows first, first / 2, ... (multiples of 64) that
// needs no more memory than there is: kept_bytes at `kept` (or null), or what
// alloc(bytes) can give (null when it cannot; asked only with may_alloc).
// bytes(w): the need of windows of w.
template <class Bytes, class Alloc>
Window fit_window(uint64_t first, Bytes&& bytes, void* kept, uint64_t kept_bytes, bool may_alloc, Alloc&& alloc) {
  Window w;
  for (w.size = first;; w.size = (w.size / 2 + 63) / 64 * 64) {
    const uint64_t need = bytes(w.size);
    w.kept = kept && need <= kept_bytes;
    w.ptr = w.kept ? kept : may_alloc ? alloc(need) : nullptr;
    if (w.ptr || w.size <= kMinWindow) return w;
  }
}

}  // namespace trc
