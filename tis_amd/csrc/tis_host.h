// Host-side pieces of a context that need no device: C++ only, so that they
// can be tested without one.
#pragma once
#include <algorithm>
#include <cstddef>

namespace tis {

// One block of pinned host memory that kernels read and write themselves: a
// report of two words, a ring that calls' inputs are copied into, and the
// outputs of a call that waits for them.
struct PinBlock {
  static constexpr size_t kHead = 256, kSmall = 64 << 10;
  char *base = nullptr;
  size_t in_cap = 0, in_at = 0, out_cap = 0;

  unsigned long long *report() const { return (unsigned long long *)base; }
  char *in() const { return base + kHead; }
  char *out() const { return base + kHead + in_cap; }
  bool holds(size_t in_bytes, size_t out_bytes) const { return base && in_bytes <= in_cap && out_bytes <= out_cap; }

  // At least in_bytes of ring and out_bytes of output (64 KB in all if that is
  // enough), with nothing under way in the present block.  Returns 0, or the
  // size that alloc had no memory for: the present block then stays as it is.
  template <class Alloc, class Free>
  size_t grow(size_t in_bytes, size_t out_bytes, Alloc alloc, Free release) {
    size_t in_new = std::max((in_bytes + 255) & ~(size_t)255, in_cap);
    const size_t out_new = std::max((out_bytes + 255) & ~(size_t)255, out_cap);
    if (kHead + in_new + out_new < kSmall) in_new = kSmall - kHead - out_new;
    char *p = (char *)alloc(kHead + in_new + out_new);
    if (!p) return kHead + in_new + out_new;
    if (base) release(base);
    base = p;
    in_cap = in_new;
    in_at = 0;
    out_cap = out_new;
    report()[0] = report()[1] = 0;
    return 0;
  }
};

}  // namespace tis
