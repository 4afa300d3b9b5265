// Host-side pieces of a context that need no device: C++ only, so that they
// can be tested without one.
#pragma once
#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <functional>
#include <queue>
#include <vector>

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

// Whether a batch that fits k_window runs faster by it than by per-step
// launches.  k_window takes one workgroup per CU (its registers), so a batch
// takes as many turns as its workgroups, in launch order, need on 256 CUs; the
// per-step launches have a fixed latency and then fill the chip.  Both sides
// by lines through what they measured: us a step with a rebuild every ten
// steps, k_window / per-step launches,
//   beads        1 system      256        512       1,024       2,048
//    95         9.1 / 13.1   9.4 / 17.5  18 / 23   36 / 31     73 / 49
//   191        10.1 / 13.2  10.7 / 22.6  20 / 28   41 / 44     81 / 73
//   254        14.7 / 15.8  15.2 / 26.8  30 / 35   60 / 60    120 / 115
//   386        20.4 / 16.0  21.6 / 31.0  42 / 47   83 / 81    165 / 184
// Batches with valence-limited systems always take k_window: a per-step launch
// waits for the longest of their passes (119 beads: 34 / 93 at 256 systems, 204
// / 300 at 2,048; 59 beads: 15 / 32 and 118 / 99).  Under the displacement trigger
// every step has a list launch in front: 128 chains of up to 389 beads 21 / 27,
// with a fixed interval 24 / 20.
struct WindowLoad {
  int32_t beads, chunk_pairs;   // chunk pairs of 64 charges
};

inline bool window_pays(const std::vector<WindowLoad> &batch, bool valence_limited, bool trigger) {
  constexpr size_t kCus = 256;
  if (valence_limited) return true;
  std::priority_queue<double, std::vector<double>, std::greater<double>> cu;   // when each CU is free
  double window = 0.0, beads = 0.0;
  int32_t pairs = 0;
  for (const WindowLoad &w : batch) {
    double at = 0.0;
    if (cu.size() == kCus) { at = cu.top(); cu.pop(); }
    at += 6.8 + 0.02 * w.beads + 1.6 * std::max(w.chunk_pairs - 1, 0);
    cu.push(at);
    window = std::max(window, at);
    beads += w.beads;
    pairs = std::max(pairs, w.chunk_pairs);
  }
  // (from some 400,000 beads on a step's data no longer stay in the L2 caches)
  double launches = (pairs > 1 ? 15.7 : 13.5) + 0.16e-3 * std::min(beads, 4e5) + 0.25e-3 * std::max(beads - 4e5, 0.0);
  if (trigger) launches += 4.0 + 0.07e-3 * beads;
  return 0.97 * window < launches;   // (equal within the lines' errors: k_window)
}

}  // namespace tis
