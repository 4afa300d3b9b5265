"""CPU tests of the context's host-only pieces (tis_amd/csrc/tis_host.h),
compiled with the host compiler."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tis_amd", "csrc")


def _run(tmp_path, body):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text('#include "tis_host.h"\n#include <cstdio>\n#include <cstdlib>\n#include <cstring>\n'
                   "using namespace tis;\n#define CHECK(x) do { if (!(x)) { std::printf(\"line %d: %s\\n\", __LINE__, #x);"
                   " return 1; } } while (0)\nint main() {\n" + body + "\nreturn 0;\n}\n")
    res = subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", CSRC, str(src), "-o", str(exe)],
                         capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0, res.stdout


def test_pinned_block_survives_a_failed_growth(tmp_path):
    """A larger block is had before the old one is given back: when there is
    no memory for it, the report, the ring and the outputs stay usable."""
    _run(tmp_path, r"""
  PinBlock b;
  int live = 0;
  bool full = false;
  auto get = [&](size_t n) -> void * { if (full) return nullptr; ++live; return std::malloc(n); };
  auto put = [&](void *p) { --live; std::free(p); };
  CHECK(!b.holds(0, 0));
  full = true;
  CHECK(b.grow(1, 1, get, put) != 0 && b.base == nullptr && !b.holds(0, 0));
  full = false;
  CHECK(b.grow(100, 1000, get, put) == 0 && live == 1);
  CHECK(b.holds(100, 1000) && PinBlock::kHead + b.in_cap + b.out_cap == PinBlock::kSmall);
  CHECK(b.report()[0] == 0 && b.report()[1] == 0);
  b.report()[0] = 7;
  b.in_at = 512;
  std::memset(b.in(), 1, b.in_cap);
  std::memset(b.out(), 2, b.out_cap);
  char *old = b.base;
  const size_t in = b.in_cap, out = b.out_cap;
  full = true;
  CHECK(b.grow(1 << 20, 1 << 20, get, put) == PinBlock::kHead + (2u << 20));
  CHECK(live == 1 && b.base == old && b.in_cap == in && b.out_cap == out && b.in_at == 512);
  CHECK(b.report()[0] == 7 && b.in()[in - 1] == 1 && b.out()[out - 1] == 2);
  full = false;
  CHECK(b.grow(0, 1 << 20, get, put) == 0 && live == 1);
  CHECK(b.in_cap >= in && b.out_cap >= (1u << 20) && b.in_at == 0 && b.report()[0] == 0);
  std::memset(b.base, 3, PinBlock::kHead + b.in_cap + b.out_cap);
  put(b.base);
""")


def test_window_rule_takes_the_faster_side(tmp_path):
    """Both sides measured (us a step, k_window and per-step launches) for
    batches of equal chains; where they differ by more than a tenth, the rule
    takes the faster one.  Mixed batches lie between."""
    # beads, chunk pairs, systems, k_window, per-step launches
    rows = [(95, 1, 1, 9.1, 13.1), (95, 1, 256, 9.4, 17.5), (95, 1, 512, 18.4, 23.1), (95, 1, 513, 27.2, 23.7),
            (95, 1, 1024, 36.5, 30.8), (95, 1, 1536, 54.7, 40.3), (95, 1, 2048, 73.0, 49.1),
            (95, 1, 4096, 145.6, 85.9),
            (128, 1, 1, 9.3, 13.1), (128, 1, 512, 19.2, 24.1), (128, 1, 1024, 38.0, 32.5), (128, 1, 2048, 75.6, 53.8),
            (191, 1, 1, 10.1, 13.2), (191, 1, 256, 10.7, 22.6), (191, 1, 512, 20.5, 28.5), (191, 1, 768, 30.7, 36.2),
            (191, 1, 2048, 81.4, 72.6),
            (254, 3, 256, 15.2, 26.8), (254, 3, 512, 30.1, 35.0), (254, 3, 513, 44.6, 37.2),
            (320, 3, 256, 17.4, 28.7), (320, 3, 512, 33.8, 41.1), (320, 3, 2048, 134.4, 148.3),
            (386, 3, 1, 20.4, 16.0), (386, 3, 256, 21.6, 31.0), (386, 3, 2048, 165.4, 184.2)]
    body = "std::vector<WindowLoad> b;\n"
    for beads, pairs, n, win, step in rows:
        assert abs(win - step) > 0.09 * min(win, step)
        body += f"b.assign({n}, WindowLoad{{{beads}, {pairs}}}); CHECK(window_pays(b, false, false) == {int(win < step)});\n"
    body += """
  for (int n : {1, 300, 5000}) { b.assign(n, WindowLoad{119, 1}); CHECK(window_pays(b, true, false)); }
  // one long chain holds no batch of short ones back, nor 255 short ones a long one
  b.assign(255, WindowLoad{95, 1});
  b.insert(b.begin(), WindowLoad{320, 3});
  CHECK(window_pays(b, false, false));
  // 128 chains of up to 389 beads (24 / 20 us; 21 / 27 under the trigger)
  b.assign(127, WindowLoad{190, 1});
  b.insert(b.begin(), WindowLoad{389, 6});
  CHECK(!window_pays(b, false, false) && window_pays(b, false, true));
"""
    _run(tmp_path, body)
