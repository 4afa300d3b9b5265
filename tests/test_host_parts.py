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
