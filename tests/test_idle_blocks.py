"""The bookkeeping of the idle-block pool (csrc/ngpb_pool.h), compiled for the host: exact
size classes, and the oldest blocks leave first when the pool is full, so that sizes nobody
asks for again cannot keep it full."""
import os
import shutil
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include "ngpb_pool.h"
#include <cassert>
#include <cstdint>
#include <cstdio>
int main() {
  ngpb::IdleBlocks q;
  auto ptr = [](uintptr_t k) { return reinterpret_cast<void*>(k); };
  std::vector<void*> out;
  assert(!q.take(1) && q.bytes() == 0);
  q.trim(0, out);
  assert(out.empty());
  for (uintptr_t k = 1; k <= 6; ++k) q.put(ptr(k), k % 2 ? 10 : 30);  // 10 30 10 30 10 30
  assert(q.bytes() == 120 && !q.take(20));
  q.trim(120, out);
  assert(out.empty());
  q.trim(100, out);  // the two oldest, though one would not do
  assert(out.size() == 2 && out[0] == ptr(1) && out[1] == ptr(2) && q.bytes() == 80);
  void* a = q.take(10);
  void* b = q.take(10);
  assert(a != b && (a == ptr(3) || a == ptr(5)) && (b == ptr(3) || b == ptr(5)) && !q.take(10));
  assert(q.bytes() == 60);
  // a pool of at most 100 bytes full of one size takes another size in
  out.clear();
  q.put(ptr(7), 40);
  q.trim(100 - 50, out);
  q.put(ptr(8), 50);
  assert(q.bytes() <= 100 && out.size() == 2 && out[0] == ptr(4) && out[1] == ptr(6));
  assert(q.take(50) == ptr(8) && q.take(40) == ptr(7) && q.bytes() == 0);
  std::puts("ok");
}
"""


def test_oldest_blocks_leave_first(tmp_path):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no host compiler")
    src = tmp_path / "pool.cpp"
    src.write_text(PROGRAM)
    subprocess.run([cxx, "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(REPO, "cudanextgenpb_amd", "csrc"),
                    str(src), "-o", str(tmp_path / "pool")], check=True)
    assert subprocess.run([str(tmp_path / "pool")], check=True, capture_output=True, text=True).stdout == "ok\n"
