"""Workgroups of the FIPPI cubature and the memory that their heaps take
(csrc/fippi_heap.h): what is reserved stays free, and the heaps of the
workgroups that it answers fit into the rest, keys and numbers included."""
import os
import subprocess

from conftest import PKG

SRC = r"""
#include <cstdio>
#include "fippi_heap.h"
using namespace scuffx;
int main()
{
  const size_t GB = (size_t)1 << 30, res = 5 * GB + GB / 2;
  int bad = 0;
  auto want = [&](bool ok, int line) { if (!ok) { std::printf("failed: line %d\n", line); bad = 1; } };
  want(kFippiHeapBytes == (size_t)15360 * 620, __LINE__);
  want(fippi_slots(100000, 200 * GB, res) == 1024, __LINE__);
  want(fippi_slots(77, 200 * GB, res) == 77, __LINE__);
  // room for 1024 heaps' records, not for their keys
  const size_t edge = (size_t)1024 * 15360 * 608 + (90 << 20);
  want(fippi_slots(100000, edge + res, res) < 1024, __LINE__);
  for (size_t f = 0; f < 40 * GB; f += 37 << 20) {
    const int n = fippi_slots(100000, f, res);
    const size_t need = kFippiHeapBytes * n;
    want(n >= 1 && n <= 1024, __LINE__);
    want(n == 1 || need + res <= f || need <= f / 8, __LINE__);        // the reserve is kept, or an eighth used
    want(n == 1024 || need + kFippiHeapBytes + res > f, __LINE__);     // and no more than that held back
  }
  if (!bad) std::printf("ok\n");
  return bad;
}
"""


def test_slots(tmp_path):
    src, exe = tmp_path / "heap.cpp", tmp_path / "heap"
    src.write_text(SRC)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(PKG, "csrc"), str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and out.stdout == "ok\n", out.stdout
