"""Admission of factorizations whose panel workgroups wait for each other
(csrc/gate.h): which shares of a GPU are admitted together, that a waiting
thread is woken, and that threads are served in order of arrival."""
import os
import subprocess

from conftest import PKG

SRC = r"""
#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <thread>
#include <vector>
#include "gate.h"
using namespace std::chrono_literals;
static void check(bool ok, const char *what) { if (!ok) { std::printf("failed: %s\n", what); std::_Exit(1); } }
// runs enter(share) on a thread of its own; whether it got in within 50 ms
struct Try {
  std::atomic<bool> in{false};
  std::thread t;
  Try(scuffx::Gate &g, double share) : t([&g, share, this] { g.enter(share); in = true; }) {}
  bool now() { for (int i = 0; i < 50 && !in; i++) std::this_thread::sleep_for(1ms); return in; }
  ~Try() { t.join(); }
};
int main()
{
  scuffx::Gate g;
  g.enter(0.25);
  { Try a(g, 0.25); check(a.now(), "a quarter beside a quarter"); }
  {
    Try b(g, 0.0625);
    check(!b.now(), "more than a half together");
    { Try c(g, 0.0); check(!c.now(), "served in order of arrival"); g.leave(0.25); check(c.now(), "woken in turn"); }
    check(b.now(), "woken by the one that left");
  }
  g.leave(0.25); g.leave(0.0625); g.leave(0.0);
  g.enter(1.0);                                     // by itself, any share
  { Try d(g, 0.01); check(!d.now(), "beside a whole GPU"); g.leave(1.0); check(d.now(), "after it"); }
  { Try e(g, 0.75); check(!e.now(), "a large share waits for all others"); g.leave(0.01); check(e.now(), "alone"); }
  g.leave(0.75);
  // never more than a half at once, or one alone; everyone gets through
  std::atomic<int> inside{0}, sum{0}, done{0};
  std::vector<std::thread> ts;
  for (int i = 0; i < 8; i++)
    ts.emplace_back([&, i] {
      for (int k = 0; k < 200; k++) {
        const int share = 1 + (7 * i + 13 * k) % 64;
        g.enter(share / 64.0);
        const int n = ++inside, s = sum += share;
        check(n == 1 || s <= 32, "admitted together");
        sum -= share;
        inside--;
        g.leave(share / 64.0);
        done++;
      }
    });
  for (auto &t : ts) t.join();
  check(done == 1600, "all served");
  std::printf("ok\n");
}
"""


def test_gate(tmp_path):
    src, exe = tmp_path / "gate.cpp", tmp_path / "gate"
    src.write_text(SRC)
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", os.path.join(PKG, "csrc"), str(src), "-o", str(exe)],
                   check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and out.stdout == "ok\n", out.stdout
