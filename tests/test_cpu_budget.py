"""The budget that admits resident sweeps and their back-off
(csrc/sa_budget.h): host code, built and run with the host compiler."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "slepc_amd", "csrc")

CODE = r"""
#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstring>
#include <thread>
#include <vector>
#include "sa_budget.h"

static void nap(int ms) { std::this_thread::sleep_for(std::chrono::milliseconds(ms)); }

// more units than there are at all: refused at once, the rest unaffected
static int too_many() {
  sa::Budget b(31);
  if (b.take(32)) return 1;
  if (!b.take(31)) return 2;
  b.give(31);
  return 0;
}

// a taker of everything gets in although half-takers keep overlapping
static int in_order() {
  sa::Budget b(32);
  std::atomic<bool> quit{false}, got{false};
  auto half = [&](int offset) {
    nap(offset);
    while (!quit) {
      if (!b.take(16)) return;
      nap(40);
      b.give(16);
    }
  };
  std::thread t1(half, 0), t2(half, 20);
  nap(60);                       // both are at work, each hands over while the other holds
  std::thread all([&] {
    if (b.take(32)) {
      got = true;
      b.give(32);
    }
  });
  for (int i = 0; i < 200 && !got; i++) nap(5);
  const bool ok = got;
  quit = true;
  t1.join();
  t2.join();
  all.join();
  return ok ? 0 : 1;
}

// never more than the total in use, everything given back
static int bounded() {
  sa::Budget b(8);
  std::atomic<int> used{0}, over{0}, done{0};
  std::vector<std::thread> t;
  for (int i = 0; i < 6; i++)
    t.emplace_back([&, i] {
      for (int k = 0; k < 300; k++) {
        const int u = 1 + (i + k) % 8;
        if (!b.take(u)) return;
        if ((used += u) > 8) over++;
        std::this_thread::yield();
        used -= u;
        b.give(u);
        done++;
      }
    });
  for (auto &x : t) x.join();
  if (!b.take(8)) return 1;
  return over || done != 1800 ? 2 : 0;
}

// the turns on which something that always fails is tried, and recovery
static int backoff() {
  sa::Backoff b;
  int tries = 0, last = 0;
  for (int turn = 1; turn <= 2000; turn++)
    if (b.due()) {
      const int gap = turn - last, want = tries == 0 ? 1 : (tries < 9 ? 1 << (tries - 1) : 256);
      if (gap != want) return 1;
      tries++;
      last = turn;
      b.failed();
    }
  while (!b.due()) {
  }
  b.succeeded();
  for (int i = 0; i < 5; i++)
    if (!b.due()) return 2;
  b.failed();                    // the first failure after a success is forgiven
  return b.due() ? 0 : 3;
}

int main(int, char **v) {
  if (!std::strcmp(v[1], "too_many")) return too_many();
  if (!std::strcmp(v[1], "in_order")) return in_order();
  if (!std::strcmp(v[1], "backoff")) return backoff();
  return bounded();
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("c++")
    if not cxx:
        pytest.skip("no host compiler")
    d = tmp_path_factory.mktemp("budget")
    (d / "t.cpp").write_text(CODE)
    subprocess.run([cxx, "-O1", "-std=c++17", "-pthread", "-I", CSRC, str(d / "t.cpp"), "-o", str(d / "t")], check=True)
    return str(d / "t")


@pytest.mark.parametrize("what", ["too_many", "in_order", "bounded", "backoff"])
def test_budget(program, what):
    """A demand beyond the total is refused instead of awaited, waiting threads
    are served in the order they came, and the units in use never exceed the
    total; what fails again and again is tried less and less often."""
    assert subprocess.run([program, what], timeout=20).returncode == 0
