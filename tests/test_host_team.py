"""Host threads of a transfer (csrc/host_team.h) when helpers cannot be
started: built for the CPU with an operator new that fails at every allocation
in turn.  Every item has to be taken, every started helper ended, and the
caller's own exception has to come through."""
import os
import subprocess

from conftest import PKG

SOURCE = r"""
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <new>
#include <stdexcept>
#include "host_team.h"

static std::atomic<int> fail_at{-1};  // the allocation that fails, counted from the arming (-1: none)
void *operator new(size_t n) {
  if (fail_at >= 0 && fail_at-- == 0) throw std::bad_alloc();
  if (void *p = malloc(n)) return p;
  throw std::bad_alloc();
}
void operator delete(void *p) noexcept { free(p); }
void operator delete(void *p, size_t) noexcept { free(p); }

int main() {
  for (int threads = 1; threads <= 8; ++threads)
    for (int at = -1; at < 3 * threads; ++at) {
      std::atomic<int> next{0}, done{0};
      fail_at = at;
      tpx::run_team(threads, [&](int) {
        while (next++ < 1000) ++done;
      });
      fail_at = -1;
      if (done != 1000) return printf("%d threads, allocation %d: %d items\n", threads, at, (int)done), 1;
    }
  std::atomic<int> ended{0};
  try {
    tpx::run_team(4, [&](int t) {
      if (t == 0) throw std::runtime_error("mine");
      ++ended;
    });
    return 2;
  } catch (const std::runtime_error &) {
  }
  return ended == 3 ? 0 : 3;
}
"""


def test_team_ends_whole_when_helpers_cannot_start(tmp_path):
    src, exe = tmp_path / "team.cpp", tmp_path / "team"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread", "-I", os.path.join(PKG, "csrc"), str(src), "-o", str(exe)],
                   check=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0, (run.returncode, run.stdout, run.stderr)
