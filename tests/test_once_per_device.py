"""OncePerDevice (csrc/pt_once.hpp), which sets the kernels' dynamic LDS limits:
a setting is made on every device that asks for it and not only on the first
one, once each, again after a failure, and by any thread."""
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "projectracer_amd" / "csrc"

PROGRAM = r"""
#include <cstdio>
#include <thread>
#include <vector>
#include "pt_once.hpp"

int main() {
  static pt::OncePerDevice once;
  int calls[3] = {0, 0, 0};
  auto on = [&](int d) { return once.apply(d, [&] { calls[d]++; return 0; }); };
  if (on(0) || on(0) || on(1) || on(1) || on(0)) return 1;
  if (calls[0] != 1 || calls[1] != 1) return 2;
  int tries = 0;
  auto failing = [&] { return ++tries < 3 ? 7 : 0; };
  if (once.apply(2, failing) != 7 || once.apply(2, failing) != 7) return 3;
  if (once.apply(2, failing) != 0 || once.apply(2, failing) != 0 || tries != 3) return 4;
  int far = 0;   // beyond the devices it remembers: set every time
  for (int k = 0; k < 3; k++) once.apply(64, [&] { far++; return 0; });
  if (far != 3) return 5;
  static pt::OncePerDevice shared;
  std::atomic<int> set[8] = {};
  std::vector<std::thread> pool;
  for (int t = 0; t < 8; t++)
    pool.emplace_back([&, t] {
      for (int k = 0; k < 1000; k++) {
        const int d = (t + k) % 8;
        shared.apply(d, [&] { set[d]++; return 0; });
        if (set[d] == 0) std::printf("device %d not set\n", d);
      }
    });
  for (std::thread& t : pool) t.join();
  for (auto& s : set)
    if (s < 1) return 6;
  std::puts("ok");
  return 0;
}
"""


def test_a_setting_is_made_once_on_every_device(tmp_path):
    cxx = shutil.which("g++") or shutil.which("clang++")
    if cxx is None:
        pytest.skip("no C++ compiler")
    (tmp_path / "once.cpp").write_text(PROGRAM)
    exe = tmp_path / "once"
    subprocess.run([cxx, "-std=c++17", "-O1", "-pthread", "-I", str(CSRC), str(tmp_path / "once.cpp"), "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", (r.returncode, r.stdout)
