"""The question tiles ask of a row's plasma runs (run_covers in
fdtd2d_amd/csrc/runs.h), compiled alone with g++: the answer against a look at
every cell, and that it reads few of the runs however many there are."""

from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent

HARNESS = r"""
#include <cstdio>
#include <random>
#include <vector>
#include "runs.h"
static long reads = 0;
struct Counted {
  int v;
  operator int() const { ++reads; return v; }
};
struct Run {
  Counted x, y;
};
int main() {
  std::mt19937 rng(11);
  long bad = 0, most = 0;
  for (int t = 0; t < 20000; ++t) {
    const int n = 1 + rng() % 400, density = 1 + rng() % 40;
    std::vector<char> cell(n);
    for (int i = 0; i < n; ++i) cell[i] = i && rng() % density ? cell[i - 1] : rng() % 2;
    std::vector<Run> r(rng() % 3, Run{{0}, {n}});  // another row's runs before the row's own
    const int first = static_cast<int>(r.size());
    fdtd2d::scan_runs(n, [&](int i) { return static_cast<int>(cell[i]); },
                      [&](int a, int b) { r.push_back(Run{{a}, {b}}); });
    const int end = static_cast<int>(r.size());
    r.push_back(Run{{0}, {n}});  // and after them
    for (int q = 0; q < 20; ++q) {
      const int c0 = rng() % n, c1 = c0 + 1 + rng() % (n - c0);
      bool want = true;
      for (int i = c0; i < c1; ++i) want = want && cell[i];
      bad += fdtd2d::run_covers(r.data(), first, end, c0, c1) != want;
    }
  }
  std::vector<Run> many;
  for (int i = 0; i < 4096; ++i) many.push_back(Run{{2 * i}, {2 * i + 1}});
  for (int c0 = 0; c0 < 8192; c0 += 64) {
    reads = 0;
    bad += fdtd2d::run_covers(many.data(), 0, 4096, c0, c0 + 64);
    most = reads > most ? reads : most;
  }
  printf("bad %ld most %ld\n", bad, most);
  return bad != 0 || most > 20;  // 13 halvings of 4096 runs and the one found
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_run_covers(tmp_path):
    src = tmp_path / "runs.cpp"
    src.write_text(HARNESS)
    exe = tmp_path / "runs"
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", "-I", str(ROOT / "fdtd2d_amd" / "csrc"),
                    str(src), "-o", str(exe)], check=True, capture_output=True, text=True, timeout=120)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.startswith("bad 0 "), r.stdout
