"""Host-only checks of libmk's native helpers, compiled with the system C++
compiler (no GPU): the per-device "done once" flag that guards the
dynamic-LDS kernel attribute (mkernel_amd/csrc/mk_once.h) and the expert
GEMMs' map from tile numbers to output tiles (mkernel_amd/csrc/mk_map.h)."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent

PROG = r"""
#include <cstdio>
#include <thread>
#include <vector>
#include "mk_once.h"
int main() {
  mk::PerDeviceFlag f;
  // every device starts clear, and setting one leaves the others clear
  for (int d : {0, 1, 7, 63, 64, 65, 200}) if (f.is_set(d)) return 1;
  f.set(1);
  if (!f.is_set(1) || f.is_set(0) || f.is_set(2)) return 2;
  f.set(70);
  if (!f.is_set(70) || f.is_set(69) || f.is_set(71) || f.is_set(6)) return 3;
  if (f.is_set(-1)) return 4;
  f.set(-1);  // ignored
  // concurrent setters on distinct devices: every bit lands
  mk::PerDeviceFlag g;
  std::vector<std::thread> ts;
  for (int d = 0; d < 96; ++d) ts.emplace_back([&g, d] { g.set(d); });
  for (auto& t : ts) t.join();
  for (int d = 0; d < 96; ++d) if (!g.is_set(d)) return 5;
  if (g.is_set(96)) return 6;
  std::puts("ok");
  return 0;
}
"""


def _run(tmp_path, name, prog):
    src = tmp_path / f"{name}_test.cpp"
    src.write_text(prog)
    exe = tmp_path / f"{name}_test"
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", str(ROOT / "mkernel_amd" / "csrc"), str(src),
                    "-o", str(exe)], check=True, capture_output=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True)
    assert res.returncode == 0 and res.stdout.strip() == "ok", (res.returncode, res.stdout, res.stderr)


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host C++ compiler")
def test_per_device_flag(tmp_path):
    _run(tmp_path, "once", PROG)


# Padded counts (multiples of 128 or not, zeros among them) whose sum is below,
# at or above the launch's rows: every tile of the launch comes up once, with
# the expert that a walk over the counts finds for its first row, and negative
# counts (no layout at all) stay inside the launch.
MAP_PROG = r"""
#include <cstdio>
#include <random>
#include <vector>
#include "mk_map.h"
static int holder(const std::vector<int>& n, int row, int& beg, int& end) {
  end = 0;
  for (size_t e = 0; e < n.size(); ++e) {
    beg = end;
    end += n[e];
    if (row < end) return (int)e;
  }
  return (int)n.size() - 1;
}
int main() {
  std::mt19937 rng(7);
  for (int it = 0; it < 20000; ++it) {
    const int E = 1 + rng() % 6, tiles_m = 1 + rng() % 9, tiles_n = 1 + rng() % 5;
    const bool wrong = it % 10 == 9;
    std::vector<int> n(E);
    for (int& x : n) x = rng() % 4 == 0 ? 0 : (int)(rng() % 5) * 128 + (rng() % 8 == 0 ? 64 : 0);
    if (wrong) n[rng() % E] = -(int)(rng() % 700);
    std::vector<int> seen(tiles_m * tiles_n, 0);
    for (int t = 0; t < tiles_m * tiles_n; ++t) {
      int beg, end, r0, r1, tm, tn, b, x;
      const int rt = t / tiles_n, e = holder(n, rt * 128, beg, end);
      mk::expert_run(rt, beg, end, e == E - 1, tiles_m, 128, r0, r1);
      mk::expert_run_tile(t, r0, r1, tiles_n, tm, tn);
      if (tm < 0 || tm >= tiles_m || tn < 0 || tn >= tiles_n) return 1;
      if (wrong) continue;
      if (++seen[tm * tiles_n + tn] != 1) return 2;
      if (holder(n, tm * 128, b, x) != e) return 3;
    }
  }
  std::puts("ok");
  return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host C++ compiler")
def test_expert_map(tmp_path):
    _run(tmp_path, "expert_map", MAP_PROG)
